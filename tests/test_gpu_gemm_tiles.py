"""Every tile of the GEMMs whose operands are copied, chosen by expected time, at sizes with partial last tiles in both
directions, rows of K that are and are not whole k-tiles, and slices of K; and linears of 1024 rows and more on
packed weights, with and without slices, with the whole workspace, with room for the converted weight alone, and
with none.

int8: sums are whole numbers, exact in 64 bits, and the epilogue is one fp32 product per output: equal bits.
16 bits: |result - exact| <= one rounding to the dtype + (k + 2) fp32 roundings of the running sum of |x| |w~|."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


@pytest.mark.parametrize("m,n,k", [(74, 2112, 256), (2051, 61, 320), (1154, 1713, 640), (1365, 1477, 448),
                                   (2198, 2856, 2880), (839, 2054, 1664), (65, 1, 64), (4099, 5003, 128),
                                   (3333, 6007, 192), (2049, 5633, 1024), (65, 700, 4224), (130, 300, 8192),
                                   (300, 2500, 7168), (700, 1001, 6208), (50, 333, 8256)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_int8_tiles(m, n, k, dtype):
    import oneflow_amd as flow
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-128, 128, (m, k), generator=gen, device="cuda", dtype=torch.int8)
    b = torch.randint(-128, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8)
    a_scale = torch.full((1,), 0.0211, device="cuda")
    b_scale = torch.rand(n, generator=gen, device="cuda") * 0.01 + 1e-3
    bias = torch.randn(n, generator=gen, device="cuda").to(dtype)
    out = flow._C.matmul_quant(a, b, a_scale, b_scale, bias, out_dtype=dtype)
    sums = a.double() @ b.double().T
    ref = (sums.float() * (a_scale * b_scale) + bias.float()).to(dtype)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("m,n,k,g,bits,symmetric", [
    (1466, 107, 640, 32, 8, True), (1244, 101, 800, 32, 4, True), (1093, 2918, 384, 32, 4, True),
    (1298, 2415, 32, 32, 4, True), (2051, 3350, 1184, 32, 8, False), (2209, 3724, 640, 32, 4, False),
    (2437, 3593, 416, 32, 4, False), (2041, 1064, 64, 32, 4, False), (2446, 3024, 32, 32, 4, True),
    (1139, 686, 128, 32, 8, False), (1190, 113, 768, 32, 4, True), (2374, 63, 672, 32, 4, True),
    (1507, 1045, 64, 64, 4, False), (1338, 61, 1792, 128, 8, True), (1161, 64, 1696, 32, 4, False),
    (1675, 132, 1888, 32, 4, True), (1024, 600, 4096, 128, 4, False), (1027, 859, 2080, 32, 8, True)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_linears_of_many_rows(m, n, k, g, bits, symmetric, dtype):
    import oneflow_amd as flow
    from oneflow_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    qdt = torch.int8 if symmetric else torch.uint8
    lo = -128 if symmetric else 0
    w = torch.randint(lo, lo + 256, (n, k * bits // 8), generator=gen, device="cuda", dtype=qdt)
    scale = (torch.rand(n, k // g, generator=gen, device="cuda") * 0.02 + 1e-3).to(dtype)
    zero = None if symmetric else (torch.randn(n, k // g, generator=gen, device="cuda") * 0.1).to(dtype)
    bias = torch.randn(n, generator=gen, device="cuda").to(dtype)
    full = flow._C.groupwise_dequantize(w, scale, zero=zero, num_bits=bits, symmetric=symmetric, group_dim=1,
                                        group_size=g).double()
    ref = x.double() @ full.T + bias.double()
    mass = x.double().abs() @ full.abs().T + bias.double().abs()
    bound = EPS[dtype] * ref.abs() + (k + 2) * 2.0 ** -24 * mass + 2.0 ** -24
    wcode = _lib.I8 if symmetric else _lib.U8
    tcode = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}[dtype]
    L = _lib.lib()
    need = L.ofq_fused_linear_gq_workspace_bytes(wcode, tcode, bits, int(symmetric), 1, g, m, n, k)
    assert need >= n * k * 2
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    for room in {need, n * k * 2, 0}:
        ws = torch.empty(max(room, 16), dtype=torch.uint8, device="cuda")
        out = torch.full((m * n + 64,), 777.0, device="cuda", dtype=dtype)
        rc = L.ofq_fused_linear_gq(torch.cuda.current_stream().cuda_stream, ptr(x), ptr(w), ptr(scale), ptr(zero),
                                   ptr(bias), ptr(out), wcode, tcode, bits, int(symmetric), 1, g, m, n, k,
                                   ptr(ws) if room else None, room)
        assert rc == 0
        assert bool(((out[:m * n].view(m, n).double() - ref).abs() <= bound).all()), room
        assert bool((out[m * n:] == 777).all())
