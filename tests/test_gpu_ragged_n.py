"""Output rows that are not whole pieces of 16 bytes: every remainder of n, through every GEMM tile and the
folds of K slices.  The int8 product is exact, and nothing may be written past the last output."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# (m, n, k): 64 x 64 tiles; 128 x 128 on 8 and on 4 waves; 256 rows x 192, 256, 384, 128; K slices on
# 128 x 128 and on 256 x 128
SHAPES = [(512, 1096, 128), (1024, 3096, 64), (100, 25000, 64), (2305, 4000, 128), (1025, 11000, 64),
          (2047, 11000, 128), (1300, 1000, 128), (200, 1000, 6272), (600, 1000, 6272)]


@pytest.mark.parametrize("rest", range(8))
@pytest.mark.parametrize("m,n0,k", SHAPES)
def test_int8_product(m, n0, k, rest):
    from oneflow_amd import _lib
    n = n0 + rest
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-3, 4, (m, k), generator=gen, device="cuda", dtype=torch.int8)
    b = torch.randint(-3, 4, (n, k), generator=gen, device="cuda", dtype=torch.int8)
    sa = torch.full((1,), 0.25, device="cuda")
    sb = torch.randint(1, 5, (n,), generator=gen, device="cuda").float() / 4
    lib = _lib.lib()
    need = lib.ofq_matmul_quant_workspace_bytes(m, n, k)
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device="cuda")
    exact = (a.float() @ b.float().T) * (sa * sb)  # sums and scales are whole 1/16: exact
    for dtype, code in ((torch.float32, _lib.F32), (torch.float16, _lib.F16), (torch.bfloat16, _lib.BF16)):
        bias = torch.randn(n, generator=gen, device="cuda").to(dtype)
        out = torch.full((m * n + 64,), 777.0, device="cuda", dtype=dtype)
        rc = lib.ofq_matmul_quant_ws(
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), a.data_ptr(), b.data_ptr(), sa.data_ptr(),
            sb.data_ptr(), bias.data_ptr(), out.data_ptr(), code, m, n, k, ws.data_ptr() if need else None,
            need)
        assert rc == 0
        assert torch.equal(out[:m * n].view(m, n), (exact + bias.float()).to(dtype)), (m, n, k, dtype)
        assert bool((out[m * n:] == 777).all()), (m, n, k, dtype)


# one slice, several, and the fold of gemm_core2's slices; |result - exact| <= one rounding to fp16
# + k fp32 roundings of the running sum of |x||w|
@pytest.mark.parametrize("rest", range(8))
@pytest.mark.parametrize("m,n0,k,bits", [(70, 9000, 128, 4), (33, 600, 1024, 4), (100, 1096, 6144, 8),
                                         (700, 1000, 4096, 8), (600, 30000, 64, 8)])
def test_linear(m, n0, k, bits, rest):
    import oneflow_amd as flow
    n, g = n0 + rest, 32
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=gen, device="cuda", dtype=torch.float16)
    w = torch.randint(0, 256, (n, k * bits // 8), generator=gen, device="cuda", dtype=torch.uint8)
    scale = (torch.rand(n, k // g, generator=gen, device="cuda") * 0.02 + 1e-3).half()
    zero = torch.randn(n, k // g, generator=gen, device="cuda").half() * 0.1
    bias = torch.randn(n, generator=gen, device="cuda").half()
    out = flow._C.fused_linear_with_groupwise_quantized_weight(
        x, w, scale, w_zero=zero, b=bias, num_bits=bits, symmetric=False, group_dim=1, group_size=g)
    full = flow._C.groupwise_dequantize(w, scale, zero=zero, num_bits=bits, symmetric=False, group_dim=1,
                                        group_size=g).double()
    ref = x.double() @ full.T + bias.double()
    bound = 2.0 ** -11 * ref.abs() + (k + 2) * 2.0 ** -24 * (x.double().abs() @ full.abs().T + 4) + 2.0 ** -24
    assert bool(((out.double() - ref).abs() <= bound).all()), (m, n, k, bits)
