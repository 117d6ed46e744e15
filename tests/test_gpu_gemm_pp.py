"""The copy-fed GEMM whose two groups of waves alternate: every width of its tiles, one to four k-tiles
with a full and a padded last one, partial last tiles in both directions, and more than 8 tiles of
rows (they share columns in panels of 8, the last panel shorter)."""
import pytest
import torch


pytestmark = pytest.mark.gpu

# (m, n): tiles of 256 x 192, 256, 384, 384 with 10, 5, 8 and 17 tiles of rows; 256 x 128 (the kernel
# whose waves stay in step) with 6 and 12
SHAPES = [(2305, 4000), (1025, 11005), (2047, 11005), (4100, 3900), (1300, 1001), (2900, 2100)]


@pytest.mark.parametrize("k", [64, 128, 192, 384, 448])
@pytest.mark.parametrize("m,n", SHAPES)
def test_int8_exact(m, n, k):
    import oneflow_amd as flow
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-128, 128, (m, k), generator=gen, device="cuda", dtype=torch.int8)
    b = torch.randint(-128, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8)
    sa = torch.full((1,), 0.013, device="cuda")
    sb = torch.rand(n, generator=gen, device="cuda") + 0.5
    bias = torch.randn(n, generator=gen, device="cuda")
    acc = (a.double() @ b.double().T).float()  # sums below 2^24: exact
    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        out = flow._C.matmul_quant(a, b, sa, sb, bias.to(dtype), out_dtype=dtype)
        ref = (acc * (sa * sb) + bias.to(dtype).float()).to(dtype)
        assert torch.equal(out, ref), (m, n, k, dtype)


# |result - exact| <= one rounding to the dtype + k fp32 roundings of the running sum of |x||w|
@pytest.mark.parametrize("k", [32, 64, 160, 256])
@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("dtype,eps", [(torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)])
def test_two_pass_linear(m, n, k, dtype, eps):
    import oneflow_amd as flow
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    w = torch.randint(-128, 128, (n, k // 2), generator=gen, device="cuda", dtype=torch.int8)
    scale = (torch.rand(n, k // 32, generator=gen, device="cuda") * 0.02 + 1e-3).to(dtype)
    out = flow._C.fused_linear_with_groupwise_quantized_weight(
        x, w, scale, num_bits=4, symmetric=True, group_dim=1, group_size=32)
    full = flow._C.groupwise_dequantize(w, scale, num_bits=4, symmetric=True, group_dim=1,
                                        group_size=32).double()
    ref = x.double() @ full.T
    bound = eps * ref.abs() + (k + 1) * 2.0 ** -24 * (x.double().abs() @ full.abs().T) + 2.0 ** -24
    assert bool(((out.double() - ref).abs() <= bound).all()), (m, n, k, dtype)


def test_replays_in_a_graph():
    import oneflow_amd as flow
    a = torch.randint(-128, 128, (2047, 384), device="cuda", dtype=torch.int8)
    b = torch.randint(-128, 128, (11005, 384), device="cuda", dtype=torch.int8)
    sa, sb = torch.ones(1, device="cuda"), torch.ones(11005, device="cuda")
    eager = flow._C.matmul_quant(a, b, sa, sb, out_dtype=torch.float32)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = flow._C.matmul_quant(a, b, sa, sb, out_dtype=torch.float32)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
