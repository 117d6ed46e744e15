"""matmul_quant of more than 64 rows: the tiles of several k-tiles under way (fewer k-tiles than stages, as many, more;
a ragged last one; ragged rows and columns), and the streaming kernel of 65 to 96 rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    # 64 x 64, five stages and three; one k-tile to more than the stages
    (130, 4018, 768), (132, 2699, 1024), (99, 133, 1088), (129, 1683, 2048), (99, 130, 2112),
    (97, 130, 64), (98, 132, 128), (98, 132, 192), (97, 133, 256), (99, 132, 448), (97, 130, 512), (98, 133, 576),
    # 128 x 64, six stages and three
    (131, 5476, 2048), (131, 5477, 2112), (500, 4099, 4096), (194, 5488, 64), (130, 5631, 192), (196, 4188, 512), (97, 8462, 640),
    # 128 x 128, five stages and two
    (1021, 4093, 4096), (1021, 4091, 4160), (467, 8204, 64), (520, 7319, 512), (514, 7351, 704),
    # 256 x 128
    (509, 11003, 4096), (509, 11002, 4160), (2000, 4100, 2048),
    # streaming
    (65, 3, 64), (66, 2048, 512), (72, 4096, 4096), (80, 11008, 4096), (81, 8200, 1088), (96, 12288, 192), (96, 12289, 576),
    (95, 300, 8192),
    # slices
    (128, 1000, 8192), (300, 2001, 6144), (256, 1024, 8000)])
def test_deep(m, n, k):
    import oneflow_amd as flow
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-128, 128, (m, k), generator=gen, device="cuda", dtype=torch.int8)
    b = torch.randint(-128, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8)
    sa = torch.full((1,), 0.0317, device="cuda")
    sb = torch.rand(n, generator=gen, device="cuda") * 0.01 + 1e-3
    sums = (a.double() @ b.double().T).float()  # exact whole numbers (|sum| < 2^27); one rounding to fp32, as in the kernel
    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        bias = torch.randn(n, generator=gen, device="cuda").to(dtype) if (m + n) % 2 or dtype == torch.float32 else None
        want = sums * (sa * sb)
        if bias is not None:
            want = want + bias.float()
        for _ in range(2):  # (what the first launch left in LDS meets the second)
            out = flow._C.matmul_quant(a, b, sa, sb, bias, out_dtype=dtype)
            assert torch.equal(out, want.to(dtype)), (m, n, k, dtype)
