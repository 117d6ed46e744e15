"""matmul_quant of 2 to 64 rows: every instance of the streaming kernel (eights of rows of a and of a block's rows of
b), ragged rows of both, K from one 64-byte half step to many steps, one and two rounds of blocks."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [64, 192, 1024, 1088, 3136])
@pytest.mark.parametrize("n", [3, 100, 2600, 5000, 7001, 9000, 11008, 13001, 16001, 16501])
@pytest.mark.parametrize("m", [2, 8, 9, 17, 32, 33, 41, 49, 64])
def test_stream(m, n, k):
    import oneflow_amd as flow
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-128, 128, (m, k), generator=gen, device="cuda", dtype=torch.int8)
    b = torch.randint(-128, 128, (n, k), generator=gen, device="cuda", dtype=torch.int8)
    sa = torch.full((1,), 0.0317, device="cuda")
    sb = torch.rand(n, generator=gen, device="cuda") * 0.01 + 1e-3
    sums = (a.double() @ b.double().T).float()  # exact whole numbers (|sum| < 2^26); one rounding to fp32, as in the kernel
    for dtype in (torch.float32, torch.float16, torch.bfloat16):
        bias = torch.randn(n, generator=gen, device="cuda").to(dtype) if (m + n) % 2 or dtype == torch.float32 else None
        out = flow._C.matmul_quant(a, b, sa, sb, bias, out_dtype=dtype)
        want = sums * (sa * sb)
        if bias is not None:
            want = want + bias.float()
        assert torch.equal(out, want.to(dtype)), (m, n, k, dtype)
