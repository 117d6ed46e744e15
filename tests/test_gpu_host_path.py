"""What csrc/ofq_torch.cpp does around a call into the library: gradients of either mode, function
transforms, streams and threads.  (Argument checks: test_functional_checks.py; results: the test
file of each function.)"""
import pytest
import torch

import oneflow_amd as flow

pytestmark = pytest.mark.gpu


def _fake_quantization(x):
    scale = torch.full((1,), 0.05, device="cuda")
    return flow._C.fake_quantization(x, scale, torch.zeros(1, device="cuda"))


@pytest.mark.parametrize("requires_grad", [False, True])
@pytest.mark.parametrize("contiguous", [True, False])
def test_fake_quantization_forward_mode(requires_grad, contiguous):
    """The straight-through rule in forward mode: the tangent passes unchanged, as a tensor of its
    own, and nothing is attached where forward mode is off."""
    import torch.autograd.forward_ad as fwd
    x = torch.randn((33, 20), device="cuda")
    x = (x if contiguous else x.t()).requires_grad_(requires_grad)
    tangent = torch.randn_like(x)
    with fwd.dual_level():
        y = _fake_quantization(fwd.make_dual(x, tangent))
        primal, got = fwd.unpack_dual(y)
        assert torch.equal(primal, _fake_quantization(x))
        assert torch.equal(got, tangent) and got.data_ptr() != tangent.data_ptr()
        assert y.requires_grad == requires_grad
        assert fwd.unpack_dual(_fake_quantization(x)).tangent is None
        # a chain through it
        z = _fake_quantization(3 * fwd.make_dual(x, tangent)) * 2
        assert torch.equal(fwd.unpack_dual(z).tangent, 6 * tangent)
