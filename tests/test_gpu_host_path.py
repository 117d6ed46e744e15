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


def _w():
    return torch.zeros((64, 64), dtype=torch.int8, device="cuda")


def _s(dtype=torch.float16):
    return torch.ones((64, 1), dtype=dtype, device="cuda")


def _one(value=0.05):
    return torch.full((1,), value, device="cuda")


_C = flow._C
_MAPPED = {
    "fused_linear": (torch.float16, lambda x: _C.fused_linear_with_groupwise_quantized_weight(
        x, _w(), _s())),
    "grouped_linear": (torch.float16, lambda x: _C.grouped_linear_with_groupwise_quantized_weight(
        [x, x], [_w(), _w()], [_s(), _s()])),
    "fused_glu": (torch.float16, lambda x: _C.fused_glu_with_groupwise_quantized_weight(
        x, _w(), _s(), activation="silu")),
    "groupwise_dequantize": (torch.int8, lambda x: _C.groupwise_dequantize(x, _s())),
    "groupwise_quantize": (torch.float16, lambda x: flow.quantize.groupwise_quantize(
        x, num_bits=8, symmetric=True, group_dim=1, group_size=64)),
    "min_max_observer": (torch.float32, lambda x: _C.min_max_observer(x)),
    "moving_average": (torch.float32, lambda x: _C.moving_average_min_max_observer(
        x, torch.zeros(1, dtype=torch.int64, device="cuda"), _one(0.), _one(0.), True, 1)),
    "quantization": (torch.float32, lambda x: _C.quantization(x, _one(), _one(0.))),
    "fake_quantization": (torch.float32, lambda x: _C.fake_quantization(x, _one(), _one(0.))),
    "layer_norm_observer": (torch.float16, lambda x: _C.fused_layer_norm_min_max_observer(x)),
    "layer_norm_quantization": (torch.float16, lambda x: _C.fused_layer_norm_quantization(x)),
    "skip_layer_norm": (torch.float16, lambda x: _C.fused_skip_layer_norm_min_max_observer(x)),
    "matmul_quant": (torch.int8, lambda x: _C.matmul_quant(
        x, _w(), _one(), _s(torch.float32)[:, 0])),
}


@pytest.mark.parametrize("dim", [0, 1, 2])
@pytest.mark.parametrize("name", list(_MAPPED))
def test_function_transforms_are_refused(name, dim):
    """A tensor that torch.vmap hands out has no storage: every entry raises, also where the mapped
    slice is not contiguous (dim 2) and its copy is what has none, and the process goes on."""
    dtype, call = _MAPPED[name]
    x = torch.ones((64, 64, 64), dtype=dtype, device="cuda")
    with pytest.raises(RuntimeError, match="storage"):
        torch.vmap(call, in_dims=dim)(x)
    call(x[0])
    torch.cuda.synchronize()
