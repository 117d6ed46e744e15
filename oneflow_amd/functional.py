"""Host-side mirror of OneFlow's ``flow._C`` entry points for the quantized-inference ops.

Signatures, keyword names, defaults and argument checks follow
``oneflow/core/functional/functional_api.yaml:1061-1093`` and the functors in
``oneflow/core/functional/impl/quantization.cpp`` (same messages), so a test written against
``flow._C.groupwise_dequantize`` / ``flow._C.fused_linear_with_groupwise_quantized_weight`` /
``flow._C.min_max_observer`` / ``flow._C.quantization`` / ``flow._C.fake_quantization`` reads the
same against this module.  Tensors are ``torch`` tensors on the GPU; torch is used only to own
device memory, to name the current stream and to record ``fake_quantization`` for autograd -- all
arithmetic happens in the HIP library behind the C ABI of ``include/ofq.h``.

This module holds the names, the defaults and their documentation; what a call does (checks,
allocation of outputs and workspaces, the launch) is native, ``csrc/ofq_torch.cpp``, since at
decode sizes the kernels are shorter than the same steps written in Python.

One deliberate difference: the reference functor routes ``m > 8`` of the fused linear through
``groupwise_dequantize`` + matmul (quantization.cpp:341-350); here every ``m`` goes to the fused
op, whose kernels cover both regimes.
"""
import torch

from ._lib import CheckFailedError  # noqa: F401  (raised by the native functions)
from ._lib import native as _native


# --------------------------------------------------------------------------------------------
# groupwise_dequantize: GroupwiseDequantizeFunctor, quantization.cpp:155-220
# --------------------------------------------------------------------------------------------
def groupwise_dequantize(in_, scale, *, zero=None, num_bits=8, symmetric=True, group_dim=-1,
                         group_size=-1):
    return _native.groupwise_dequantize(in_, scale, zero, num_bits, symmetric, group_dim,
                                       group_size)


# --------------------------------------------------------------------------------------------
# fused_linear_with_groupwise_quantized_weight:
# FusedLinearWithGroupwiseQuantizedWeightFunctor, quantization.cpp:264-372
# --------------------------------------------------------------------------------------------
def fused_linear_with_groupwise_quantized_weight(x, w, w_scale, *, w_zero=None, b=None,
                                                 num_bits=8, symmetric=True, group_dim=-1,
                                                 group_size=-1):
    return _native.fused_linear(x, w, w_scale, w_zero, b, num_bits, symmetric, group_dim,
                                group_size)


def groupwise_repack(w, num_bits=4):
    """Extension (no counterpart in the reference): the tile-major copy of row-major 4-bit codes
    ``w`` [n, k/2] that ``fused_linear_with_tiled_groupwise_quantized_weight`` reads, as a flat
    uint8 / int8 tensor of ``ofq_groupwise_repack_bytes`` elements.  Done once, offline."""
    return _native.groupwise_repack(w, num_bits)


def fused_linear_with_tiled_groupwise_quantized_weight(x, w_tiled, w_scale, *, w_zero=None, b=None,
                                                       num_bits=4, symmetric=True, group_dim=-1,
                                                       group_size=-1):
    """``fused_linear_with_groupwise_quantized_weight`` on the copy ``groupwise_repack`` made of
    ``w`` (n and k are taken from ``w_scale`` and ``x``); the same bits as the row-major call.
    For up to 16 rows of ``x`` in fp16 with groups of a multiple of 128 along K; raises
    ``OfqError`` (unsupported) otherwise -- keep the row-major weight for those calls."""
    return _native.fused_linear_tiled(x, w_tiled, w_scale, w_zero, b, num_bits, symmetric,
                                      group_dim, group_size)


def grouped_linear_with_groupwise_quantized_weight(xs, ws, w_scales, *, w_zeros=None, bs=None,
                                                   num_bits=8, symmetric=True, group_dim=-1,
                                                   group_size=-1):
    """``fused_linear_with_groupwise_quantized_weight`` over tuples of problems, the quantised
    counterpart of ``grouped_matmul_bias(xs, weights, biases)`` (functional_api.yaml:2759-2760;
    checks of GroupedMatmulBiasFunctor: equal tuple lengths).  Problems of equal (m, k) with
    m <= 16 run as one launch.  Returns the list of outputs."""
    return _native.grouped_linear(xs, ws, w_scales, w_zeros, bs, num_bits, symmetric, group_dim,
                                  group_size)


def fused_glu_with_groupwise_quantized_weight(x, w, w_scale, *, w_zero=None, b=None, v=None,
                                              v_scale=None, v_zero=None, c=None,
                                              activation="none", num_bits=8, symmetric=True,
                                              group_dim=-1, group_size=-1):
    """``fused_glu(x, w, b, v, c, activation)`` (functional_api.yaml:774-775, checks of
    FusedGluFunctor, nn_functor.cpp:3724-3800) with groupwise-quantised ``w`` / ``v``:
    ``y = (x w~^T + b) * act(x v~^T + c)``; without ``v`` the 2n rows of ``w`` hold the
    hidden-state rows first and the gate rows second."""
    return _native.fused_glu(x, w, w_scale, w_zero, b, v, v_scale, v_zero, c, activation, num_bits,
                             symmetric, group_dim, group_size)


# --------------------------------------------------------------------------------------------
# min_max_observer / quantization / fake_quantization
# functors quantization.cpp:34-153; attribute checks oneflow/user/ops/min_max_observer_op.cpp:58-70,
# quantization_op.cpp:92-104
# --------------------------------------------------------------------------------------------
def min_max_observer(in_, quantization_formula="google", quantization_bit=8,
                     quantization_scheme="symmetric", per_layer_quantization=True):
    """Returns ``(scale, zero_point)``; shape ``[1]`` per layer or ``[in.shape[0]]`` per channel
    (min_max_observer_op.cpp:21-38)."""
    return _native.min_max_observer(in_, quantization_formula, quantization_bit,
                                    quantization_scheme, per_layer_quantization)


def moving_average_min_max_observer(in_, current_train_step, moving_max, moving_min, training,
                                    stop_update_after_iters, quantization_formula="google",
                                    quantization_bit=8, quantization_scheme="symmetric",
                                    momentum=0.95):
    """MovingAverageMinMaxObserverFunctor (quantization.cpp:59-91, functional_api.yaml:1079-1084).
    ``moving_max`` / ``moving_min`` (shape ``[1]``, dtype of ``in``) are updated in place while
    training and ``current_train_step <= stop_update_after_iters``; ``current_train_step`` is a
    device tensor of one int64 and is read on the device.  Returns ``(scale, zero_point)``."""
    return _native.moving_average_min_max_observer(
        in_, current_train_step, moving_max, moving_min, training, stop_update_after_iters,
        quantization_formula, quantization_bit, quantization_scheme, momentum)


def quantization(in_, scale, zero_point, quantization_formula="google", quantization_bit=8,
                 quantization_scheme="symmetric", *, out_dtype=None, zp_mode="float"):
    """``out_dtype`` (extension): ``torch.int8`` / ``torch.uint8`` to get integer codes instead
    of codes stored in the input dtype.  ``zp_mode`` selects how an affine zero point is read:
    ``"float"`` (the CUDA kernel's rule) or ``"uint8"`` (the CPU kernel's rule)."""
    return _native.quantization(in_, scale, zero_point, quantization_formula, quantization_bit,
                                quantization_scheme, out_dtype, zp_mode)


def fake_quantization(in_, scale, zero_point, quantization_formula="google", quantization_bit=8,
                      quantization_scheme="symmetric", *, zp_mode="float"):
    """Differentiable in ``in_``: the output gradient passes to it unchanged, scale and zero_point
    get none (oneflow/core/autograd/gradient_funcs/fake_quantization.cpp:36-42).  In forward mode
    the tangent of ``in_`` becomes the tangent of the result."""
    return _native.fake_quantization(in_, scale, zero_point, quantization_formula, quantization_bit,
                                     quantization_scheme, zp_mode)


# --------------------------------------------------------------------------------------------
# Ops named by the task but absent from the reference tree
# --------------------------------------------------------------------------------------------
def fused_layer_norm_min_max_observer(x, gamma=None, beta=None, epsilon=1e-5, quantization_bit=8,
                                      *, exact_statistics=False):
    """LayerNorm over the last axis + per-tensor symmetric observer of the result.
    Returns ``(y, scale, zero_point)`` with fp32 ``scale`` / ``zero_point`` of shape ``[1]``.
    ``exact_statistics``: mean and variance of a row accumulated in fp64 and rounded once (the
    correctly rounded fp32 statistics, independent of the order of summation) instead of
    accumulated in fp32."""
    return _native.layer_norm_observer(x, gamma, beta, epsilon, quantization_bit, exact_statistics)


def fused_layer_norm_quantization(x, gamma=None, beta=None, epsilon=1e-5, quantization_bit=8,
                                  *, exact_statistics=False):
    """``fused_layer_norm_min_max_observer`` followed by ``quantization`` (symmetric, per layer,
    int8 codes) of its output -- the dynamic activation quantisation in front of
    ``matmul_quant``.  Returns ``(codes, scale, zero_point)``; the normalised tensor is not
    returned.  For fp16 rows of 512, 1024, 2048 or 4096 elements with gamma and beta the library
    runs it as two kernels that never write the normalised tensor; every other case is the two
    ops in a row.  The codes and the scale carry the same bits either way."""
    return _native.layer_norm_quantization(x, gamma, beta, epsilon, quantization_bit,
                                           exact_statistics)


def fused_skip_layer_norm_min_max_observer(x, gamma=None, beta=None, bias=None, skip=None,
                                           epsilon=1e-5, alpha=1e1, quantization_bit=8,
                                           *, exact_statistics=False):
    """``skip_layer_norm`` (same arguments and defaults as the reference functional,
    functional_api.yaml:1545-1546: the row normalised is ``(x + bias) + skip * alpha`` in the
    dtype of x) + per-tensor symmetric observer of the result.  Returns
    ``(y, scale, zero_point)``."""
    return _native.skip_layer_norm_observer(x, gamma, beta, bias, skip, epsilon, alpha,
                                            quantization_bit, exact_statistics)


def matmul_quant(a, b, a_scale, b_scale, bias=None, out_dtype=torch.float16):
    """int8 ``a[m,k]`` x int8 ``b[n,k]`` -> ``out_dtype[m,n]``; exact int32 accumulation, then
    ``acc * (a_scale * b_scale[n]) + bias[n]``."""
    return _native.matmul_quant(a, b, a_scale, b_scale, bias, out_dtype)
