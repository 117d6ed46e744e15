"""Weight quantiser + packer: fp16/bf16/fp32 weights -> the groupwise int4/int8 format that
``_C.groupwise_dequantize`` and ``_C.fused_linear_with_groupwise_quantized_weight`` consume.

The reference has no op for this; the format is defined by the helpers of its own test
(``python/oneflow/test/modules/test_groupwise_quantization.py:26-81``), whose signature and
arithmetic ``groupwise_quantize`` follows: ``(num_bits, symmetric, x, group_dim, group_size,
quant_type) -> (quantized, scale, zero)``.
"""
import torch

from ._lib import CheckFailedError
from ._lib import native as _native


def groupwise_quantize(x, *, num_bits=8, symmetric=True, group_dim=-1, group_size=-1,
                       quant_type=torch.int8):
    """x: 2-D weight [n, k] on the GPU.  Returns ``(quantized, scale, zero)``; ``zero`` is None
    when ``symmetric``.  4-bit codes are packed two per byte along k, element 2i in the high
    nibble; scale/zero have the dtype of x."""
    return _native.groupwise_quantize(x, num_bits, symmetric, group_dim, group_size, quant_type)


__all__ = ["groupwise_quantize", "CheckFailedError"]
