"""Loader for the in-tree HIP library ``csrc/libofq_hip.so`` (the C ABI of ``include/ofq.h``) and
for ``csrc/ofq_torch.so``, the extension module that calls it with torch tensors.

There is no CPU fallback: if a library is missing the first call fails, and every call checks the
returned status and raises.
"""
import ctypes
import importlib.machinery
import importlib.util
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "csrc", "libofq_hip.so")
TORCH_LIB_PATH = os.path.join(_HERE, "csrc", "ofq_torch.so")

# mirror of the enums in include/ofq.h
OK = 0
ERR_UNSUPPORTED = 5
F32, F16, BF16, F64, I8, U8 = 0, 1, 2, 3, 4, 5
SCHEME = {"symmetric": 0, "affine": 1}
FORMULA = {"google": 0, "cambricon": 1}
ZP_MODE = {"float": 0, "uint8": 1}
LN_STATS_FP32, LN_STATS_FP64 = 0, 1

_vp = ctypes.c_void_p
_i = ctypes.c_int
_i64 = ctypes.c_int64
_sz = ctypes.c_size_t

# name -> (restype, argtypes); must match include/ofq.h exactly
SIGNATURES = {
    "ofq_status_string": (ctypes.c_char_p, [_i]),
    "ofq_abi_version": (_i, []),
    "ofq_groupwise_dequantize": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i64, _i64, _i64]),
    "ofq_fused_linear_gq_workspace_bytes": (_sz, [_i, _i, _i, _i, _i, _i64, _i64, _i64, _i64]),
    "ofq_fused_linear_gq": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i64,
                                 _i64, _i64, _i64, _vp, _sz]),
    "ofq_min_max_observer_workspace_bytes": (_sz, [_i, _i64, _i64]),
    "ofq_min_max_observer": (_i, [_vp, _vp, _vp, _vp, _i, _i64, _i64, _i, _i, _i, _vp, _sz]),
    "ofq_moving_average_min_max_observer_workspace_bytes": (_sz, [_i, _i64]),
    "ofq_moving_average_min_max_observer": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i64, _i,
                                                 _i, _i, ctypes.c_float, _i64, _i, _vp, _sz]),
    "ofq_quantization": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i, _i64, _i64, _i, _i, _i, _i]),
    "ofq_fake_quantization": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i64, _i64, _i, _i, _i, _i]),
    "ofq_fused_layer_norm_min_max_observer_workspace_bytes": (_sz, [_i, _i64, _i64]),
    "ofq_fused_layer_norm_min_max_observer": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i64,
                                                   _i64, ctypes.c_double, _i, _vp, _sz]),
    "ofq_fused_layer_norm_min_max_observer_static": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i,
                                                          _i64, _i64, ctypes.c_double, _i]),
    "ofq_fused_skip_layer_norm_min_max_observer": (_i, [_vp, _vp, _vp, _vp, ctypes.c_double, _vp,
                                                        _vp, _vp, _vp, _vp, _i, _i64, _i64,
                                                        ctypes.c_double, _i, _vp, _sz]),
    "ofq_fused_layer_norm_min_max_observer_stats": (_i, [_vp, _vp, _vp, _vp, ctypes.c_double, _i,
                                                         _vp, _vp, _vp, _vp, _vp, _i, _i64, _i64,
                                                         ctypes.c_double, _i, _i, _vp, _sz]),
    "ofq_fused_layer_norm_quantization": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i64, _i64,
                                               ctypes.c_double, _i, _i, _vp, _sz]),
    "ofq_fused_layer_norm_quantization_any_row": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i64, _i64,
                                                       ctypes.c_double, _i, _i, _vp, _sz]),
    "ofq_fused_layer_norm_quantization_workspace_bytes": (_sz, [_i, _i64, _i64]),
    "ofq_grouped_linear_gq": (_i, [_vp, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i,
                                   _i, _i, _i64]),
    "ofq_fused_glu_gq": (_i, [_vp] * 13 + [_i, _i, _i, _i, _i, _i, _i64, _i64, _i64, _i64]),
    "ofq_groupwise_quantize": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i64, _i64, _i64]),
    "ofq_matmul_quant": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i64, _i64, _i64]),
    "ofq_matmul_quant_workspace_bytes": (_sz, [_i64, _i64, _i64]),
    "ofq_matmul_quant_ws": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i64, _i64, _i64, _vp, _sz]),
    "ofq_groupwise_repack_bytes": (_sz, [_i, _i64, _i64]),
    "ofq_groupwise_repack": (_i, [_vp, _vp, _vp, _i, _i64, _i64]),
    "ofq_fused_linear_gq_tiled": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i64,
                                       _i64, _i64, _i64]),
}


class OfqError(RuntimeError):
    """A C-ABI call returned a non-zero ofq_status."""

    def __init__(self, fn, status, text):
        super().__init__(f"{fn} failed with status {status}: {text}")
        self.status = status


_lib = None


def _require(path):
    if not os.path.exists(path):
        raise RuntimeError(
            f"{path} is missing: build it with `make -C {os.path.dirname(path)}` "
            "(or __graft_entry__.build()); there is no CPU fallback")


def lib():
    """The loaded library with prototypes set.  Raises if it has not been built."""
    global _lib
    if _lib is None:
        _require(LIB_PATH)
        handle = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype = res
            fn.argtypes = args
        _lib = handle
    return _lib


class CheckFailedError(RuntimeError):
    """Raised where the reference functor's CHECK_OR_RETURN would fail."""


class _Native:
    """The functions of ``csrc/ofq_torch.cpp``.  The module is loaded when the first of them is
    looked up; from then on each is a plain attribute of this object."""

    def __getattr__(self, name):
        _require(LIB_PATH)
        _require(TORCH_LIB_PATH)
        loader = importlib.machinery.ExtensionFileLoader("ofq_torch", TORCH_LIB_PATH)
        module = importlib.util.module_from_spec(
            importlib.util.spec_from_loader("ofq_torch", loader))
        loader.exec_module(module)
        module.set_errors(CheckFailedError, OfqError)
        self.__dict__.update({k: v for k, v in vars(module).items() if not k.startswith("_")})
        try:
            return self.__dict__[name]
        except KeyError:
            raise AttributeError(name) from None


native = _Native()
