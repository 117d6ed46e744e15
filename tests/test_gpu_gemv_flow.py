"""gemv_flow: linears, several of them and gated units of 1 to 48 rows of x; every number of tiles, ragged rows and K,
eight waves and six, groups of a lane's share up to whole chunks, with and without a zero point."""
import ctypes

import pytest
import torch

from oneflow_amd import _lib
from test_stream_plan import LinearJob, _job

pytestmark = pytest.mark.gpu


class FlowPlan(ctypes.Structure):  # csrc/ofq_internal.h
    _fields_ = [(f, ctypes.c_int) for f in ("grid", "rows_per_block", "mx", "tl", "nw", "tiled")] + [("lds", ctypes.c_size_t)]


def flow_plan(ns, m, k, g, bits, symmetric, dtype, glu):
    f = _lib.lib()["_ZN3ofq16gemv_flow_choiceERKNS_9LinearJobEPNS_8FlowPlanE"]
    f.restype, f.argtypes = ctypes.c_bool, [ctypes.POINTER(LinearJob), ctypes.POINTER(FlowPlan)]
    plan = FlowPlan()
    return plan if m > 16 or f(ctypes.byref(_job(ns, m, k, g, bits, symmetric, dtype, glu)), ctypes.byref(plan)) else None


def _linear(gen, n, k, dtype, bits, symmetric, g, bias):
    import oneflow_amd as flow
    dense = torch.nn.Linear(k, n, bias=bias, device="cuda", dtype=dtype)
    with torch.no_grad():
        dense.weight.copy_(torch.randn(n, k, device="cuda", generator=gen) * k ** -0.5)
        if bias:
            dense.bias.copy_(torch.randn(n, device="cuda", generator=gen))
    mod = flow.nn.QuantizedLinear.from_float(dense, num_bits=bits, symmetric=symmetric, group_size=g,
                                             quant_type=torch.int8 if symmetric else torch.uint8)
    full = flow._C.groupwise_dequantize(mod.weight, mod.weight_scale, zero=None if symmetric else mod.weight_zero,
                                        num_bits=bits, symmetric=symmetric, group_dim=1, group_size=g)
    return mod, full.double(), dense.bias.double() if bias else torch.zeros(n, device="cuda", dtype=torch.float64)


def _exact(x, full, bias, dtype):
    """The product in 64 bits, and how far one rounding to T, k fp32 roundings of the running sum of |x||w|
    (and of as many sums of waves) and, where the scale multiplies sums, w~ left unrounded may take it."""
    ref = x.double() @ full.T + bias
    size = x.double().abs() @ full.abs().T
    eps = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    late = 2.0 ** -11 if dtype == torch.float16 else 0.0
    bound = eps * ref.abs() + (1 + eps) * size * (late + (x.shape[1] + 16) * 2.0 ** -24) + 2.0 ** -24
    return ref, bound


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits,symmetric", [(4, True), (4, False), (8, True), (8, False)])
@pytest.mark.parametrize("mode,m,n,k,g", [
    ("one", 5, 2560, 128, 128), ("one", 9, 33, 32, 32), ("one", 16, 7, 96, 32), ("one", 8, 4099, 1184, 32),
    ("one", 3, 5000, 4096, 128), ("one", 5, 9001, 384, 64), ("one", 13, 8000, 4160, 32), ("one", 16, 11008, 2816, 128),
    ("one", 1, 4200, 4224, 128), ("one", 2, 4200, 256, 128), ("one", 12, 13000, 1152, 128), ("one", 8, 16384, 640, 128), ("one", 4, 16001, 576, 64),
    ("one", 10, 300, 11008, 64),
    ("one", 17, 2560, 1152, 128), ("one", 32, 33, 96, 32), ("one", 33, 4099, 1184, 32), ("one", 48, 11008, 1024, 128),
    ("one", 24, 16001, 576, 64), ("one", 41, 13000, 640, 128),
    ("several", 25, 1500, 2080, 32), ("several", 48, 4096, 768, 128), ("glu", 20, 4100, 1184, 32), ("glu", 48, 11008, 512, 128),
    ("several", 2, 2048, 1024, 128), ("several", 11, 1500, 2080, 32), ("several", 16, 4096, 768, 128),
    ("glu", 8, 3000, 1024, 64), ("glu", 9, 11008, 1152, 128), ("glu", 16, 12288, 512, 32), ("glu", 6, 7000, 1408, 128),
    ("glu", 15, 4100, 2080, 32)])
def test_flow(mode, m, n, k, g, bits, symmetric, dtype):
    import oneflow_amd as flow
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    ns = {"one": [n], "several": [n, n // 4, 33], "glu": [n, n]}[mode]
    code = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}[dtype]
    assert flow_plan(ns, m, k, g, bits, symmetric, code, mode == "glu") is not None
    parts = [_linear(gen, each, k, dtype, bits, symmetric, g, m % 2 == 0) for each in ns]
    x = torch.randn(m, k, device="cuda", generator=gen).to(dtype)
    want = [_exact(x, full, bias, dtype) for _, full, bias in parts]
    if mode == "one":
        got = [parts[0][0](x)]
    elif mode == "several":
        got = flow.nn.GroupedQuantizedLinear([p[0] for p in parts])(x)
    else:
        got = []
        y = flow.nn.QuantizedGLU(parts[0][0], parts[1][0], activation="silu")(x)
        (h, hb), (u, ub) = want
        # |d(h silu(u))| <= |silu(u)| dh + 1.1 |h| du, and three roundings to T
        act = torch.nn.functional.silu(u)
        bound = act.abs() * hb + 1.1 * (h.abs() + hb) * ub + 2.0 ** (-9 if dtype == torch.float16 else -6) * (h * act).abs() + 1e-6
        assert bool(((y.double() - h * act).abs() <= bound).all())
    for out, (ref, bound) in zip(got, want):
        assert bool(((out.double() - ref).abs() <= bound).all())
