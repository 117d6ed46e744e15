"""Which tile and how many K slices gemm_wr is launched with (host code of the library: no GPU)."""
import ctypes

import pytest

from oneflow_amd import _lib


class LinearArgs(ctypes.Structure):  # csrc/ofq_internal.h
    _fields_ = ([(f, ctypes.c_void_p) for f in ("x", "w", "scale", "zero", "bias", "out")]
                + [("t_dtype", ctypes.c_int), ("w_signed", ctypes.c_bool), ("bits", ctypes.c_int),
                   ("symmetric", ctypes.c_bool), ("group_dim", ctypes.c_int)]
                + [(f, ctypes.c_int64) for f in ("group_size", "m", "n", "k")])


class WrPlan(ctypes.Structure):
    _fields_ = [("tile", ctypes.c_int), ("splits", ctypes.c_int)]


TILES = [(32, 128), (64, 128), (96, 128), (128, 256), (192, 256)]  # enum WrTile


def _plan(m, n, k, bits, symmetric, dtype, workspace, group=128):
    f = _lib.lib()["_ZN3ofq12gemm_wr_planERKNS_10LinearArgsEbPNS_6WrPlanE"]
    f.restype, f.argtypes = ctypes.c_bool, [ctypes.POINTER(LinearArgs), ctypes.c_bool,
                                            ctypes.POINTER(WrPlan)]
    args = LinearArgs(t_dtype=dtype, w_signed=symmetric, bits=bits, symmetric=symmetric,
                      group_dim=1, group_size=group, m=m, n=n, k=k)
    plan = WrPlan(-1, -1)
    return plan if f(ctypes.byref(args), workspace, ctypes.byref(plan)) else None


def _blocks(plan, m, n):
    bm, bn = TILES[plan.tile]
    return -(-m // bm) * -(-n // bn)


@pytest.mark.parametrize("dtype", [_lib.F16, _lib.BF16])
@pytest.mark.parametrize("bits,symmetric", [(4, True), (4, False), (8, True), (8, False)])
@pytest.mark.parametrize("m,n,k", [(70, 5120, 5120), (100, 4096, 11008), (128, 4096, 14336),
                                   (140, 5120, 13824), (256, 4096, 4096), (333, 1536, 8192)])
def test_without_a_workspace_the_tiles_alone_cover_the_chip(m, n, k, bits, symmetric, dtype):
    """A tile chosen for many slices leaves most of the 256 CUs idle when there is no workspace for
    them (128 x 256 on 70 x 5120: 20 blocks, twice the time of the in-tile GEMM's 160)."""
    plan = _plan(m, n, k, bits, symmetric, dtype, workspace=False)
    if plan is None:
        return  # the in-tile GEMM, on tiles of its own
    assert plan.splits == 1
    least = min(128, -(-m // 64) * -(-n // 128))
    assert _blocks(plan, m, n) >= least, (TILES[plan.tile], _blocks(plan, m, n), least)


@pytest.mark.parametrize("m", [17, 64, 65, 200, 1000])
def test_with_a_workspace_no_slice_is_empty(m):
    for n, k in ((600, 1024), (4096, 11008), (32000, 4096), (1001, 2112)):
        plan = _plan(m, n, k, 4, True, _lib.F16, workspace=True, group=32)
        if plan is not None and plan.splits > 1:
            step = 128 if TILES[plan.tile][1] == 128 else 64
            steps = -(-k // step)
            per = -(-steps // plan.splits)
            assert (plan.splits - 1) * per < steps


@pytest.mark.parametrize("m", [17, 64, 65, 200, 1000])
@pytest.mark.parametrize("n,k", [(600, 1024), (4096, 11008), (32000, 4096), (11008, 4096), (1001, 2112)])
def test_the_workspace_is_what_the_slices_take(m, n, k):
    """No slices, no workspace; else whole 32 x 32 tiles of fp32 sums, rounded up to whole [m, n], and at
    least what the in-tile GEMM's slices (at most 8) would take."""
    for bits, symmetric in ((4, True), (8, False)):
        plan = _plan(m, n, k, bits, symmetric, _lib.F16, workspace=True, group=32)
        if plan is None:
            continue
        need = _lib.lib().ofq_fused_linear_gq_workspace_bytes(
            _lib.I8 if symmetric else _lib.U8, _lib.F16, bits, symmetric, 1, 32, m, n, k)
        if need == 0:  # one slice, or left to the streaming kernel
            assert plan.splits == 1 or m <= 64
            continue
        tiles = plan.splits * -(-m // 32) * -(-n // 32) * 4096
        most = max(tiles + 4 * m * n - 1, 8 * 4 * m * n if m > 64 else 0)
        assert plan.splits > 1 and tiles <= need <= most, (m, n, k, plan.splits, need)
