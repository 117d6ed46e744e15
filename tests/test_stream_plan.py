"""Which streaming kernel a linear, several of them or a gated unit are launched with, and how (host code of the
library: no GPU)."""
import ctypes
import random

import pytest

import test_gpu_gemv_ring as ring_tests
from oneflow_amd import _lib
from test_gemm_plan import LinearArgs

LDS = 160 * 1024


class LinearJob(ctypes.Structure):  # csrc/ofq_internal.h, as the plans below
    _fields_ = [("pr", ctypes.POINTER(LinearArgs)), ("count", ctypes.c_int), ("glu", ctypes.c_bool),
                ("y", ctypes.c_void_p), ("act", ctypes.c_int)]


class RingPlan(ctypes.Structure):
    _fields_ = ([(f, ctypes.c_int) for f in ("grid", "rows_per_block", "tr", "tl", "wk_shift", "phase_steps",
                                             "phases")] + [("lds", ctypes.c_size_t)])


class RingMtPlan(ctypes.Structure):
    _fields_ = ([(f, ctypes.c_int) for f in ("grid", "rows_per_block", "tl", "wk", "depth", "buffers", "phases")]
                + [("lds", ctypes.c_size_t)])


class MtChoice(ctypes.Structure):
    _fields_ = [("ring", ctypes.c_bool), ("plan", RingMtPlan), ("us", ctypes.c_double)]


def _job(ns, m, k, g, bits, symmetric, dtype, glu):
    pr = (LinearArgs * len(ns))(*[
        LinearArgs(t_dtype=dtype, w_signed=symmetric, bits=bits, symmetric=symmetric, group_dim=1, group_size=g,
                   m=m, n=n, k=k) for n in ns])
    return LinearJob(pr, len(ns), glu, None, 0)


def ring_plan(ns, m, k, g, bits, symmetric, dtype=_lib.F16, glu=False):
    """The plan of gemv_ring (1 to 16 rows of x), or None where another kernel serves."""
    f = _lib.lib()["_ZN3ofq16gemv_ring_choiceERKNS_9LinearJobEPNS_8RingPlanE"]
    f.restype, f.argtypes = ctypes.c_bool, [ctypes.POINTER(LinearJob), ctypes.POINTER(RingPlan)]
    plan = RingPlan()
    return plan if f(ctypes.byref(_job(ns, m, k, g, bits, symmetric, dtype, glu)), ctypes.byref(plan)) else None


def ring_mt_plan(ns, m, k, g, bits, symmetric, dtype=_lib.F16, glu=False):
    """The plan of gemv_ring_mt (17 to 64 rows of x), or None where gemv_rows_mt is the streaming kernel."""
    f = _lib.lib()["_ZN3ofq14gemv_mt_choiceERKNS_9LinearJobEPNS_8MtChoiceE"]
    f.restype, f.argtypes = None, [ctypes.POINTER(LinearJob), ctypes.POINTER(MtChoice)]
    choice = MtChoice()
    f(ctypes.byref(_job(ns, m, k, g, bits, symmetric, dtype, glu)), ctypes.byref(choice))
    return choice.plan if choice.ring else None


def _random_job(rng, m):
    bits, g = rng.choice([4, 8]), rng.choice([32, 64, 96, 128])
    k = g * rng.randint(1, 14336 // g)
    mode = rng.choice(["one", "several", "glu"])
    ns = [rng.randint(1, 32000)] if mode == "one" else [k, max(1, k // 4), max(1, k // 4)]
    if mode == "glu":
        ns = [rng.randint(1, 20000)] * 2
    return ns, m, k, g, bits, rng.choice([True, False]), rng.choice([_lib.F16, _lib.BF16]), mode == "glu"


def _scale_bytes(rows, groups):
    return (rows * groups * 2 + 16 + 15) & ~15


def test_every_plan_of_the_ring_is_what_the_kernel_assumes():
    """All rows and all of K are covered, what the kernel lays out in LDS fits, and the counts that its waits
    are written for are kept."""
    rng, seen = random.Random(0), 0
    for _ in range(20000):
        job = ns, m, k, g, bits, symmetric, _, glu = _random_job(rng, rng.randint(1, 16))
        p = ring_plan(*job)
        if p is None:
            continue
        seen += 1
        mats, lists = (2, ns[:1]) if glu else (1, ns)
        ck = 128 if bits == 4 else 64
        sub = 2 if m <= 8 else 1
        steps, wk = -(-k // (ck * sub)), 1 << p.wk_shift
        tiles = mats * -(-p.rows_per_block // p.tr)
        depth = {1: 3, 2: 2, 3: 1, 4: 1}[p.tl]
        assert p.tr == (8 if m <= 8 else 16), job
        assert p.grid == sum(-(-n // p.rows_per_block) for n in lists), job
        assert (16 >> p.wk_shift) * p.tl >= tiles, job
        assert p.phases * p.phase_steps >= steps > (p.phases - 1) * p.phase_steps, job
        assert p.phases == 1 or p.phase_steps % wk == 0, job
        scales = mats * (1 if symmetric else 2) * _scale_bytes(p.rows_per_block, k // g)
        x = (p.phase_steps * sub * m * ck * 2 + 1023) & ~1023
        used = ((scales + 1023) & ~1023) + 16 * depth * p.tl * 1024 + x * (1 if p.phases == 1 else 2)
        assert max(used, tiles * wk * m * 64) <= p.lds <= LDS, job
    assert seen > 5000


# (rows of the weights, rows of x, k, group, bits, symmetric, gated) -> served by gemv_ring
@pytest.mark.parametrize("ns,m,k,g,bits,symmetric,glu,ring", [
    ([11008], 8, 4096, 32, 4, True, False, True), ([11008], 12, 4096, 64, 8, False, False, True),
    ([1024], 4, 8192, 64, 4, True, False, True),    # short blocks, whole turns of waves
    ([1024], 4, 4096, 64, 4, True, False, False),   # the same, one turn
    ([4096], 4, 4096, 64, 4, True, False, False),   # one 16-row tile a block
    ([11008], 1, 4096, 64, 4, True, False, False), ([11008], 1, 4128, 32, 4, True, False, True),
    ([8200], 16, 8192, 64, 8, True, False, False),  # more than 8 rows of x in four parts or more
    ([4672] * 2, 3, 1536, 32, 8, False, True, True), ([4096, 1024, 1024], 4, 4096, 64, 4, True, False, True),
    # blocks of whole 16-row tiles: 25 to 32 rows of one linear, 9 to 16 and 25 to 32 of several
    ([8097], 5, 1664, 128, 8, False, False, False), ([8097], 5, 1024, 128, 8, False, False, True),
    ([6949], 2, 5632, 128, 8, True, False, True), ([6949], 2, 4096, 128, 8, True, False, False),
    ([8193], 5, 1664, 128, 8, False, False, True), ([8097], 9, 1664, 128, 8, False, False, True),
    ([2176] * 3, 7, 2176, 32, 4, False, False, False), ([2176, 272, 272], 3, 2176, 64, 4, False, False, False),
    ([2176, 272, 272], 4, 2176, 64, 4, False, False, True), ([2048, 256, 256], 3, 2048, 64, 4, False, False, True),
    ([2560] * 3, 3, 4608, 64, 4, False, False, True),
    ([11008], 17, 4096, 64, 4, True, False, False),  # up to 16 rows of x
    ([11008], 8, 4104, 24, 4, True, False, False)])  # groups of whole lanes
def test_where_the_ring_serves(ns, m, k, g, bits, symmetric, glu, ring):
    for dtype in (_lib.F16, _lib.BF16):
        assert (ring_plan(ns, m, k, g, bits, symmetric, dtype, glu) is not None) == ring, dtype


def test_every_plan_of_17_to_64_rows_is_what_the_kernel_assumes():
    rng, seen = random.Random(1), 0
    for _ in range(20000):
        job = ns, m, k, g, bits, symmetric, _, glu = _random_job(rng, rng.randint(17, 64))
        p = ring_mt_plan(*job)
        if p is None:
            continue
        seen += 1
        mats, lists = (2, ns[:1]) if glu else (1, ns)
        ck = 128 if bits == 4 else 64
        steps, tiles = -(-k // ck), mats * -(-p.rows_per_block // 16)
        assert tiles >= 3 and p.grid == sum(-(-n // p.rows_per_block) for n in lists), job
        assert 12 % p.wk == 0 and 12 // p.wk * p.tl >= tiles and 1 <= p.tl <= 3, job
        assert 1 <= p.depth and p.depth * p.tl <= 4 and 2 <= p.buffers <= 4, job
        assert p.phases == -(-steps // p.wk), job
        x = (p.wk * m * ck * 2 + 1023) & ~1023
        assert x <= 64 * 1024, job  # what four waves copy in 16 copies each
        scales = mats * (1 if symmetric else 2) * _scale_bytes(p.rows_per_block, k // g)
        used = ((scales + 1023) & ~1023) + 12 * p.depth * p.tl * 1024 + p.buffers * x
        assert max(used, tiles * p.wk * m * 64) <= p.lds <= LDS, job
    assert seen > 3000


@pytest.mark.parametrize("ns,m,k,g,bits,symmetric,glu,ring", [
    ([11008], 48, 4096, 128, 4, True, False, True), ([11008], 48, 4096, 128, 4, False, False, True),
    ([11008], 56, 4096, 128, 4, True, False, True), ([11008], 56, 4096, 128, 4, False, False, True),
    ([11008], 64, 4096, 128, 4, True, False, True), ([11008], 64, 4096, 128, 4, False, False, True),
    ([11008], 64, 4096, 128, 8, True, False, True), ([8192], 64, 4096, 128, 4, True, False, False),  # two tiles a block
    ([9536], 44, 640, 64, 8, False, False, False), ([9536], 44, 1088, 64, 8, False, False, True),
    ([9536], 44, 640, 64, 4, False, False, True), ([12300], 44, 640, 64, 8, False, False, True),
    ([4096], 17, 4096, 128, 4, True, False, False), ([4096] * 3, 33, 4096, 32, 4, True, False, True),
    ([4096] * 2, 33, 4096, 32, 4, True, True, False), ([4352] * 2, 33, 4096, 32, 4, True, True, True)])
def test_three_tiles_of_rows_a_block_and_more_are_the_copying_waves(ns, m, k, g, bits, symmetric, glu, ring):
    for dtype in (_lib.F16, _lib.BF16):
        assert (ring_mt_plan(ns, m, k, g, bits, symmetric, dtype, glu) is not None) == ring, dtype


def test_the_shortest_expansion_stays_with_the_ring():
    """fp16 with 4-bit codes and no zero point, on blocks of whole 16-row tiles."""
    for ns, m, k in (([6949], 2, 5632), ([2176] * 3, 7, 2176), ([2176, 272, 272], 3, 2176)):
        assert ring_plan(ns, m, k, 64, 4, True, _lib.F16) is not None
        assert ring_plan(ns, m, k, 64, 4, True, _lib.BF16) is None


def _kernels(ns, m, k, g, glu=False):
    """What the variants of ring_tests run for one of its shapes; None stands for a kernel that is not a ring."""
    mode = "gated" if glu else "one" if len(ns) == 1 else "several"
    for bits, symmetric, _ in ring_tests.VARIANTS:
        for dtype in (_lib.F16, _lib.BF16):
            p = (ring_plan if m <= 16 else ring_mt_plan)(ns, m, k, g, bits, symmetric, dtype, glu)
            if p is None:
                yield None
            elif m <= 16:
                yield from ((p.tr, mode, p.tl), ("waves over K", 1 << p.wk_shift),
                            ("x in parts", p.tr, mode, p.phases > 1))
            else:
                yield from ((-(-m // 16), "tiles of x", mode, p.tl), ("workers over K", p.wk),
                            ("buffers", p.buffers), ("phases", min(p.phases, 3)))


def test_the_gpu_tests_run_every_ring_kernel():
    t, seen = ring_tests, set()
    for m, n, k, g in t.ONE + t.MANY_TILES:
        seen |= set(_kernels([n], m, k, g))
    for m, k, g, ns in t.SEVERAL + t.MANY_TILES_SEVERAL:
        seen |= set(_kernels(list(ns), m, k, g))
    for m, n, k, g in t.GATED + t.MANY_TILES_GATED:
        seen |= set(_kernels([n, n], m, k, g, True))
    modes = ("one", "several", "gated")
    want = {(tr, mode, tl) for tr in (8, 16) for mode in modes for tl in (1, 2, 3, 4)}
    want |= {("waves over K", 1 << s) for s in range(5)}
    want |= {("x in parts", tr, mode, parts) for tr in (8, 16) for mode in modes for parts in (False, True)}
    want |= {(mt, "tiles of x", mode, tl) for mt in (2, 3, 4) for mode in modes for tl in (1, 2, 3)}
    want |= {("workers over K", w) for w in (1, 2, 3, 4, 6, 12)}
    want |= {("buffers", b) for b in (2, 3, 4)} | {("phases", p) for p in (1, 2, 3)}
    assert want <= seen, sorted(want - seen, key=str)


def test_the_gpu_tests_of_many_tiles_run_the_copying_waves():
    t = ring_tests
    jobs = [([n], m, k, g, False) for m, n, k, g in t.MANY_TILES]
    jobs += [(list(ns), m, k, g, False) for m, k, g, ns in t.MANY_TILES_SEVERAL]
    jobs += [([n, n], m, k, g, True) for m, n, k, g in t.MANY_TILES_GATED]
    for job in jobs:
        assert None not in set(_kernels(*job)), job
