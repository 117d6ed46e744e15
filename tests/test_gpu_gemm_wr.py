"""The GEMM that expands weights in the registers of the wave that multiplies them: a shape for each of
its tiles of rows of x by columns, alone and with slices of K, with partial last tiles in both
directions, a last step of K that is not full, and scales that take several panels."""
import numpy as np
import pytest

import helpers as H
from oracle import ofq_oracle as O

pytestmark = pytest.mark.gpu

VARIANTS = [(4, True, np.int8), (4, True, np.uint8), (4, False, np.uint8), (8, True, np.int8),
            (8, True, np.uint8), (8, False, np.uint8)]


def _check(m, n, k, g, t, num_bits, symmetric, qdt):
    import oneflow_amd as flow
    rng = np.random.Generator(np.random.PCG64(m * 5 + n + k))
    x = H.as_T((rng.standard_normal((m, k)) / 2).astype(np.float32), t)
    wf = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    b = H.as_T((rng.standard_normal(n) * 0.01).astype(np.float32), t)
    w, scale, zero = H.quantize_groupwise(wf, num_bits, symmetric, 1, g, qdt, t)
    got = H.to_numpy(flow._C.fused_linear_with_groupwise_quantized_weight(
        H.to_torch(x), H.to_torch(w), H.to_torch(scale), w_zero=H.to_torch(zero), b=H.to_torch(b),
        num_bits=num_bits, symmetric=symmetric, group_dim=1, group_size=g))
    ref = O.fused_linear(x, w, scale, zero, b, num_bits, symmetric, 1, g)
    H.assert_linear_parity(got, ref, t, f"{t} b{num_bits} m={m} n={n} k={k} {symmetric} {qdt}")


# whatever the dispatch chooses: 1, 31 and 32 rows beyond whole tiles, 1 or 2 columns, steps of K that
# are not full, with and without slices (each tile by name: test_every_tile_alone_and_sliced)
@pytest.mark.parametrize("m,n,k,g", [(65, 130, 640, 32), (95, 700, 512, 128), (96, 127, 96, 96),
                                     (24, 600, 4640, 32), (129, 257, 4096, 64), (129, 9000, 160, 32),
                                     (193, 9000, 160, 160), (192, 1001, 2112, 32), (100, 16600, 320, 64)])
@pytest.mark.parametrize("t", ["f16", "bf16"])
def test_tiles(m, n, k, g, t):
    for num_bits, symmetric, qdt in VARIANTS:
        _check(m, n, k, g, t, num_bits, symmetric, qdt)


# large outputs with 33 and 20 columns beyond whole tiles; rows of so many short groups that the scales
# and zeros of a block of 128 x 256 (1 KB a group) do not fit LDS at a time
@pytest.mark.parametrize("m,n,k,g", [(545, 14100, 224, 32), (33, 16500, 7200, 32)])
def test_tall_tiles_and_panels(m, n, k, g):
    _check(m, n, k, g, "f16", 4, False, np.uint8)


@pytest.mark.parametrize("tile", range(5))
@pytest.mark.parametrize("k", [320, 416, 1024])
@pytest.mark.parametrize("slices", [1, 2, 3])
@pytest.mark.parametrize("t", ["f16", "bf16"])
def test_every_tile_alone_and_sliced(tile, k, slices, t):
    """Each tile whatever the dispatch prefers: a last tile of one row by 33 columns, steps of 64 and 128
    that K fills (1024), fills in part (320 for steps of 128) and never fills (416), one slice of K
    and a last slice shorter than the others."""
    import ctypes

    import torch
    from oneflow_amd import _lib
    from test_gemm_plan import TILES, LinearArgs, WrPlan
    bm, bn = TILES[tile]
    steps = -(-k // (128 if bn == 128 else 64))
    per = -(-steps // slices)
    slices = -(-steps // per)  # no empty last slice
    m, n, g = bm + 1, bn + 33, 32
    launch = _lib.lib()[f"_ZN3ofq{15 + len(t)}launch_gemm_wr_{t}"
                        "EP12ihipStream_tRKNS_10LinearArgsERKNS_6WrPlanEPf"]
    launch.argtypes = [ctypes.c_void_p, ctypes.POINTER(LinearArgs), ctypes.POINTER(WrPlan),
                       ctypes.c_void_p]
    rng = np.random.Generator(np.random.PCG64(tile * 100 + k + slices))
    x = H.as_T((rng.standard_normal((m, k)) / 2).astype(np.float32), t)
    wf = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    b = H.as_T((rng.standard_normal(n) * 0.01).astype(np.float32), t)
    partials = torch.empty(slices * -(-m // 32) * -(-n // 32) * 1024, device="cuda")
    for num_bits, symmetric, qdt in VARIANTS:
        if num_bits == 8 and tile in (2, 4):
            continue  # 4-bit codes only
        w, scale, zero = H.quantize_groupwise(wf, num_bits, symmetric, 1, g, qdt, t)
        on_gpu = [H.to_torch(a) for a in (x, w, scale, zero, b)]
        out = torch.empty((m, n), dtype=on_gpu[0].dtype, device="cuda")
        args = LinearArgs(*[a.data_ptr() if a is not None else None for a in on_gpu], out.data_ptr(),
                          _lib.F16 if t == "f16" else _lib.BF16, qdt == np.int8, num_bits, symmetric, 1,
                          g, m, n, k)
        rc = launch(torch.cuda.current_stream().cuda_stream, ctypes.byref(args),
                    ctypes.byref(WrPlan(tile, slices)), partials.data_ptr())
        assert rc == 0
        ref = O.fused_linear(x, w, scale, zero, b, num_bits, symmetric, 1, g)
        H.assert_linear_parity(H.to_numpy(out), ref, t, f"tile {tile} {t} b{num_bits} k={k} x{slices}")
