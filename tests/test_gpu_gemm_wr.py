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


# 32 x 128 alone (1, 31 and 32 rows in the last tile; 2 columns) and with slices, 64 x 128 (1 row),
# 96 x 128 (1 and 96 rows), 128 x 256 with 212 columns
@pytest.mark.parametrize("m,n,k,g", [(65, 130, 640, 32), (95, 700, 512, 128), (96, 127, 96, 96),
                                     (24, 600, 4640, 32), (129, 257, 4096, 64), (129, 9000, 160, 32),
                                     (193, 9000, 160, 160), (192, 1001, 2112, 32), (100, 16600, 320, 64)])
@pytest.mark.parametrize("t", ["f16", "bf16"])
def test_tiles(m, n, k, g, t):
    for num_bits, symmetric, qdt in VARIANTS:
        _check(m, n, k, g, t, num_bits, symmetric, qdt)


# 192 x 256 with a last tile of 161 rows by 20 columns; rows of so many short groups that the scales and
# zeros of a block (1 KB a group) do not fit LDS at a time
@pytest.mark.parametrize("m,n,k,g", [(545, 14100, 224, 32), (33, 16500, 7200, 32)])
def test_tall_tiles_and_panels(m, n, k, g):
    _check(m, n, k, g, "f16", 4, False, np.uint8)
