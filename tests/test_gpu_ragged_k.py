"""Rows whose length is not a whole number of a kernel's chunks (128 / 64 elements of codes in the
streaming kernels, 128 bytes of K in the GEMM), through every range of m: the part of the last chunk
past the end of a row must add nothing, whatever the neighbouring row holds."""
import numpy as np
import pytest

import helpers as H
from oracle import ofq_oracle as O

pytestmark = pytest.mark.gpu

VARIANTS = [(4, True, np.int8), (4, True, np.uint8), (4, False, np.uint8), (8, True, np.int8),
            (8, False, np.uint8)]


def _linear(x, w, scale, zero, b, num_bits, symmetric, g):
    import oneflow_amd as flow
    return H.to_numpy(flow._C.fused_linear_with_groupwise_quantized_weight(
        H.to_torch(x), H.to_torch(w), H.to_torch(scale), w_zero=H.to_torch(zero), b=H.to_torch(b),
        num_bits=num_bits, symmetric=symmetric, group_dim=1, group_size=g))


# 9 groups of 32 (a quarter of a chunk past 256), one short row, 43 groups of 64, long rows whose x
# does not fit LDS
@pytest.mark.parametrize("n,k,g", [(300, 288, 32), (33, 32, 32), (530, 2752, 64), (70, 9248, 32)])
@pytest.mark.parametrize("m", [1, 3, 16, 17, 33, 64, 65, 130, 300])
@pytest.mark.parametrize("t", ["f16", "bf16"])
def test_linear_ragged_k(m, n, k, g, t):
    rng = np.random.Generator(np.random.PCG64(m * 31 + n + k))
    x = H.as_T((rng.standard_normal((m, k)) / 2).astype(np.float32), t)
    wf = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    b = H.as_T((rng.standard_normal(n) * 0.01).astype(np.float32), t)
    for num_bits, symmetric, qdt in VARIANTS:
        w, scale, zero = H.quantize_groupwise(wf, num_bits, symmetric, 1, g, qdt, t)
        ref = O.fused_linear(x, w, scale, zero, b, num_bits, symmetric, 1, g)
        got = _linear(x, w, scale, zero, b, num_bits, symmetric, g)
        H.assert_linear_parity(got, ref, t, f"{t} b{num_bits} m={m} n={n} k={k} {symmetric} {qdt}")
        if m == 1:
            continue
        # rows next to one of NaN: the bytes that follow a row in memory take no part in its sums
        x2 = x.copy()
        x2[1] = np.float16(np.nan) if t == "f16" else np.uint16(0x7FC0)
        got2 = O.to_f32(_linear(x2, w, scale, zero, b, num_bits, symmetric, g))
        keep = np.arange(m) != 1
        assert np.array_equal(got2[keep], O.to_f32(got)[keep]) and np.isnan(got2[1]).all()


@pytest.mark.parametrize("m,n,k", [(1, 40, 288), (5, 70, 2752)])
@pytest.mark.parametrize("t", ["f16", "bf16"])
def test_grouped_linear_ragged_k(m, n, k, t):
    import oneflow_amd as flow
    g = 32
    rng = np.random.Generator(np.random.PCG64(m + n + k))
    x = H.as_T((rng.standard_normal((m, k)) / 2).astype(np.float32), t)
    packs = [H.quantize_groupwise((rng.standard_normal((rows, k)) * 0.05).astype(np.float32), 4, False,
                                  1, g, np.uint8, t) for rows in (n, 16, 3 * n)]
    got = flow._C.grouped_linear_with_groupwise_quantized_weight(
        [H.to_torch(x)] * 3, [H.to_torch(p[0]) for p in packs], [H.to_torch(p[1]) for p in packs],
        w_zeros=[H.to_torch(p[2]) for p in packs], num_bits=4, symmetric=False, group_dim=1,
        group_size=g)
    for out, (w, scale, zero) in zip(got, packs):
        H.assert_linear_parity(H.to_numpy(out), O.fused_linear(x, w, scale, zero, None, 4, False, 1, g),
                               t, "grouped")


def test_prefill_ragged_k_two_pass():
    """1030 rows: the weight is dequantised into the workspace and both operands are ragged."""
    m, n, k, g = 1030, 264, 608, 32
    rng = np.random.Generator(np.random.PCG64(7))
    x = H.as_T((rng.standard_normal((m, k)) / 2).astype(np.float32), "bf16")
    wf = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    w, scale, zero = H.quantize_groupwise(wf, 8, False, 1, g, np.uint8, "bf16")
    ref = O.fused_linear(x, w, scale, zero, None, 8, False, 1, g)
    H.assert_linear_parity(_linear(x, w, scale, zero, None, 8, False, g), ref, "bf16", "two-pass")


@pytest.mark.parametrize("m", [65, 200, 520, 800])
@pytest.mark.parametrize("n,k", [(264, 192), (1100, 4160), (130, 8256)])
def test_matmul_quant_ragged_k(m, n, k):
    import torch
    import oneflow_amd as flow
    rng = np.random.Generator(np.random.PCG64(m + n + k))
    a = rng.integers(-128, 128, size=(m, k)).astype(np.int8)
    b = rng.integers(-128, 128, size=(n, k)).astype(np.int8)
    a_scale = np.array([0.0317], np.float32)
    b_scale = rng.uniform(1e-3, 1e-2, size=n).astype(np.float32)
    got = H.to_numpy(flow._C.matmul_quant(H.to_torch(a), H.to_torch(b), H.to_torch(a_scale),
                                          H.to_torch(b_scale), None, torch.float16))
    acc = a.astype(np.float64) @ b.astype(np.float64).T
    assert np.array_equal(got, (acc.astype(np.float32) * (a_scale[0] * b_scale)[None]).astype(np.float16))
