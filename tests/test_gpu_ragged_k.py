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


def _overflowing_weight(n, k, g, num_bits, symmetric, qdt, t, rng):
    """Codes around zero, and three rows in which a product code * scale overflows T:
      row 0  only if the codes of the row's last 128 elements met the scale of its first group
      row 1  in its first group, row 2 where its last 128 elements begin: the results are infinite"""
    signed = qdt == np.int8
    neutral = 0 if signed or not symmetric else 2 ** (num_bits - 1) - 1
    most = -2 ** (num_bits - 1) if signed else 2 ** num_bits - 1
    # (neutral + 1) * huge is finite, most * huge is not
    huge = {("f16", 4): (8000.0, 9000.0), ("f16", 8): (511.0, 515.0),
            ("bf16", 4): (4.2e37,), ("bf16", 8): (2.6e36,)}[t, num_bits][signed]
    codes = (neutral + rng.integers(-1 if symmetric else 0, 2, size=(n, k))).astype(qdt)
    scale = np.full((n, k // g), 0.01, np.float32)
    tail = (k - 1) // 128 * 128
    codes[:3] = neutral
    codes[0, 5] = neutral + 1
    codes[0, tail:] = most
    scale[0, 0] = huge
    codes[1, 7] = most
    scale[1, 0] = huge
    codes[2, tail + 3] = most
    scale[2, tail // g] = huge
    w = H.pack_int4(codes) if num_bits == 4 else codes
    zero = None if symmetric else H.as_T(np.zeros_like(scale), t)
    return w, H.as_T(scale, t), zero


@pytest.mark.parametrize("n,k,g", [(70, 288, 32), (33, 160, 32), (150, 2752, 64), (40, 9248, 32)])
@pytest.mark.parametrize("m", [1, 3, 16, 17, 40, 64, 65, 130, 300])
@pytest.mark.parametrize("t", ["f16", "bf16"])
def test_linear_ragged_k_overflowing_products(m, n, k, g, t):
    """What a kernel multiplies past the end of a row is zero whatever the weights hold: a finite
    result stays finite, an infinite one infinite (with NaN in neither)."""
    rng = np.random.Generator(np.random.PCG64(m * 13 + n + k))
    x = rng.uniform(0.25, 1.0, size=(m, k)) * rng.choice([-1.0, 1.0], size=(m, k))
    x = H.as_T(x.astype(np.float32), t)
    for num_bits, symmetric, qdt in VARIANTS:
        if t == "bf16" and qdt == np.int8:
            continue  # no product there overflows: 2^(b-1) * s has to be finite in fp32
        w, scale, zero = _overflowing_weight(n, k, g, num_bits, symmetric, qdt, t, rng)
        ref = O.to_f32(O.fused_linear(x, w, scale, zero, None, num_bits, symmetric, 1, g))
        assert np.isinf(ref[:, 1:3]).all() and np.isfinite(np.delete(ref, [1, 2], 1)).all()
        got = O.to_f32(_linear(x, w, scale, zero, None, num_bits, symmetric, g))
        what = f"{t} b{num_bits} m={m} n={n} k={k} {symmetric} {qdt}"
        assert np.array_equal(got[:, 1:3], ref[:, 1:3]), what
        # one product and sums of tiny ones in row 0: one rounding of T either way
        assert np.allclose(got[:, 0], ref[:, 0], rtol=2.0 ** (-9 if t == "f16" else -6), atol=0), what
        H.assert_linear_parity(H.as_T(got[:, 3:], t), H.as_T(ref[:, 3:], t), t, what)
