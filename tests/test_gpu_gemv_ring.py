"""The streaming kernels for one linear, several and a gated unit.  Up to 16 rows of x, the one whose operands
all come by counted copies: tiles of 8 and 16 rows with partial last ones, one to four of them a wave, rows of K that
end inside a chunk and inside a step, groups that are not powers of two, scale arrays that end inside a 16-byte piece,
every split of the waves over tiles and K, and x that passes LDS whole and in parts.  17 to 64 rows: two, three and
four tiles of x, one to three tiles of rows a wave, every split of the workers, two to four buffers of x.  Which
kernel each shape runs, and that together they run every kernel there is: test_stream_plan.py.

|result - exact| <= one rounding to the dtype + (k + 2) fp32 roundings of the running sum of |x| |w~|, and w~ is
formed exactly as groupwise_dequantize forms it."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
VARIANTS = [(4, True, torch.int8), (4, True, torch.uint8), (4, False, torch.uint8), (8, True, torch.int8),
            (8, True, torch.uint8), (8, False, torch.uint8)]


def _weight(gen, n, k, g, bits, symmetric, qdt, dtype):
    lo = -128 if qdt == torch.int8 else 0
    w = torch.randint(lo, lo + 256, (n, k * bits // 8), generator=gen, device="cuda", dtype=qdt)
    scale = (torch.rand(n, k // g, generator=gen, device="cuda") * 0.02 + 1e-3).to(dtype)
    zero = None if symmetric else (torch.randn(n, k // g, generator=gen, device="cuda") * 0.1).to(dtype)
    return w, scale, zero, torch.randn(n, generator=gen, device="cuda").to(dtype)


def _exact(x, weight, g, bits, symmetric):
    import oneflow_amd as flow
    w, scale, zero, bias = weight
    full = flow._C.groupwise_dequantize(w, scale, zero=zero, num_bits=bits, symmetric=symmetric, group_dim=1,
                                        group_size=g).double()
    bound = x.double().abs() @ full.abs().T + bias.double().abs()
    return x.double() @ full.T + bias.double(), bound


def _check(out, x, weight, g, bits, symmetric, what):
    ref, mass = _exact(x, weight, g, bits, symmetric)
    bound = EPS[x.dtype] * ref.abs() + (x.shape[1] + 2) * 2.0 ** -24 * mass + 2.0 ** -24
    assert bool(((out.double() - ref).abs() <= bound).all()), what


# blocks of more than 16 rows, short blocks on long rows, x in three parts and more
ONE = [(2, 4100, 1184, 32), (8, 5001, 480, 96), (7, 4129, 2784, 32), (9, 4353, 544, 32), (16, 8200, 320, 64),
       (3, 9001, 160, 160), (5, 30011, 128, 64), (2, 1031, 8224, 32), (1, 4111, 4160, 32), (16, 4200, 3616, 32),
       (8, 4300, 11296, 32), (6, 7354, 2720, 32), (15, 8308, 2880, 64), (9, 13707, 3968, 128), (16, 5309, 4224, 64),
       (13, 11247, 4192, 32), (10, 5925, 5088, 32), (15, 15095, 1664, 64), (4, 14747, 11008, 64)]


@pytest.mark.parametrize("m,n,k,g", ONE)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_one(m, n, k, g, dtype):
    import oneflow_amd as flow
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    for bits, symmetric, qdt in VARIANTS:
        weight = _weight(gen, n, k, g, bits, symmetric, qdt, dtype)
        out = flow._C.fused_linear_with_groupwise_quantized_weight(
            x, weight[0], weight[1], w_zero=weight[2], b=weight[3], num_bits=bits, symmetric=symmetric,
            group_dim=1, group_size=g)
        _check(out, x, weight, g, bits, symmetric, (m, n, k, g, bits, symmetric, qdt, dtype))


# 17 to 64 rows of x and three tiles of rows a block or more: two, three and four tiles of x with partial last ones,
# one to three tiles of rows a wave, two to four buffers of x, one to eight phases with K ending inside them
MANY_TILES = [(31, 21517, 1184, 32), (20, 30011, 544, 32), (48, 17003, 1184, 32), (33, 28100, 480, 96),
              (64, 20999, 1056, 32), (49, 9001, 2208, 32), (64, 32003, 96, 32), (64, 11008, 4096, 128),
              (41, 9821, 1184, 32), (28, 8988, 1152, 128), (18, 10203, 1056, 96), (33, 11963, 3456, 128)]


@pytest.mark.parametrize("m,n,k,g", MANY_TILES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_many_tiles(m, n, k, g, dtype):
    test_one(m, n, k, g, dtype)


MANY_TILES_SEVERAL = [(40, 2016, 32, (16000, 40)), (64, 1184, 32, (9000, 2200, 2200)), (40, 2048, 128, (8988, 10, 44)),
                      (25, 1920, 128, (8365, 380, 244)), (29, 320, 64, (7973, 1546, 417)),
                      (49, 288, 32, (14144, 1152, 1176)), (34, 3328, 64, (3328, 3328, 3328))]


@pytest.mark.parametrize("m,k,g,ns", MANY_TILES_SEVERAL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_many_tiles_several(m, k, g, ns, dtype):
    test_several(m, k, g, ns, dtype)


MANY_TILES_GATED = [(32, 9001, 1184, 32), (33, 11003, 480, 96), (48, 6001, 2208, 32), (64, 14001, 544, 32),
                    (49, 9001, 1056, 32), (20, 30000, 160, 32), (33, 8433, 864, 96)]


@pytest.mark.parametrize("m,n,k,g", MANY_TILES_GATED)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_many_tiles_gated_unit(m, n, k, g, dtype):
    test_gated_unit(m, n, k, g, dtype)


def test_many_tiles_an_infinite_x_stays_in_its_row():
    import oneflow_amd as flow
    gen = torch.Generator(device="cuda").manual_seed(4)
    m, n, k, g = 49, 9001, 2208, 32
    x = torch.randn(m, k, generator=gen, device="cuda").half()
    w, scale, _, bias = _weight(gen, n, k, g, 4, True, torch.int8, torch.float16)
    run = lambda a: flow._C.fused_linear_with_groupwise_quantized_weight(  # noqa: E731
        a, w, scale, b=bias, num_bits=4, symmetric=True, group_dim=1, group_size=g)
    plain = run(x)
    x2 = x.clone()
    x2[48, k - 1] = float("inf")
    out = run(x2)
    assert torch.equal(out[:48], plain[:48])
    assert not bool(torch.isfinite(out[48][(w[:, -1] & 15) != 0]).any())


SEVERAL = [(1, 96, 32, (7, 1, 300)), (5, 1696, 32, (1111, 139, 139)), (8, 4128, 96, (4096, 17, 9)),
           (9, 736, 32, (515, 16, 33)), (17, 1696, 32, (1111, 139, 139)), (33, 1184, 32, (4097, 9, 1030)),
           (64, 544, 32, (9000, 2200)), (49, 224, 32, (16000, 40)), (40, 480, 96, (300, 301, 5)),
           (16, 1568, 32, (9000, 2)), (16, 64, 32, (40, 4099, 17)), (4, 11040, 32, (700, 300)),
           (6, 1920, 128, (6449, 519, 936)), (16, 1280, 64, (2614, 461, 1470)), (7, 2400, 96, (6563, 25, 29)),
           (16, 4512, 96, (5770, 261, 297)), (7, 9152, 32, (5164, 353, 283)), (15, 544, 32, (10861, 694, 769)),
           (11, 4224, 32, (4224, 1056, 1056))]


@pytest.mark.parametrize("m,k,g,ns", SEVERAL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_several(m, k, g, ns, dtype):
    import oneflow_amd as flow
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    for bits, symmetric, qdt in VARIANTS:
        ws = [_weight(gen, n, k, g, bits, symmetric, qdt, dtype) for n in ns]
        outs = flow._C.grouped_linear_with_groupwise_quantized_weight(
            [x] * len(ns), [w[0] for w in ws], [w[1] for w in ws],
            w_zeros=None if symmetric else [w[2] for w in ws], bs=[w[3] for w in ws], num_bits=bits,
            symmetric=symmetric, group_dim=1, group_size=g)
        for out, w in zip(outs, ws):
            _check(out, x, w, g, bits, symmetric, (m, k, g, ns, bits, symmetric, qdt, dtype))


GATED = [(1, 37, 96, 32), (2, 700, 1184, 32), (8, 4671, 480, 96), (7, 9001, 224, 32), (9, 1030, 1568, 32),
         (16, 11008, 160, 32), (8, 300, 11040, 32), (4, 30000, 64, 64), (17, 1030, 1184, 32), (32, 5021, 480, 96),
         (33, 37, 2208, 32), (48, 9001, 160, 32), (49, 2700, 544, 32), (64, 14001, 96, 32), (14, 326, 4224, 96),
         (8, 3970, 2208, 96), (14, 6434, 2944, 128), (8, 5654, 1408, 128), (15, 8683, 288, 32), (14, 5248, 1792, 64),
         (12, 12224, 3968, 64)]


@pytest.mark.parametrize("m,n,k,g", GATED)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gated_unit(m, n, k, g, dtype):
    """Both linears and y = hidden * relu(gate), whose only roundings are the two of T; nothing past the outputs."""
    from oneflow_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    code = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}[dtype]
    for bits, symmetric, qdt in VARIANTS:
        w = _weight(gen, n, k, g, bits, symmetric, qdt, dtype)
        v = _weight(gen, n, k, g, bits, symmetric, qdt, dtype)
        outs = [torch.full((m * n + 64,), 777.0, device="cuda", dtype=dtype) for _ in range(3)]
        ptr = lambda a: None if a is None else a.data_ptr()  # noqa: E731
        rc = _lib.lib().ofq_fused_glu_gq(
            torch.cuda.current_stream().cuda_stream, ptr(x), *map(ptr, w), *map(ptr, v), *map(ptr, outs), 2,
            _lib.I8 if qdt == torch.int8 else _lib.U8, code, bits, int(symmetric), 1, g, m, n, k)
        assert rc == 0
        what = (m, n, k, g, bits, symmetric, qdt, dtype)
        y, hidden, gate = (o[:m * n].view(m, n) for o in outs)
        _check(hidden, x, w, g, bits, symmetric, what)
        _check(gate, x, v, g, bits, symmetric, what)
        assert torch.equal(y, hidden * gate.clamp(min=0)), what
        assert all(bool((o[m * n:] == 777).all()) for o in outs), what


def test_an_infinite_x_stays_in_its_row():
    """The last chunk of a ragged row meets zeros, not a neighbour's values: an infinity in one row of x does not
    reach the others, and in its own row nothing but infinities and NaN come of it."""
    import oneflow_amd as flow
    gen = torch.Generator(device="cuda").manual_seed(3)
    m, n, k, g = 3, 4500, 160, 32
    x = torch.randn(m, k, generator=gen, device="cuda").half()
    w, scale, _, bias = _weight(gen, n, k, g, 4, True, torch.int8, torch.float16)
    run = lambda a: flow._C.fused_linear_with_groupwise_quantized_weight(  # noqa: E731
        a, w, scale, b=bias, num_bits=4, symmetric=True, group_dim=1, group_size=g)
    plain = run(x)
    x2 = x.clone()
    x2[1, 0] = float("inf")
    out = run(x2)
    assert torch.equal(out[0], plain[0]) and torch.equal(out[2], plain[2])
    assert not bool(torch.isfinite(out[1][w[:, 0] < 16]).all())
