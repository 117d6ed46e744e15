"""The work that users of this package have it do, as cases that can be timed and compared.

A case is a dict of plain values; ``prepare`` makes what a program holds before the call (inputs,
quantised weights, modules, a captured step), ``run`` is one pass through the public entry points.
Five kinds of use:

  linear   one ``nn.QuantizedLinear``: a token, a serving batch, a prompt (m rows of x)
  layer    the quantised linears of decoder layers as modules: q/k/v grouped, o, gate/up as a GLU,
           down; called directly, or replayed from a HIP graph as a serving loop does
  int8     dynamic int8: LayerNorm (+ residual) -> codes -> ``matmul_quant``
  qat      a quantization-aware convolution's observers and fake quantisation, and their gradients
  weight   a weight quantised into the packed format and read back

Ranges (``draw``): 1 to 4096 rows of x (to 8192 for int8, to 64 in a decoder layer), weights of 512 to 32000 rows
and 512 to 14336 columns with any number of rows and any number of whole groups (tensor-parallel
shards and vocabularies give ragged ones), 4- and 8-bit codes with and without a zero point,
groups of 32, 64 and 128 along k, fp16 and bf16; activations of a convolution from 0.1 to 32
million elements in fp32.
"""
import math

import torch

import oneflow_amd as flow

_DTYPE = {"f16": torch.float16, "bf16": torch.bfloat16}
# no drawn case costs more than the largest listed one (int8_prompt)
_MOST_MACS = 4096 * 11008 * 4096
_MOST_LAYER_BYTES = 430 << 20
_MOST_WEIGHT = 120 << 20


def _linear(m, n, k, dtype, bits, symmetric, group, bias):
    return {"kind": "linear", "m": m, "n": n, "k": k, "dtype": dtype, "bits": bits,
            "symmetric": symmetric, "group": group, "bias": bias}


def _layer(layers, m, hidden, kv, inter, dtype, bits, symmetric, group, graph):
    return {"kind": "layer", "layers": layers, "m": m, "hidden": hidden, "kv": kv, "inter": inter,
            "dtype": dtype, "bits": bits, "symmetric": symmetric, "group": group, "graph": graph}


def _int8(m, n, k, dtype, skip, bias):
    return {"kind": "int8", "m": m, "n": n, "k": k, "dtype": dtype, "skip": skip, "bias": bias}


def _qat(batch, channels, size, out_channels, scheme, per_layer):
    return {"kind": "qat", "batch": batch, "channels": channels, "size": size,
            "out_channels": out_channels, "scheme": scheme, "per_layer": per_layer}


def _weight(n, k, dtype, bits, symmetric, group):
    return {"kind": "weight", "n": n, "k": k, "dtype": dtype, "bits": bits,
            "symmetric": symmetric, "group": group}


def listed():
    return [
        # the smallest call there is: one token through one projection, called from Python
        dict(_linear(1, 4096, 4096, "f16", 4, True, 128, False), name="linear_token"),
        # one token through a decoder layer, module by module: generation without a graph
        dict(_layer(1, 1, 4096, 4096, 11008, "f16", 4, True, 128, False), name="layer_token"),
        # the same work in a serving loop that replays its captured step, four layers of it
        dict(_layer(4, 1, 4096, 4096, 11008, "f16", 4, True, 128, True), name="step_token_graph"),
        # eight sequences decoded together, captured
        dict(_layer(4, 8, 4096, 4096, 11008, "f16", 4, True, 128, True), name="step_batch_graph"),
        # a quarter of a down projection (tensor parallel over four: 43 groups of 64 columns) with
        # a few sequences, bf16 with a zero point
        dict(_linear(5, 4096, 2752, "bf16", 4, False, 64, False), name="linear_shard"),
        # a full serving batch
        dict(_linear(48, 11008, 4096, "f16", 4, False, 128, True), name="linear_serving"),
        # a short prompt of odd length through the longest rows
        dict(_linear(333, 4096, 11008, "f16", 4, True, 128, False), name="linear_prompt_short"),
        # a long prompt in bf16 with 8-bit codes and a zero point
        dict(_linear(2048, 11008, 4096, "bf16", 8, False, 64, False), name="linear_prompt_long"),
        # dynamic int8 with a residual for a handful of tokens
        dict(_int8(7, 11008, 4096, "f16", True, True), name="int8_tokens"),
        # dynamic int8 for long prompts: the largest case
        dict(_int8(8192, 11008, 4096, "f16", False, False), name="int8_prompt"),
        # a convolution of a network trained with quantization in mind, forward and backward
        dict(_qat(32, 64, 56, 128, "symmetric", False), name="qat_conv"),
        # a weight packed to 4 bits when a model is converted, and read back
        dict(_weight(11008, 4096, "f16", 4, True, 128), name="weight_roundtrip"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _whole(value, step):
    return max(step, value // step * step)


def draw(rng):
    kind = rng.choice(["linear"] * 4 + ["layer"] * 3 + ["int8"] * 2 + ["qat", "weight"])
    dtype = rng.choice(["f16", "f16", "bf16"])
    bits, symmetric = rng.choice([4, 4, 8]), rng.choice([True, False])
    group = rng.choice([32, 64, 128, 128])
    if kind == "linear":
        n, k = _log_int(rng, 512, 32000), _whole(_log_int(rng, 512, 14336), group)
        m = min(_log_int(rng, 1, 4096), _MOST_MACS // (n * k))
        return _linear(m, n, k, dtype, bits, symmetric, group, rng.choice([True, False]))
    if kind == "layer":
        hidden = _whole(_log_int(rng, 1024, 5120), 128)
        inter = _whole(int(hidden * rng.uniform(2.5, 3.6)), group)
        kv = hidden // rng.choice([1, 4, 8])
        m, graph = _log_int(rng, 1, 64), rng.choice([True, False])
        one = _layer(1, m, hidden, kv, inter, dtype, bits, symmetric, group, graph)
        most = min(4, _MOST_LAYER_BYTES // work(one)["bytes"], 128 // m)
        return dict(one, layers=rng.randint(1, most))
    if kind == "int8":
        n, k = _log_int(rng, 512, 14336), _whole(_log_int(rng, 512, 8192), 64)
        m = min(_log_int(rng, 1, 8192), _MOST_MACS // (n * k))
        return _int8(m, n, k, dtype, rng.choice([True, False]), rng.choice([True, False]))
    if kind == "qat":
        channels, size = rng.choice([16, 32, 48, 64, 96, 128, 256]), rng.choice([7, 14, 28, 56, 112])
        batch = max(1, _log_int(rng, 100000, 32000000) // (channels * size * size))
        return _qat(batch, channels, size, rng.choice([32, 64, 96, 128, 256]),
                    rng.choice(["symmetric", "affine"]), rng.choice([True, False]))
    k = _whole(_log_int(rng, 512, 14336), group)
    n = _log_int(rng, 512, min(32000, _MOST_WEIGHT // k))
    return _weight(n, k, dtype, bits, symmetric, group)


def _normal(gen, shape, std=1.0, dtype=torch.float32):
    return (torch.randn(shape, device="cuda", generator=gen) * std).to(dtype)


def _quantized_linear(gen, n, k, case, bias=False):
    """A dense linear's weights (std 1/sqrt(k), as trained layers have) in the packed format."""
    dtype = _DTYPE[case["dtype"]]
    dense = torch.nn.utils.skip_init(torch.nn.Linear, k, n, bias=bias, device="cuda", dtype=dtype)
    with torch.no_grad():
        dense.weight.copy_(_normal(gen, (n, k), k ** -0.5))
        if bias:
            dense.bias.copy_(_normal(gen, (n,), 0.02))
    return flow.nn.QuantizedLinear.from_float(
        dense, num_bits=case["bits"], symmetric=case["symmetric"], group_size=case["group"],
        quant_type=torch.int8 if case["symmetric"] else torch.uint8)


class _DecoderLayer:
    """The quantised linears of a decoder layer; what lies between them (attention, norms) is the
    user's own, its result `attended` stands for it."""

    def __init__(self, gen, case):
        h, kv, inter = case["hidden"], case["kv"], case["inter"]
        lin = lambda n, k: _quantized_linear(gen, n, k, case)  # noqa: E731
        self.qkv = flow.nn.GroupedQuantizedLinear([lin(h, h), lin(kv, h), lin(kv, h)])
        self.o = lin(h, h)
        self.glu = flow.nn.QuantizedGLU(lin(inter, h), lin(inter, h), activation="silu")
        self.down = lin(h, inter)

    def __call__(self, x, attended):
        q, k, v = self.qkv(x)
        o = self.o(attended)
        return q, k, v, o, self.down(self.glu(o))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "linear":
        module = _quantized_linear(gen, case["n"], case["k"], case, case["bias"])
        return {"kind": kind, "module": module,
                "x": _normal(gen, (case["m"], case["k"]), dtype=_DTYPE[case["dtype"]])}
    if kind == "layer":
        layers = [_DecoderLayer(gen, case) for _ in range(case["layers"])]
        xs = [_normal(gen, (2, case["m"], case["hidden"]), dtype=_DTYPE[case["dtype"]])
              for _ in layers]
        step = lambda: [layer(x[0], x[1]) for layer, x in zip(layers, xs)]  # noqa: E731
        if not case["graph"]:
            return {"kind": kind, "step": step}
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = step()
        return {"kind": kind, "graph": graph, "out": out, "keep": (layers, xs)}
    if kind == "int8":
        m, n, k, dtype = case["m"], case["n"], case["k"], _DTYPE[case["dtype"]]
        w = _normal(gen, (n, k), k ** -0.5)
        w_scale = w.abs().amax(1) / 127
        return {"kind": kind, "dtype": dtype, "x": _normal(gen, (m, k), dtype=dtype),
                "gamma": (1 + _normal(gen, (k,), 0.1)).to(dtype),
                "beta": _normal(gen, (k,), 0.1, dtype),
                "skip": _normal(gen, (m, k), dtype=dtype) if case["skip"] else None,
                "pre_bias": _normal(gen, (k,), 0.1, dtype) if case["skip"] else None,
                "w": (w / w_scale[:, None]).round().to(torch.int8), "w_scale": w_scale,
                "bias": _normal(gen, (n,), 0.02, dtype) if case["bias"] else None}
    if kind == "qat":
        shape = (case["batch"], case["channels"], case["size"], case["size"])
        conv = flow.qat.QatConv2d(case["channels"], case["out_channels"], 3, padding=1, bias=False,
                                  quantization_scheme=case["scheme"],
                                  weight_quant_per_layer=case["per_layer"]).cuda()
        with torch.no_grad():
            conv.weight.copy_(_normal(gen, conv.weight.shape, (9 * case["channels"]) ** -0.5))
        x = _normal(gen, shape).relu_().requires_grad_()  # behind a ReLU, as in such networks
        return {"kind": kind, "conv": conv, "x": x, "grad_x": _normal(gen, shape, 1e-3),
                "grad_w": _normal(gen, conv.weight.shape, 1e-3)}
    w = _normal(gen, (case["n"], case["k"]), case["k"] ** -0.5, _DTYPE[case["dtype"]])
    return {"kind": kind, "w": w, "bits": case["bits"], "symmetric": case["symmetric"],
            "group": case["group"]}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["module"](state["x"])
    if kind == "layer":
        if "graph" not in state:
            return state["step"]()
        state["graph"].replay()
        return state["out"]
    if kind == "int8":
        x, gamma, beta = state["x"], state["gamma"], state["beta"]
        if state["skip"] is None:
            codes, scale, _ = flow._C.fused_layer_norm_quantization(x, gamma, beta)
        else:
            y, scale, zero = flow._C.fused_skip_layer_norm_min_max_observer(
                x, gamma, beta, state["pre_bias"], state["skip"], alpha=1.0)
            codes = flow._C.quantization(y, scale, zero, out_dtype=torch.int8)
        out = flow._C.matmul_quant(codes, state["w"], scale, state["w_scale"], state["bias"],
                                   out_dtype=state["dtype"])
        return codes, scale, out
    if kind == "qat":
        conv, x = state["conv"], state["x"]
        fake_x, fake_w = flow.qat.get_conv_fake_quantized(
            x, conv.input_min_max_observer, conv.current_train_step, conv.weight,
            conv.weight_min_max_observer, conv.fake_quantizer)
        grads = torch.autograd.grad((fake_x, fake_w), (x, conv.weight),
                                    (state["grad_x"], state["grad_w"]))
        observer = conv.input_min_max_observer
        return fake_x.detach(), fake_w.detach(), grads, observer.moving_max, observer.moving_min
    codes, scale, zero = flow.quantize.groupwise_quantize(
        state["w"], num_bits=state["bits"], symmetric=state["symmetric"], group_dim=1,
        group_size=state["group"], quant_type=torch.int8 if state["symmetric"] else torch.uint8)
    back = flow._C.groupwise_dequantize(codes, scale, zero=zero, num_bits=state["bits"],
                                        symmetric=state["symmetric"], group_dim=1,
                                        group_size=state["group"])
    return codes, scale, zero, back


def _packed_bytes(n, k, case, size=2):
    groups = n * (k // case["group"]) * size * (1 if case["symmetric"] else 2)
    return n * k * case["bits"] // 8 + groups


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _packed_bytes(n, k, case) + 2 * (m * k + m * n + n * case["bias"]),
                "flops": 2 * m * n * k}
    if kind == "layer":
        m, h, kv, inter = case["m"], case["hidden"], case["kv"], case["inter"]
        shapes = [(h, h), (kv, h), (kv, h), (h, h), (inter, h), (inter, h), (h, inter)]
        # x, attended, q, k, v, o and the result; what stays inside the layer (the GLU's result)
        # is counted as one write and one read
        values = m * (5 * h + 2 * kv + 2 * inter)
        return {"bytes": case["layers"] * (sum(_packed_bytes(n, k, case) for n, k in shapes)
                                           + 2 * values),
                "flops": case["layers"] * 2 * m * sum(n * k for n, k in shapes)}
    if kind == "int8":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": m * k * (5 if case["skip"] else 3) + n * k + 4 * n + 2 * m * n + 2 * k
                * (3 if case["skip"] else 2) + 2 * n * case["bias"], "flops": 2 * m * n * k}
    if kind == "qat":
        x = case["batch"] * case["channels"] * case["size"] ** 2
        w = case["out_channels"] * case["channels"] * 9
        return {"bytes": 8 * (x + w), "flops": 8 * (x + w)}
    n, k = case["n"], case["k"]
    return {"bytes": 4 * n * k + _packed_bytes(n, k, case), "flops": 8 * n * k}


def tolerance(case):
    """Whole linears in fp16 / bf16: the rounding of the result and, where an implementation may
    leave it out, of the expanded weights; a chain of them in a layer.  Observers, codes and fake
    quantisation carry the same bits whatever the order of evaluation, except that the row
    statistics of a LayerNorm (fp32 sums) may move a value across a rounding boundary."""
    kind = case["kind"]
    if kind in ("qat", "weight"):
        return "exact"
    rel = {"f16": 1e-3, "bf16": 6e-3}[case["dtype"]]
    if kind == "layer":
        rel *= 1.5
    if kind == "int8":
        return {"rel": rel, "differ": 2e-4}
    return {"rel": rel}
