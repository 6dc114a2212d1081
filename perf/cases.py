"""Workloads of the quantized linear path, as programs run it.

A case names one of five programs, its sizes, its quantization mode and its
16-bit type:

  decoder   the projections of decoder layers in the order a decoder calls
            them: RMSNorm -> codes, qkv; the quantized linear o_proj on the
            attention output (made here, attention is outside the path);
            residual + RMSNorm -> codes, gate_up; SiLU gate -> codes, down.
  encoder   the feed-forward half of encoder layers: LayerNorm -> codes, a
            projection with bias and tanh-GeLU, quantization, a projection
            back, bias + residual.
  linear    one quantized linear on 16-bit rows: quantize, then the GEMM.
  project   a stack of small LayerNorm -> projection calls (hidden <= 512).
  quantize  the row quantizer: weights at load time, activations per call.

`captured` programs keep one HIP graph per shape, as a server does for its
decode steps and for prompt lengths that come again: the graph is made once in
prepare() and a pass replays it. The others call the library eagerly.

A stack's layers have distinct weights, so that a pass reads them from HBM as
a model's step does, and each starts from a hidden state of its own: a value
that rounds the other way stays in its layer instead of moving the codes of
all that follow.
"""
import math

import torch

from breeze_tts_cpp_amd import qlinear

# mode -> (code format, K group, H128 rotation)
MODES = {"int8": (qlinear.I8, 0, 0), "fp8": (qlinear.FP8, 0, 0),
         "group_int8": (qlinear.I8, 128, 128), "group_fp8": (qlinear.FP8, 128, 128)}
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
EPS = 1e-5


def _decoder(rows, mode, layers, captured, dtype="bf16", hidden=2048, qkv=4096, inter=6144):
    return {"kind": "decoder", "rows": rows, "mode": mode, "layers": layers, "captured": captured,
            "dtype": dtype, "hidden": hidden, "qkv": qkv, "inter": inter}


def _encoder(rows, mode, layers, captured, dtype="f16", hidden=1024, inter=4096):
    return {"kind": "encoder", "rows": rows, "mode": mode, "layers": layers, "captured": captured,
            "dtype": dtype, "hidden": hidden, "inter": inter}


def _project(rows, mode, layers, dtype="bf16", k=512, n=2048):
    return {"kind": "project", "rows": rows, "mode": mode, "layers": layers, "captured": True,
            "dtype": dtype, "k": k, "n": n}


def _linear(rows, mode, N, K, dtype="bf16"):
    return {"kind": "linear", "rows": rows, "mode": mode, "captured": False, "dtype": dtype,
            "N": N, "K": K}


def _quantize(rows, mode, cols, dtype="bf16"):
    return {"kind": "quantize", "rows": rows, "mode": mode, "captured": False, "dtype": dtype,
            "cols": cols}


def listed():
    return [
        # One voice being spoken: every step decodes a single token, half of
        # the 16 layers of the decoder the benchmark uses.
        dict(_decoder(1, "int8", 8, True), name="step_m1_int8"),
        # 32 requests decoded together (the benchmark's decode workload).
        dict(_decoder(32, "int8", 8, True), name="step_m32_int8"),
        # A batch whose request count fills no tile, with K-group scales.
        dict(_decoder(20, "group_fp8", 8, True), name="step_m20_group_fp8"),
        # Close to the largest decode batch, with the f16 type.
        dict(_decoder(57, "fp8", 8, True, dtype="f16"), name="step_m57_fp8"),
        # The prompt of a short request: a sentence and a voice sample.
        dict(_decoder(187, "int8", 4, True), name="prompt_m187_int8"),
        # A longer prompt, or a few short ones packed into one call.
        dict(_decoder(431, "fp8", 4, True), name="prompt_m431_fp8"),
        # A paragraph, with K-group scales.
        dict(_decoder(730, "group_int8", 2, True), name="prompt_m730_group_int8"),
        # Two full contexts of 2048 tokens at once: the largest call.
        dict(_decoder(4096, "int8", 1, False), name="prefill_m4096_int8"),
        # One projection of a packed prefill of uneven lengths.
        dict(_linear(2900, "fp8", 12288, 2048), name="linear_m2900_fp8"),
        # Ten seconds of audio frames through an auxiliary encoder.
        dict(_encoder(499, "int8", 4, True), name="encoder_m499_int8"),
        # The small projections of an auxiliary model over a phoneme sequence.
        dict(_project(150, "int8", 8), name="project_m150_int8"),
        # A projection's weights quantized while a model is loaded.
        dict(_quantize(12288, "group_int8", 2048), name="quantize_load_group_int8"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["step", "step", "prompt", "prompt", "prompt", "prefill", "linear",
                       "encoder", "project", "quantize"])
    mode = rng.choice(list(MODES))
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if kind in ("step", "prompt", "prefill"):
        # Hidden sizes from 1024 up; heads and the gated width follow it.
        hidden = 128 * rng.randint(8, 16)
        sizes = {"dtype": dtype, "hidden": hidden, "qkv": 16 * rng.randint(hidden // 12, hidden // 8),
                 "inter": min(8192, 128 * rng.randint(hidden // 64, hidden // 40))}
        if kind == "step":
            return _decoder(_log(rng, 1, 64), mode, rng.randint(4, 8), True, **sizes)
        if kind == "prompt":
            return _decoder(_log(rng, 65, 1100), mode, rng.randint(1, 3), True, **sizes)
        return _decoder(_log(rng, 1100, 3000), mode, 1, False, **sizes)
    if kind == "linear":
        K = 128 * rng.randint(8, 48) if mode.startswith("group") else 16 * rng.randint(64, 384)
        return _linear(_log(rng, 300, 4096), mode, 16 * rng.randint(128, 768), K, dtype)
    if kind == "encoder":
        hidden = 128 * rng.randint(4, 12)
        return _encoder(_log(rng, 30, 2000), mode, rng.randint(2, 4), True, dtype, hidden,
                        hidden * rng.choice([2, 3, 4]))
    if kind == "project":
        return _project(_log(rng, 1, 400), mode.replace("group_", ""), rng.randint(4, 8), dtype,
                        4 * rng.randint(32, 128), rng.randint(200, 2400))
    cols = 128 * rng.randint(8, 64) if mode.startswith("group") else rng.randint(1000, 8192)
    return _quantize(_log(rng, 1000, 12288), mode, cols, dtype)


# ---------------------------------------------------------------- inputs
class _Inputs:
    """16-bit tensors drawn in a fixed order from one seed, on the GPU."""

    def __init__(self, case, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = DTYPES[case["dtype"]]

    def normal(self, *shape, scale=1.0, offset=0.0):
        return (offset + scale * torch.randn(*shape, generator=self.gen, device="cuda")).to(self.dtype)

    def activations(self, rows, cols):
        """N(0, 1) rows; half a percent of the channels are 20 times larger."""
        x = torch.randn(rows, cols, generator=self.gen, device="cuda")
        channels = torch.randperm(cols, generator=self.gen, device="cuda")[:round(0.005 * cols)]
        x[:, channels] *= 20.0
        return x.to(self.dtype)

    def weights(self, n, k):
        return self.normal(n, k, scale=0.02)


def _decoder_layer(case, inputs):
    h, inter = case["hidden"], case["inter"]
    return {"x": inputs.activations(case["rows"], h),
            "norm1": inputs.normal(h, scale=0.1, offset=1.0),
            "norm2": inputs.normal(h, scale=0.1, offset=1.0),
            "attention": inputs.activations(case["rows"], h),
            "qkv": inputs.weights(case["qkv"], h), "o": inputs.weights(h, h),
            "gate_up": inputs.weights(2 * inter, h), "down": inputs.weights(h, inter)}


def _encoder_layer(case, inputs):
    h, inter = case["hidden"], case["inter"]
    return {"x": inputs.normal(case["rows"], h),
            "norm_weight": inputs.normal(h, scale=0.1, offset=1.0),
            "norm_bias": inputs.normal(h, scale=0.1), "up_bias": inputs.normal(inter, scale=0.1),
            "down_bias": inputs.normal(h, scale=0.1), "up": inputs.weights(inter, h),
            "down": inputs.weights(h, inter)}


def _project_layer(case, inputs):
    k, n = case["k"], case["n"]
    return {"x": inputs.normal(case["rows"], k, offset=0.2),
            "norm_weight": inputs.normal(k, scale=0.1, offset=1.0),
            "norm_bias": inputs.normal(k, scale=0.1), "bias": inputs.normal(n, scale=0.1),
            "w": inputs.weights(n, k)}


_LAYERS = {"decoder": (_decoder_layer, ("qkv", "o", "gate_up", "down")),
           "encoder": (_encoder_layer, ("up", "down")), "project": (_project_layer, ("w",))}


# ---------------------------------------------------------------- the programs
def prepare(case, seed):
    fmt, group, rotation = MODES[case["mode"]]
    inputs = _Inputs(case, seed)
    rows, dtype, dev = case["rows"], DTYPES[case["dtype"]], "cuda"
    state = {"case": case, "fmt": fmt, "group": group, "rotation": rotation}

    def codes(cols):
        return (torch.empty((rows, cols), dtype=torch.uint8, device=dev),
                torch.empty(((cols + group - 1) // group, rows) if group else (rows,),
                            dtype=torch.float32, device=dev))

    def empty(*shape):
        return torch.empty(shape, dtype=dtype, device=dev)

    def plan(n, k):
        return qlinear.plan(rows, n, k, fmt, group, group)

    if case["kind"] in _LAYERS:
        make, quantized = _LAYERS[case["kind"]]
        state["layers"] = []
        for _ in range(case["layers"]):
            layer = make(case, inputs)
            for name in quantized:
                n, k = layer[name].shape
                layer[name] = qlinear.row_quantize(layer[name], fmt, group, rotation) + (plan(n, k),)
            state["layers"].append(layer)
    count = case.get("layers", 1)
    if case["kind"] == "decoder":
        h, inter = case["hidden"], case["inter"]
        state["codes"], state["gated"] = codes(h), codes(inter)
        state["hidden"] = torch.stack([layer.pop("x") for layer in state["layers"]])
        state["out"] = {"qkv": empty(count, rows, case["qkv"]), "o": empty(count, rows, h),
                        "gate_up": empty(count, rows, 2 * inter), "down": empty(count, rows, h),
                        "residual": empty(count, rows, h)}
    elif case["kind"] == "encoder":
        h, inter = case["hidden"], case["inter"]
        state["codes"], state["inner"] = codes(h), codes(inter)
        state["projected"] = empty(rows, h)
        state["out"] = {"up": empty(count, rows, inter), "y": empty(count, rows, h)}
    elif case["kind"] == "project":
        state["out"] = {"y": empty(count, rows, case["n"])}
    elif case["kind"] == "linear":
        n, k = case["N"], case["K"]
        state["x"] = inputs.activations(rows, k)
        state["w"] = qlinear.row_quantize(inputs.weights(n, k), fmt, group, rotation) + (plan(n, k),)
        state["codes"] = codes(k)
        state["out"] = {"y": empty(rows, n), "codes": state["codes"][0], "scales": state["codes"][1]}
    else:
        state["x"] = inputs.weights(rows, case["cols"])
        state["codes"] = codes(case["cols"])
        state["out"] = {"codes": state["codes"][0], "scales": state["codes"][1]}
    if case["captured"]:
        _PROGRAMS[case["kind"]](state)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            _PROGRAMS[case["kind"]](state)
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
    else:
        _PROGRAMS[state["case"]["kind"]](state)
    return state["out"]


def _gemm(s, codes, weight, out):
    w, sw, path = weight
    qlinear.gemm(codes[0], codes[1], w, sw, s["fmt"], input_group=s["group"],
                 weight_group=s["group"], path=path, out=out)


def _run_decoder(s):
    fmt, layout = s["fmt"], {"group": s["group"], "rotation": s["rotation"]}
    out, codes, gated = s["out"], s["codes"], s["gated"]
    out["residual"].copy_(s["hidden"])  # updated in place
    for i, layer in enumerate(s["layers"]):
        residual = out["residual"][i]
        qlinear.quantized_norm(residual, layer["norm1"], fmt, eps=EPS, values=codes[0],
                               scales=codes[1], **layout)
        _gemm(s, codes, layer["qkv"], out["qkv"][i])
        w, sw, path = layer["o"]
        qlinear.linear(layer["attention"], w, sw, fmt, path=path, scratch=codes, out=out["o"][i],
                       **layout)
        qlinear.quantized_norm(residual, layer["norm2"], fmt, update=out["o"][i], eps=EPS,
                               values=codes[0], scales=codes[1], **layout)
        _gemm(s, codes, layer["gate_up"], out["gate_up"][i])
        qlinear.quantized_gated(out["gate_up"][i], fmt, values=gated[0], scales=gated[1], **layout)
        _gemm(s, gated, layer["down"], out["down"][i])


def _run_encoder(s):
    fmt, layout = s["fmt"], {"group": s["group"], "rotation": s["rotation"]}
    out, codes, inner = s["out"], s["codes"], s["inner"]
    for i, layer in enumerate(s["layers"]):
        x = layer["x"]
        qlinear.layer_norm_quantize(x, fmt, layer["norm_weight"], layer["norm_bias"], eps=EPS,
                                    values=codes[0], scales=codes[1], **layout)
        w, sw, path = layer["up"]
        qlinear.gemm_finish(codes[0], codes[1], w, sw, fmt, bias=layer["up_bias"],
                            activation=qlinear.FINISH_GELU_TANH, input_group=s["group"],
                            weight_group=s["group"], path=path, out=out["up"][i])
        qlinear.row_quantize(out["up"][i], fmt, values=inner[0], scales=inner[1], **layout)
        _gemm(s, inner, layer["down"], s["projected"])
        qlinear.pointwise(s["projected"], qlinear.epilogue(bias=layer["down_bias"], residual=x),
                          out=out["y"][i])


def _run_project(s):
    for i, layer in enumerate(s["layers"]):
        w, sw, _ = layer["w"]
        qlinear.norm_linear(layer["x"], w, sw, s["fmt"], layer["norm_weight"], layer["norm_bias"],
                            bias=layer["bias"], eps=EPS, out=s["out"]["y"][i])


def _run_linear(s):
    w, sw, path = s["w"]
    qlinear.linear(s["x"], w, sw, s["fmt"], s["group"], s["rotation"], path=path,
                   scratch=s["codes"], out=s["out"]["y"])


def _run_quantize(s):
    qlinear.row_quantize(s["x"], s["fmt"], s["group"], s["rotation"], s["codes"][0], s["codes"][1])


_PROGRAMS = {"decoder": _run_decoder, "encoder": _run_encoder, "project": _run_project,
             "linear": _run_linear, "quantize": _run_quantize}


# ---------------------------------------------------------------- work and tolerance
def _projections(case):
    """(N, K) of every GEMM of one layer."""
    if case["kind"] == "decoder":
        h, inter = case["hidden"], case["inter"]
        return [(case["qkv"], h), (h, h), (2 * inter, h), (h, inter)]
    if case["kind"] == "encoder":
        return [(case["inter"], case["hidden"]), (case["hidden"], case["inter"])]
    if case["kind"] == "project":
        return [(case["n"], case["k"])]
    return [(case["N"], case["K"])] if case["kind"] == "linear" else []


def work(case):
    m, group = case["rows"], MODES[case["mode"]][1]

    def scales(rows, cols):
        return 4 * rows * (-(-cols // group) if group else 1)

    if case["kind"] == "quantize":
        cols = case["cols"]
        return {"bytes": 3 * m * cols + scales(m, cols), "flops": 4 * m * cols}
    count = case.get("layers", 1)
    pairs = _projections(case)
    weights = sum(n * k + scales(n, k) for n, k in pairs)
    outputs = sum(2 * m * n for n, _ in pairs)
    flops = sum(2 * m * n * k for n, k in pairs)
    if case["kind"] == "decoder":  # hidden state and attention output in, the residual out
        return {"bytes": count * (weights + outputs + 6 * m * case["hidden"]), "flops": count * flops}
    if case["kind"] == "encoder":
        return {"bytes": count * (weights + outputs + 2 * m * case["hidden"]), "flops": count * flops}
    if case["kind"] == "project":
        return {"bytes": count * (weights + outputs + 2 * m * case["k"]), "flops": count * flops}
    k = case["K"]
    return {"bytes": weights + outputs + 3 * m * k + scales(m, k), "flops": flops}


def tolerance(case):
    # Codes, scales and INT8 sums have one right value. Measured between paths
    # that sum in another order: INT8 none, FP8 and FP8 groups up to 1.7e-5
    # (largest 5e-3) in `down`, where a value that rounded the other way has
    # moved a code of the next projection. Beyond the order, the epilogue's two
    # scale products may round either way: up to one unit of the 16-bit type,
    # and in a stack the codes that such a unit moves.
    if case["kind"] == "quantize":
        return "exact"
    if case["kind"] in ("linear", "project"):
        return {"rel": 2e-3, "max": 0.02}
    return {"rel": 5e-3, "max": 0.1}


# ---------------------------------------------------------------- 64-bit results
def _signs(cols):
    """The Rademacher signs of the H128 rotation, by absolute column."""
    mask = 0xFFFFFFFF
    h = torch.arange(cols, dtype=torch.int64, device="cuda") * 0x45D9F3B & mask
    h = (h ^ (h >> 16)) * 0x45D9F3B & mask
    return ((h ^ (h >> 16)) & 1) * 2.0 - 1.0


def _hadamard():
    h = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    while h.shape[0] < 128:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(128.0)


def _quantized(v, case):
    """Rows as the codes and scales of the mode stand for them, in 64 bits;
    and the scales in their layout."""
    fmt, group, rotation = MODES[case["mode"]]
    v = v.double()
    rows, cols = v.shape
    if rotation:
        v = ((v * _signs(cols)).view(rows, cols // 128, 128) @ _hadamard()).view(rows, cols)
    top = 127.0 if fmt == qlinear.I8 else 448.0
    g = group or cols
    padded = torch.nn.functional.pad(v, (0, -cols % g)).view(rows, -1, g)
    amax = padded.abs().amax(2, keepdim=True)
    scale = torch.where(amax == 0, torch.ones_like(amax), amax / top)
    q = (padded / scale).clamp(-top, top)
    q = q.round() if fmt == qlinear.I8 else q.float().to(torch.float8_e4m3fn).double()
    values = (q * scale).view(rows, -1)[:, :cols]
    return values, (scale[:, :, 0].t().contiguous() if group else scale.view(rows))


def exact(case, seed):
    inputs = _Inputs(case, seed)
    rows, dtype = case["rows"], DTYPES[case["dtype"]]

    def stored(t):  # rounded to the 16-bit type that the programs hand on
        return t.to(dtype).double()

    def product(values, weight):
        return stored(values @ _quantized(weight, case)[0].t())

    if case["kind"] == "quantize":
        return {"codes": None, "scales": _quantized(inputs.weights(rows, case["cols"]), case)[1]}
    if case["kind"] == "linear":
        values, scales = _quantized(inputs.activations(rows, case["K"]), case)
        return {"y": product(values, inputs.weights(case["N"], case["K"])), "codes": None,
                "scales": scales}
    out = {}

    def keep(name, value):
        out.setdefault(name, []).append(value)
        return value

    make, _ = _LAYERS[case["kind"]]
    if case["kind"] == "decoder":
        def rms(residual, weight):
            unit = residual / torch.sqrt(residual.square().mean(1, keepdim=True) + EPS)
            return _quantized(stored(stored(unit) * weight.double()), case)[0]

        for _ in range(case["layers"]):
            layer = make(case, inputs)
            x = layer["x"].double()
            keep("qkv", product(rms(x, layer["norm1"]), layer["qkv"]))
            o = keep("o", product(_quantized(layer["attention"], case)[0], layer["o"]))
            x = keep("residual", stored(x + o))
            gate, up = keep("gate_up", product(rms(x, layer["norm2"]), layer["gate_up"])).chunk(2, 1)
            gated = stored(stored(gate * torch.sigmoid(gate)) * up)
            keep("down", product(_quantized(gated, case)[0], layer["down"]))

    def layer_norm(layer):
        x = layer["x"].double()
        unit = (x - x.mean(1, keepdim=True)) / torch.sqrt(x.var(1, unbiased=False, keepdim=True) + EPS)
        n = stored(unit * layer["norm_weight"].double() + layer["norm_bias"].double())
        return _quantized(n, case)[0]

    if case["kind"] == "encoder":
        for _ in range(case["layers"]):
            layer = make(case, inputs)
            v = stored(product(layer_norm(layer), layer["up"]) + layer["up_bias"].double())
            v = keep("up", stored(torch.nn.functional.gelu(v, approximate="tanh")))
            v = stored(product(_quantized(v, case)[0], layer["down"]) + layer["down_bias"].double())
            keep("y", stored(v + layer["x"].double()))
    elif case["kind"] == "project":
        for _ in range(case["layers"]):
            layer = make(case, inputs)
            keep("y", stored(product(layer_norm(layer), layer["w"]) +
                             layer["bias"].double()))
    return {k: torch.stack(v) for k, v in out.items()}
