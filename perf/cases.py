"""The work that programs built on this package have it do, as measurable cases.

A case is one pass of a program: a quantized linear layer called on a batch of token rows
(`ConvRotLinear.forward`, `forward_modulated`, `forward_gelu`), eagerly or as the replay of a HIP
graph that holds several layers, or the conversion of a dense weight into a layer.  Sizes are
those of the FLUX.1-dev transformer, the Wan 2.2 and LTX 2.5 projections and the weight-only
linears that bench.py, examples/ and tests/ use, and sizes around them.

Fields of a case
  op        "linear" or "convert"
  rows      token rows; k, n: input and output features; group: the rotation's group
  dtype     "bfloat16", "float16" or "float32" activations and outputs
  backend   "hip-w4a4" (4-bit activations) or "hip-w4a16" (16-bit activations)
  producer  "plain": layer(x); "modulate": adaLN LayerNorm and modulation in front, one vector for
            all rows; "gelu": tanh GELU in front, of an x that is a slice of a wider projection,
            behind `head` features that are taken as they are
  residual  "none", "add" (residual + linear) or "gate" (residual + gate * linear)
  layers    layers a pass runs, each with its own weights and input
  graph     the pass is the replay of a captured HIP graph
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "convrot-mlx_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from convrot_mlx_amd import ConvRotLinear, quantize_convrot_weight  # noqa: E402

_DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}
_LINEAR = {"op": "linear", "rows": 1, "k": 3072, "n": 3072, "group": 256, "dtype": "bfloat16", "backend": "hip-w4a4",
           "producer": "plain", "head": 0, "residual": "none", "layers": 1, "graph": False}
_CONVERT = {"op": "convert", "k": 3072, "n": 12288, "group": 256, "dtype": "bfloat16"}


def listed() -> list[dict]:
    def linear(name, **kw):
        return {**_LINEAR, "name": name, **kw}

    return [
        # One adaLN modulation layer of a diffusion transformer (a single conditioning row), called
        # eagerly: the smallest call there is, its latency is launches and host work.
        linear("modulation row eager", rows=1, n=18432, group=64),
        # The modulation layers of consecutive blocks, in the HIP graph that a sampler replays.
        linear("modulation rows graph", rows=1, n=9216, group=64, layers=8, graph=True),
        # Weight-only layers on a single row, one after another: a decoder's up projections.
        linear("w4a16 row graph", rows=1, n=12288, backend="hip-w4a16", layers=8, graph=True),
        # The same for the down projections of 32 rows served together.
        linear("w4a16 32 rows graph", rows=32, k=12288, n=3072, backend="hip-w4a16", layers=8, graph=True),
        # A short prompt's text stream: fewer rows than one tile, an odd number of them.
        linear("77 rows", rows=77, group=64, layers=4, graph=True),
        # The text stream's qkv projection of a double block, with the modulated norm in front.
        linear("512 rows modulated", rows=512, n=9216, group=64, producer="modulate", layers=2, graph=True),
        # The second linear of a single block: [attention | gelu(mlp)], gated back into the stream.
        linear("1536 rows gelu gated", rows=1536, k=15360, group=64, producer="gelu", head=3072, residual="gate"),
        # The up projection at 4096 image and 512 text tokens.
        linear("4608 rows", rows=4608, n=12288),
        # A video model's contraction, the largest call.
        linear("8800 rows contraction", rows=8800, k=16384, n=4096),
        # A ragged video shape in float16: neither the rows nor the features fill whole tiles.
        linear("10017 rows float16", rows=10017, k=2688, n=2688, group=64, dtype="float16"),
        # Weight-only on an image's token rows.
        linear("w4a16 1536 rows", rows=1536, n=12288, backend="hip-w4a16"),
        # Offline: one dense weight quantized and installed in a layer.
        {**_CONVERT, "name": "convert a weight"},
    ]


_COST = 8800 * 16384 * 4096


def draw(rng) -> dict:
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if rng.random() < 0.1:
        group = rng.choice([64, 256])
        return {**_CONVERT, "k": spread(1024 // group, 15360 // group) * group, "n": spread(512, 18432), "group": group,
                "dtype": rng.choice(["bfloat16", "bfloat16", "float16", "float32"])}
    case = dict(_LINEAR)
    case["backend"] = rng.choice(["hip-w4a4", "hip-w4a4", "hip-w4a16"])
    kinds = ["bfloat16"] * 6 + ["float16"] * 2 + (["float32"] if case["backend"] == "hip-w4a4" else [])
    case["dtype"] = rng.choice(kinds)
    case["group"] = group = rng.choice([64, 256])
    case["rows"] = rows = rng.choice([1, spread(1, 64), spread(1, 8800), spread(64, 8800)])
    # most features are multiples of 128 or more, as a model's are; some are odd ones
    k = spread(1024, 16384)
    k = max(group, k // 512 * 512 if rng.random() < 0.6 else k // group * group)
    n = spread(1024, 21504)
    n = n // 128 * 128 if rng.random() < 0.75 else n
    # a weight-only product runs its matrix instructions at 16 bits: a quarter of the work
    while rows * k * n > _COST // (4 if case["backend"] == "hip-w4a16" else 1):
        k, n = max(group, k // 2 // group * group), max(512, n // 2)
    case["k"], case["n"] = k, n
    case["producer"] = rng.choice(["plain", "plain", "modulate", "gelu"])
    if case["producer"] == "gelu" and rng.random() < 0.5:
        case["head"] = k // 4 // 64 * 64
    case["residual"] = rng.choice(["none", "none", "add", "gate"])
    if rows * k * n <= 2 ** 34:
        case["layers"], case["graph"] = rng.choice([(1, False), (1, True), (4, True)])
    return case


# ------------------------------------------------------------------ inputs


def _normal(gen, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * std).to(dtype)


def _activation(gen, rows, k, dtype):
    """N(0, 1) with one channel in 200 twenty times as large: a transformer's outlier channels."""
    gain = torch.ones(k, device="cuda")
    gain[torch.randperm(k, generator=gen, device="cuda")[: max(1, k // 200)]] = 20.0
    return (torch.randn((rows, k), generator=gen, device="cuda") * gain).to(dtype)


def _weight(gen, n, k, dtype):
    """N(0, 0.02^2) with one input channel in 100 ten times as large."""
    gain = torch.full((k,), 0.02, device="cuda")
    gain[torch.randperm(k, generator=gen, device="cuda")[: max(1, k // 100)]] = 0.2
    return (torch.randn((n, k), generator=gen, device="cuda") * gain).to(dtype)


def _inputs(case: dict, seed: int):
    """The tensors of each layer of a pass, made from the seed alone (a dict a layer)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    if case["op"] == "convert":
        yield {"weight": _weight(gen, case["n"], case["k"], dtype), "bias": _normal(gen, case["n"], std=0.02)}
        return
    rows, k, n = case["rows"], case["k"], case["n"]
    for _ in range(case["layers"]):
        t = {"weight": _weight(gen, n, k, torch.bfloat16), "bias": _normal(gen, n, std=0.02)}
        if case["producer"] == "gelu":
            t["wide"] = _activation(gen, rows, 1024 + k - case["head"], dtype)  # x is its last features
            t["head"] = _activation(gen, rows, case["head"], dtype) if case["head"] else None
        else:
            t["x"] = _activation(gen, rows, k, dtype)
        if case["producer"] == "modulate":
            t["shift"], t["scale"] = (_normal(gen, 1, k, dtype=dtype, std=0.2) for _ in range(2))
        if case["residual"] != "none":
            t["residual"] = _normal(gen, rows, n, dtype=dtype)
        if case["residual"] == "gate":
            t["gate"] = _normal(gen, 1, n, dtype=dtype, std=0.5)
        yield t


def _call(case: dict, layer: ConvRotLinear, t: dict) -> torch.Tensor:
    more = {"residual": t["residual"], "gate": t.get("gate")} if "residual" in t else {}
    if case["producer"] == "modulate":
        return layer.forward_modulated(t["x"], t["shift"], t["scale"], **more)
    if case["producer"] == "gelu":
        return layer.forward_gelu(t["wide"][:, 1024:], t["head"], **more)
    return layer(t["x"], **more)


_stream = None


def _capture(passes) -> tuple:
    """The pass as a HIP graph, captured after a warm-up on one side stream that this process keeps."""
    global _stream
    _stream = _stream or torch.cuda.Stream()
    _stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(_stream):
        passes()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=_stream):
        out = passes()
    return graph, out


@torch.no_grad()
def prepare(case: dict, seed: int) -> dict:
    state = {"case": case}
    if case["op"] == "convert":
        state.update(next(_inputs(case, seed)))
        return state
    layers, tensors = [], []
    for t in _inputs(case, seed):
        layer = ConvRotLinear(case["k"], case["n"], group_size=case["group"], backend=case["backend"], device="cuda")
        codes, scales = quantize_convrot_weight(t.pop("weight"), case["group"])
        layers.append(layer.load_nk_weight(codes, scales, t.pop("bias")))
        tensors.append(t)
    state["pass"] = lambda: [_call(case, layer, t) for layer, t in zip(layers, tensors)]
    if case["graph"]:
        state["graph"], state["out"] = _capture(state["pass"])
    else:
        state["pass"]()  # a layer lays its weights out for the kernels at its first call
    return state


@torch.no_grad()
def run(state: dict):
    case = state["case"]
    if case["op"] == "convert":
        codes, scales = quantize_convrot_weight(state["weight"], case["group"])
        layer = ConvRotLinear(case["k"], case["n"], group_size=case["group"], backend="hip-w4a4", device="cuda")
        layer.load_nk_weight(codes, scales, state["bias"])
        return {"codes": codes, "scales": layer.scales, "qweight": layer.qweight}
    if case["graph"]:
        state["graph"].replay()
        return state["out"]
    return state["pass"]()


# ------------------------------------------------------------------ work and accuracy


def work(case: dict) -> dict:
    size = 4 if case["dtype"] == "float32" else 2
    k, n = case["k"], case["n"]
    if case["op"] == "convert":  # read the weight, write the packed codes, the laid out codes and the scales
        return {"bytes": n * k * size + n * k + 4 * n, "flops": n * k * (4 * round(math.log(case["group"], 4)) + 4)}
    rows = case["rows"]
    moved = rows * k * size + n * k / 2 + 8 * n + rows * n * size  # activations, weights, scales and bias, result
    if case["producer"] == "modulate":
        moved += 2 * k * size
    if case["residual"] != "none":
        moved += rows * n * size
    if case["residual"] == "gate":
        moved += n * size
    return {"bytes": case["layers"] * moved, "flops": case["layers"] * 2.0 * rows * k * n}


def tolerance(case: dict):
    """4-bit activations: integers are summed exactly and every later step is one fixed float32
    operation, so any correct implementation gives the same bits.  16-bit activations: float32 sums
    in another order move a few results across a rounding of the output type.  Against 64-bit sums
    rounded once, up to 2.4e-6 (bfloat16) and 3.6e-5 (float16) of the results move by one step of the
    type, 1.2e-5 and 4.1e-6 of the 2-norm; among the 1024 results of a small call a single step is
    1.2e-4 and 1.5e-5 of it.  The tolerances are two to four times that, and a step through the
    roundings of a gated residual."""
    if case["op"] == "convert" or case["backend"] == "hip-w4a4":
        return "exact"
    return {"rel": 2.5e-4, "max": 2e-2} if case["dtype"] == "bfloat16" else {"rel": 4e-5, "max": 2.5e-3}


def _rotate(x: torch.Tensor, group: int) -> torch.Tensor:
    """The regular Hadamard rotation of each group of features, every sum rounded to x's type."""
    rows, k = x.shape
    y, stride = x, 1
    while stride < group:
        a, b, c, d = y.reshape(rows, k // (4 * stride), 4, stride).unbind(2)
        y = torch.stack([a + b + c - d, a + b - c + d, a - b + c + d, -a + b + c + d], 2)
        stride *= 4
    return (y.reshape(rows, k).float() / math.sqrt(group)).to(x.dtype)


def _codes(y: torch.Tensor):
    """4-bit codes and float32 scales of rows, every step rounded to y's type."""
    floor = torch.tensor(1e-10, dtype=y.dtype, device=y.device)
    scale = (torch.maximum(y.abs().amax(1, keepdim=True), floor).float() / 7.0).to(y.dtype)
    ratio = (y.float() / scale.float()).to(y.dtype).float()
    return torch.where(scale > 0, ratio, 0.0).round().clamp(-7, 7), scale.float()


def _produced(case: dict, t: dict) -> torch.Tensor:
    """What the layer rotates, rounded where the layer's contract rounds."""
    if case["producer"] == "gelu":
        x = t["wide"][:, 1024:]
        g = torch.nn.functional.gelu(x.double(), approximate="tanh").to(x.dtype)
        return g if t["head"] is None else torch.cat([t["head"], g], 1)
    x = t["x"]
    if case["producer"] == "modulate":
        d = x.double()
        mean, mean2 = d.mean(1, keepdim=True), (d * d).mean(1, keepdim=True)
        rstd = 1.0 / torch.sqrt((mean2 - mean * mean).clamp_min(0.0) + 1e-6)
        norm = ((x.float() - mean.float()) * rstd.float()).to(x.dtype)
        return (1 + t["scale"]) * norm + t["shift"]
    return x


@torch.no_grad()
def exact(case: dict, seed: int):
    """The rounded steps of the contract in torch, the products, sums and epilogue in 64 bits."""
    results = []
    for t in _inputs(case, seed):
        w_codes, w_scale = _codes(_rotate(t["weight"], case["group"]))
        if case["op"] == "convert":
            return {"codes": None, "scales": w_scale[:, 0].double(), "qweight": None}
        y = _rotate(_produced(case, t), case["group"])
        a, a_scale = _codes(y) if case["backend"] == "hip-w4a4" else (y, torch.ones(1, device=y.device))
        out = a.double() @ w_codes.double().t().contiguous()
        out = out * a_scale.double() * w_scale[:, 0].double() + t["bias"].double()
        if case["residual"] != "none":
            out = t["residual"].double() + out * (t["gate"].double() if "gate" in t else 1.0)
        results.append(out)
    return results
