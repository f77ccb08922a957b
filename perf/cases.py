"""The work this framework is used for, as cases that can be timed and compared.

Each case runs through the public entry points a program uses: `RocmTarget().compile(graph)`
gives an executable, `launch()` queues one pass over inputs that are already on the device,
`run()` takes host arrays and returns host arrays, and `DecodeLoop.decode()` generates tokens.
Graphs come from the repository's own model builders and lowering, so a case sees what the
compiler gives the target.

    listed()             the fixed cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  the compiled plan and the inputs (made from the seed, on the GPU)
    run(state)           one pass and its whole outputs
    work(case)           the bytes and operations a pass cannot do without
    tolerance(case)      how far another correct implementation may be off
    exact(case, seed)    the same pass in 64 bits, in plain torch

Kinds of case
    dense    one W8A8 dense layer (rows x K -> N)
    mlp      the 50M-parameter MLP, W8A8 or with int8 weights only
    resnet   W8A8 ResNet-18 on 224 x 224 images
    mobile   W8A8 MobileNetV2 on 224 x 224 images
    block    one residual block of two 3x3 convolutions, its whole feature map as the output
    attn     one decoder layer's attention half: layernorm, q/k/v projections, attention over the cache
    step     one decode step of the character-level GPT for a batch of sequences
    decode   a whole greedy decode of that GPT: prompt in, tokens out
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from harness import lowering, models
from harness.decode import DeviceDecoder
from harness.graph import Graph
from harness.runner import Runner
from mira_amd import get_target

DEV = "cuda:0"


def listed() -> list:
    return [
        # the smallest call there is: one dense layer of a small classifier, one batch of rows
        {"name": "dense_256x64x10", "kind": "dense", "rows": 256, "k": 64, "n": 10, "relu": False},
        # serving one request: every weight byte is read for one row
        {"name": "mlp50m_b1", "kind": "mlp", "batch": 1, "weight_only": False},
        # offline scoring in large batches: the int8 matrix products themselves
        {"name": "mlp50m_b4096", "kind": "mlp", "batch": 4096, "weight_only": False},
        # weight-only int8 (f32 activations and sums) at a ragged batch of queued requests
        {"name": "mlp50m_w8_b33", "kind": "mlp", "batch": 33, "weight_only": True},
        # one image from host memory to logits in host memory, as the compiler's driver calls the target
        {"name": "resnet18_b1_host", "kind": "resnet", "batch": 1, "precision": "f32", "host": True},
        # image throughput on device-resident data
        {"name": "resnet18_b256", "kind": "resnet", "batch": 256, "precision": "f32", "host": False},
        # one stage's residual block in the f16 precision accelerator targets get, an odd batch
        {"name": "block_f16_c128_b37", "kind": "block", "batch": 37, "c_in": 128, "c": 128, "side": 28, "stride": 1,
         "precision": "f16"},
        # one image through the mobile network: many small launches in a row
        {"name": "mobilenetv2_b1", "kind": "mobile", "batch": 1, "precision": "f32"},
        # the mobile network's throughput: depthwise and short-K convolutions
        {"name": "mobilenetv2_b128", "kind": "mobile", "batch": 128, "precision": "f32"},
        # the attention half of a decoder layer for many sequences, at full context
        {"name": "attn_b512", "kind": "attn", "batch": 512, "d": 64, "heads": 4, "context": 272},
        # one decode step for many sequences
        {"name": "gpt_step_b512", "kind": "step", "batch": 512, "layers": 2, "d": 64, "heads": 4, "ff": 128,
         "vocab": 65, "context": 272},
        # one user's greedy decode: a 16-token prompt and 256 generated tokens, one after another
        {"name": "gpt_decode_b1", "kind": "decode", "batch": 1, "layers": 2, "d": 64, "heads": 4, "ff": 128,
         "vocab": 65, "context": 272, "prompt": 16, "new": 256},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    """A case of the listed kinds over their whole ranges: batches of 1 to the listed largest, odd
    channel counts and widths, both precisions, other strides and context lengths."""
    kind = rng.choice(["dense", "mlp", "resnet", "mobile", "block", "attn", "step", "decode"])
    if kind == "dense":
        return {"kind": kind, "rows": _log_int(rng, 1, 4096), "k": _log_int(rng, 17, 4096), "n": _log_int(rng, 10, 4096),
                "relu": rng.random() < 0.5}
    if kind == "mlp":
        weight_only = rng.random() < 0.4
        return {"kind": kind, "batch": _log_int(rng, 1, 1024 if weight_only else 4096), "weight_only": weight_only}
    if kind == "resnet":
        host = rng.random() < 0.25
        return {"kind": kind, "batch": _log_int(rng, 1, 16 if host else 256), "precision": rng.choice(["f32", "f16"]),
                "host": host}
    if kind == "mobile":
        return {"kind": kind, "batch": _log_int(rng, 1, 128), "precision": rng.choice(["f32", "f16"])}
    if kind == "block":
        c, stride, side = _log_int(rng, 16, 512), rng.choice([1, 1, 2]), _log_int(rng, 7, 56)
        c_in = c if stride == 1 else max(16, c // 2)
        most = min(256, int(5e7 / (c * side * side)), int(2e11 / (36.0 * c * c * side * side)))
        return {"kind": kind, "batch": _log_int(rng, 1, max(2, most)), "c_in": c_in, "c": c, "side": side,
                "stride": stride, "precision": rng.choice(["f32", "f16"])}
    heads, hd = rng.choice([1, 2, 3, 4, 8]), rng.choice([16, 32])
    d, context = heads * hd, rng.randrange(40, 321)
    if kind == "attn":
        return {"kind": kind, "batch": _log_int(rng, 1, 512), "d": d, "heads": heads, "context": context}
    ends = {"layers": rng.choice([1, 2, 3]), "d": d, "heads": heads, "ff": rng.choice([2, 4]) * d,
            "vocab": rng.randrange(30, 129), "context": context}
    if kind == "step":
        return {"kind": kind, "batch": _log_int(rng, 1, 512), **ends}
    prompt = rng.randrange(1, 25)
    return {"kind": kind, "batch": _log_int(rng, 1, 64), **ends, "prompt": prompt,
            "new": rng.randrange(8, min(context - prompt, 96) + 1)}


# ---------------------------------------------------------------- graphs

def _normal(rng, shape, std: float) -> np.ndarray:
    return (rng.standard_normal(shape, dtype=np.float32) * np.float32(std)).astype(np.float32)


def _dense_graph(rows: int, k: int, n: int, relu: bool) -> Graph:
    rng = np.random.default_rng(1)
    g = Graph("dense")
    y = g.op("add", [g.op("matmul", [g.input("x", (rows, k)), g.const(_normal(rng, (k, n), k ** -0.5))]),
                     g.const(_normal(rng, (n,), 0.1))])
    g.outputs = [g.op("relu", [y]) if relu else y]
    return g


def _block_graph(batch: int, c_in: int, c: int, side: int, stride: int) -> Graph:
    """A residual block: 3x3 conv + bias + relu, 3x3 conv + bias, + shortcut, relu; the shortcut is
    a 1x1 convolution where the shape changes."""
    rng = np.random.default_rng(1)
    g = Graph("block")

    def conv(x, o, kk, s, p):
        ci = x.type.shape[1]
        y = g.op("conv2d", [x, g.const(_normal(rng, (o, ci, kk, kk), math.sqrt(2.0 / (o * kk * kk))))],
                 {"stride": (s, s), "padding": (p, p)})
        return g.op("add", [y, g.const(_normal(rng, (o, 1, 1), 0.1))])

    x = g.input("x", (batch, c_in, side, side))
    y = conv(g.op("relu", [conv(x, c, 3, stride, 1)]), c, 3, 1, 1)
    y = g.op("relu", [g.op("add", [y, x if stride == 1 and c_in == c else conv(x, c, 1, stride, 0)])])
    g.outputs = [g.op("reshape", [y], {"shape": (batch, y.type.numel // batch)})]
    return g


def _attn_graph(batch: int, d: int, heads: int, context: int) -> Graph:
    """The attention half of models.gpt_decode_step's layer, ending at the context vectors."""
    rng = np.random.default_rng(1)
    hd, T = d // heads, context
    g = Graph("attn")
    h, mask = g.input("h", (batch, d)), g.input("mask", (1, 1, 1, T + 1))
    kc, vc = g.input("kc0", (batch, T, d)), g.input("vc0", (batch, T, d))
    gain, bias = models.mira_random_weight(rng, (d,)), models.mira_random_weight(rng, (d,))
    x = g.op("layernorm", [h, g.const(gain), g.const(bias)], {"eps": 1e-5})
    q, k, v = (g.op("matmul", [x, g.const(models.mira_random_weight(rng, (d, d)))]) for _ in range(3))
    q4 = g.op("transpose", [g.op("reshape", [q], {"shape": (batch, 1, heads, hd)})], {"perm": (0, 2, 1, 3)})
    keys = g.op("concat", [kc, g.op("reshape", [k], {"shape": (batch, 1, d)})], {"axis": 1})
    vals = g.op("concat", [vc, g.op("reshape", [v], {"shape": (batch, 1, d)})], {"axis": 1})
    k4 = g.op("transpose", [g.op("reshape", [keys], {"shape": (batch, T + 1, heads, hd)})], {"perm": (0, 2, 3, 1)})
    v4 = g.op("transpose", [g.op("reshape", [vals], {"shape": (batch, T + 1, heads, hd)})], {"perm": (0, 2, 1, 3)})
    s = g.op("add", [g.op("mul", [g.op("matmul", [q4, k4]), g.const(np.float32(1.0 / np.sqrt(hd)))]), mask])
    o4 = g.op("matmul", [g.op("softmax", [s], {"axis": -1}), v4])
    g.outputs = [g.op("reshape", [g.op("transpose", [o4], {"perm": (0, 2, 1, 3)})], {"shape": (batch, d)}), k, v]
    return g


def _config(case: dict):
    return models.GPTConfig(case["layers"], case["d"], case["heads"], case["ff"], case["vocab"], case["context"])


@functools.lru_cache(maxsize=4)
def _params(layers: int, d: int, heads: int, ff: int, vocab: int, context: int) -> dict:
    return models.gpt_params(models.GPTConfig(layers, d, heads, ff, vocab, context), seed=0)


def _gpt_params(case: dict) -> dict:
    return _params(case["layers"], case["d"], case["heads"], case["ff"], case["vocab"], case["context"])


def _float_graph(case: dict, batch: int) -> Graph:
    kind = case["kind"]
    if kind == "dense":
        return _dense_graph(batch, case["k"], case["n"], case["relu"])
    if kind == "mlp":
        return models.mlp_50m(batch=batch, seed=0)
    if kind == "resnet":
        return models.resnet18(batch=batch, seed=0)
    if kind == "mobile":
        return models.mobilenet_v2(batch=batch, seed=0)
    if kind == "block":
        return _block_graph(batch, case["c_in"], case["c"], case["side"], case["stride"])
    if kind == "attn":
        return _attn_graph(batch, case["d"], case["heads"], case["context"])
    return models.gpt_decode_step(_config(case), batch, _gpt_params(case))


def _batch(case: dict) -> int:
    return case["rows"] if case["kind"] == "dense" else case["batch"]


_GRAPHS: dict = {}


def _graph(case: dict) -> Graph:
    """The case's quantized graph, kept as a program keeps its model (the last few only).  Its
    activation scales are the peaks of a small batch of the same weights."""
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "host", "prompt", "new")))
    if key not in _GRAPHS:
        while len(_GRAPHS) >= 2:
            _GRAPHS.pop(next(iter(_GRAPHS)))
        precision = "f16" if case.get("precision") == "f16" else None
        g = lowering.prepare(_float_graph(case, _batch(case)), precision)
        if case.get("weight_only"):
            lowering.weight_only(g)
        else:
            twin = lowering.prepare(_float_graph(case, 2), precision)
            watch = [op.inputs[0] for op in lowering.w8a8_candidates(twin)]
            env = _evaluate(twin, _inputs(case, twin, 12345), watch)
            lowering.w8a8(g, peaks=[float(env[v].abs().max()) for v in watch])
        _GRAPHS[key] = g
    return _GRAPHS[key]


# ---------------------------------------------------------------- inputs and plans

def _inputs(case: dict, g: Graph, seed: int) -> dict:
    """{graph input: f32 tensor on the GPU}: images U(0, 1), rows N(0, 1); a decode step gets an
    embedded token, caches filled up to its position and the mask that hides the rest."""
    gen = torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)
    out = {}
    written = None
    for v in g.inputs:
        shape = tuple(v.type.shape)
        if v.name == "mask":
            T = shape[-1] - 1
            written = T - 1 - int(torch.randint(0, max(1, T // 8), (1,), generator=gen, device=DEV))
            m = torch.full(shape, -10000.0, device=DEV)
            m[..., :written] = 0.0
            m[..., T] = 0.0
            out[v] = m
        elif case["kind"] in ("resnet", "mobile"):
            out[v] = torch.rand(shape, generator=gen, device=DEV)
        elif case["kind"] == "block":
            out[v] = torch.relu(torch.randn(shape, generator=gen, device=DEV))     # a relu's feature map
        else:
            out[v] = torch.randn(shape, generator=gen, device=DEV)
            if v.name[:2] in ("kc", "vc"):
                out[v][:, written:] = 0.0
    return out


class _State:
    """What a program holds between calls: the executable (or decode loop) and its inputs."""


def prepare(case: dict, seed: int) -> _State:
    g = _graph(case)
    s = _State()
    target = get_target("rocm", approx_f32=case["kind"] in ("attn", "step", "decode"))
    if case["kind"] == "decode":
        s.loop = DeviceDecoder(Runner(g, target), _config(case), _gpt_params(case), case["batch"])
        s.prompt = np.random.default_rng(seed).integers(0, case["vocab"], (case["batch"], case["prompt"])).astype(np.int32)
        s.new = case["new"]
        s.loop.reset(s.prompt)
        s.loop.capture(1)
        return s
    s.exe = target.compile(g)
    feeds = _inputs(case, g, seed)
    if case.get("host"):
        s.feeds = {v: t.cpu().numpy() for v, t in feeds.items()}
        return s
    s.feeds = None
    for v, t in feeds.items():
        s.exe.device_input(v).copy_(t)
    s.outputs = [s.exe.device_output(v) for v in g.outputs]
    return s


def run(state: _State):
    if hasattr(state, "loop"):
        tokens = state.loop.decode(state.prompt, state.new, use_graph=True)
        return {"tokens": tokens, "logits": state.loop.logits, "caches": list(state.loop.caches)}
    if state.feeds is not None:
        return list(state.exe.run(state.feeds).values())
    state.exe.launch()
    return state.outputs


# ---------------------------------------------------------------- work and tolerance

def work(case: dict) -> dict:
    kind, b = case["kind"], _batch(case)
    if kind == "dense":
        k, n = case["k"], case["n"]
        return {"bytes": 4.0 * b * k + k * n + 8.0 * n + 4.0 * b * n, "flops": 2.0 * b * k * n}
    if kind in ("attn", "step", "decode"):
        d, T = case["d"], case["context"]
        layers = case.get("layers", 1)
        weights = 3 * d * d if kind == "attn" else layers * (4 * d * d + 2 * d * case["ff"]) + d * case["vocab"]
        outs = 3 * d if kind == "attn" else 2 * layers * d + case["vocab"]
        if kind == "decode":
            steps = case["prompt"] + case["new"] - 1
            rows = steps * (steps - 1) / 2.0                       # cache rows written before each step, summed
        else:
            steps, rows = 1, float(T)
        return {"bytes": steps * weights + b * (8.0 * layers * d * rows + 4.0 * steps * (d + outs)),
                "flops": b * (2.0 * steps * weights + 4.0 * layers * d * (rows + steps))}
    g = _graph(case)
    flops, weights = 0.0, 0.0
    for op in g.ops:
        if op.kind in ("qmatmul", "qconv2d", "matmul", "conv2d"):
            w = op.attrs["q"] if op.kind[0] == "q" else _const(op.inputs[1])
            weights += w.size * w.dtype.itemsize
            flops += 2.0 * op.result.type.numel * (w.shape[0] if "matmul" in op.kind else w[0].size)
    return {"bytes": weights + 4.0 * sum(v.type.numel for v in [*g.inputs, *g.outputs]), "flops": flops}


def _const(v) -> np.ndarray:
    return v.producer.attrs["q" if v.producer.kind == "dequantize" else "value"]


def tolerance(case: dict):
    if case["kind"] == "mlp" and case["weight_only"]:
        return {"rel": 7e-6}                # f32 sums of 4096 products in another order, four layers (1.7e-6 off 64 bits)
    if case["kind"] == "attn":
        return {"rel": 1e-6}                # f32 softmax and sums over the cache in another order (2.4e-7 off 64 bits)
    if case["kind"] in ("step", "decode"):
        # another order of the attention's f32 sums moves a few of the values that are rounded to
        # int8 behind it by one step (7.5e-4 off 64 bits at batch 512, where 64 bits moves some;
        # one moved value weighs more in a single sequence)
        return {"rel": 1e-2}
    return "exact"                          # int8 products, int32 sums, one IEEE f32 operation per step


# ---------------------------------------------------------------- the same in 64 bits

def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


_STEP = {"add": torch.add, "sub": torch.sub, "mul": torch.mul, "div": torch.div, "maximum": torch.maximum,
         "minimum": torch.minimum}
_UNARY = {"relu": torch.relu, "gelu": _gelu, "sigmoid": torch.sigmoid, "tanh": torch.tanh}


def _f64(a) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV).double()


def _conv(x, w, a: dict):
    """One matrix product per kernel tap (or one product per channel where every channel is its own group)."""
    (sh, sw), (ph, pw) = a["stride"], a["padding"]
    dh, dw = a.get("dilation", (1, 1))
    n, c, hh, ww = x.shape
    o, cg, kh, kw = w.shape
    oh, ow = (hh + 2 * ph - dh * (kh - 1) - 1) // sh + 1, (ww + 2 * pw - dw * (kw - 1) - 1) // sw + 1
    xp = torch.nn.functional.pad(x, (pw, pw, ph, ph))
    acc = torch.zeros((n, o, oh, ow) if cg == 1 and c == o else (n * oh * ow, o), dtype=torch.float64, device=DEV)
    for i in range(kh):
        for j in range(kw):
            t = xp[:, :, i * dh:i * dh + sh * (oh - 1) + 1:sh, j * dw:j * dw + sw * (ow - 1) + 1:sw]
            if acc.dim() == 4:
                acc += t * w[:, 0, i, j].reshape(1, c, 1, 1)
            else:
                acc += t.permute(0, 2, 3, 1).reshape(-1, c) @ w[:, :, i, j].t().contiguous()
    return acc if acc.dim() == 4 else acc.reshape(n, oh, ow, o).permute(0, 3, 1, 2)


def _quantize(x, xs: float):
    return torch.clamp(torch.round(x / float(np.float32(xs))), -127, 127)


def _op(op, xs: list):
    k, a = op.kind, op.attrs
    if k == "const":
        return _f64(a["value"])
    if k == "dequantize":
        shape = [1] * a["q"].ndim
        shape[a["axis"]] = -1
        return _f64(a["q"]) * _f64(a["scale"]).reshape(shape)
    if k in ("qmatmul", "qconv2d"):
        q, s = _f64(a["q"]), float(a["x_scale"]) * _f64(a["w_scale"])
        xq = _quantize(xs[0], a["x_scale"])
        y = (xq @ q) * s if k == "qmatmul" else _conv(xq, q, a) * s.reshape(1, -1, 1, 1)
    elif k == "matmul":
        y = torch.matmul(xs[0], xs[1].contiguous())
    elif k == "conv2d":
        y = _conv(xs[0], xs[1], a)
    elif k == "layernorm":
        mu = xs[0].mean(-1, keepdim=True)
        var = ((xs[0] - mu) ** 2).mean(-1, keepdim=True)
        return (xs[0] - mu) / torch.sqrt(var + a["eps"]) * xs[1] + xs[2]
    elif k == "softmax":
        return torch.softmax(xs[0], a["axis"])
    elif k == "pad":
        (t, b), (l, r) = a["pads"][2:]
        return torch.nn.functional.pad(xs[0], (l, r, t, b), value=float(a.get("value", 0)))
    elif k == "maxpool2d":
        win = xs[0].unfold(2, a["size"], a["stride"]).unfold(3, a["size"], a["stride"])
        return win.amax((-2, -1))
    elif k == "reduce_mean":
        return xs[0].mean(tuple(a["axes"]), keepdim=a["keepdims"])
    elif k == "reshape":
        return xs[0].reshape(tuple(a["shape"]))
    elif k == "transpose":
        return xs[0].permute(tuple(a["perm"]))
    elif k == "concat":
        return torch.cat(xs, a["axis"])
    elif k == "cast":
        return xs[0]
    elif k in _STEP:
        return _STEP[k](xs[0], xs[1])
    elif k in _UNARY:
        return _UNARY[k](xs[0])
    else:
        raise NotImplementedError(k)
    for fn, idx, swapped in a.get("epilogue", ()):
        if idx is None:
            y = _UNARY[fn](y)
        else:
            y = _STEP[fn](xs[idx], y) if swapped else _STEP[fn](y, xs[idx])
    return y


def _evaluate(g: Graph, feeds: dict, keep: list) -> dict:
    """The values of `keep` for these inputs, in float64; others are dropped after their last use."""
    last = {}
    for i, op in enumerate(g.ops):
        for v in op.inputs:
            last[v] = i
    env = {v: t.double() for v, t in feeds.items()}
    kept = set(keep)
    for i, op in enumerate(g.ops):
        env[op.result] = _op(op, [env[v] for v in op.inputs])
        for v in set(op.inputs):
            if last[v] == i and v not in kept:
                env.pop(v, None)
    return {v: env[v] for v in keep}


def exact(case: dict, seed: int):
    if case["kind"] in ("step", "decode"):
        # behind the attention each value is rounded to int8: two correct f32 orders of its sums
        # differ by a whole int8 step at times, and so does 64 bits; `attn` holds that attention
        return None
    g = _graph(case)
    out = _evaluate(g, _inputs(case, g, seed), list(g.outputs))
    outs = [out[v] for v in g.outputs]
    return [t.cpu().numpy() for t in outs] if case.get("host") else outs
