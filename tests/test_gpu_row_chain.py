"""Runs of row-local ops in one launch (mr_row_chain) against the same ops launched one by one,
and the wave-wide pairwise sums behind their layernorms against the oracle."""
import numpy as np
import pytest

from harness import lowering as LW
from harness import models
from harness.graph import Graph
from harness.runner import Runner
from mira_amd import _lib as L
from mira_amd.target import ROW_CHAIN_ROWS, ROW_CHAIN_WEIGHTS, RocmTarget
from oracle import golden as G

from gpu_util import T, empty, stream, sync

pytestmark = pytest.mark.gpu


def _both(g, exe, feeds) -> tuple:
    """(g's outputs from the launches one by one, from the queued program)."""
    def outputs() -> list:
        return [exe.device_output(v).cpu().numpy().copy() for v in g.outputs]

    exe.upload({v: feeds[v.name] for v in exe.g.inputs})
    for _name, fn in exe.launches:
        fn(stream())
    sync()
    want = outputs()
    for v in g.outputs:
        exe.device_output(v).fill_(-7.0)
    exe.launch()
    sync()
    return want, outputs()


def _mlp(rows: int, widths: list) -> Graph:
    """layernorm -> (matmul, bias, residual or relu)..., quantized."""
    rng = np.random.default_rng(rows + sum(widths))
    g = Graph("chain")
    y = g.input("x", (rows, widths[0]))
    for i, (k, n) in enumerate(zip(widths, widths[1:])):
        r = y
        if i % 2 == 0:
            gain, bias = (rng.standard_normal(k).astype(np.float32) for _ in range(2))
            y = g.op("layernorm", [y, g.const(gain), g.const(bias)], {"eps": 1e-5})
        w = (rng.standard_normal((k, n)) * k ** -0.5).astype(np.float32)
        y = g.op("add", [g.op("matmul", [y, g.const(w)]), g.const(rng.standard_normal(n).astype(np.float32))])
        y = g.op("add", [y, r]) if k == n else g.op("relu", [y])
    g.outputs = [y]
    return g


@pytest.mark.parametrize("rows,widths", [(1, [64, 64, 10]), (2, [17, 33, 33, 5]), (8, [100, 256, 256]), (9, [129, 40, 40]),
                                         (255, [192, 70, 1]), (257, [512, 96, 96, 31]), (511, [64, 1000, 12]),
                                         (512, [48, 48, 100])])
def test_chain_equals_the_launches(rows, widths):
    """Bit for bit: the same int8 products, the same f32 operations per element."""
    g = LW.prepare(_mlp(rows, widths))
    cal = [{"x": np.random.default_rng(s).standard_normal((rows, widths[0])).astype(np.float32)} for s in (2, 3)]
    LW.w8a8(g, cal)
    (exe,) = Runner(g, RocmTarget()).executables("rocm")
    assert len(exe.program) < len(exe.launches)
    want, got = _both(g, exe, cal[0])
    for a, b in zip(want, got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("rows,k", [(64, 320), (ROW_CHAIN_ROWS + 1, 64)])
def test_large_weights_and_many_rows_stay_launches(rows, k):
    assert k * k > ROW_CHAIN_WEIGHTS or rows > ROW_CHAIN_ROWS
    g = LW.prepare(_mlp(rows, [k, k, k]))
    LW.w8a8(g, [{"x": np.random.default_rng(1).standard_normal((rows, k)).astype(np.float32)}])
    (exe,) = Runner(g, RocmTarget()).executables("rocm")
    assert len(exe.program) == len(exe.launches)


@pytest.mark.parametrize("batch,heads,hd,context", [(1, 4, 16, 272), (2, 3, 16, 41), (5, 3, 32, 100), (3, 1, 16, 1),
                                                    (257, 2, 16, 65), (512, 4, 32, 320), (1, 2, 64, 1023), (7, 1, 32, 7)])
def test_chain_attention(batch, heads, hd, context):
    """One layer's attention half, bit for bit: the run keeps attention_decode_kernel's order of
    every f32 sum."""
    d = heads * hd
    rng = np.random.default_rng(batch + d + context)
    g = Graph("attn")
    h, mask = g.input("h", (batch, d)), g.input("mask", (1, 1, 1, context + 1))
    kc, vc = g.input("kc0", (batch, context, d)), g.input("vc0", (batch, context, d))
    x = g.op("layernorm", [h, g.const(np.ones(d, np.float32)), g.const(np.zeros(d, np.float32))], {"eps": 1e-5})
    q, k, v = (g.op("matmul", [x, g.const((rng.standard_normal((d, d)) * d ** -0.5).astype(np.float32))]) for _ in range(3))
    q4 = g.op("transpose", [g.op("reshape", [q], {"shape": (batch, 1, heads, hd)})], {"perm": (0, 2, 1, 3)})
    keys = g.op("concat", [kc, g.op("reshape", [k], {"shape": (batch, 1, d)})], {"axis": 1})
    vals = g.op("concat", [vc, g.op("reshape", [v], {"shape": (batch, 1, d)})], {"axis": 1})
    k4 = g.op("transpose", [g.op("reshape", [keys], {"shape": (batch, context + 1, heads, hd)})], {"perm": (0, 2, 3, 1)})
    v4 = g.op("transpose", [g.op("reshape", [vals], {"shape": (batch, context + 1, heads, hd)})], {"perm": (0, 2, 1, 3)})
    s = g.op("add", [g.op("mul", [g.op("matmul", [q4, k4]), g.const(np.float32(1.0 / np.sqrt(hd)))]), mask])
    o4 = g.op("matmul", [g.op("softmax", [s], {"axis": -1}), v4])
    g.outputs = [g.op("reshape", [g.op("transpose", [o4], {"perm": (0, 2, 1, 3)})], {"shape": (batch, d)}), k, v]
    g = LW.prepare(g)
    feeds = {"h": rng.standard_normal((batch, d)).astype(np.float32),
             "kc0": rng.standard_normal((batch, context, d)).astype(np.float32),
             "vc0": rng.standard_normal((batch, context, d)).astype(np.float32),
             "mask": np.where(np.arange(context + 1) % 3 == 1, np.float32(-10000.0), np.float32(0.0)).reshape(1, 1, 1, -1)}
    LW.w8a8(g, [feeds])
    (exe,) = Runner(g, RocmTarget(approx_f32=True)).executables("rocm")
    assert exe.kernel_counts["attention"] == 1 and len(exe.program) == 1
    want, got = _both(g, exe, feeds)
    for a, b in zip(want, got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_decode_step_matches_the_launches():
    """A whole two-layer step, bit for bit."""
    cfg = models.GPTConfig()
    params = models.gpt_params(cfg, 0)
    g = LW.prepare(models.gpt_decode_step(cfg, 3, params))
    r = np.random.default_rng(5)
    toks = r.integers(0, cfg.V, (3, cfg.T)).astype(np.int32)
    caches = [tuple(r.standard_normal((3, cfg.T, cfg.D)).astype(np.float32) for _ in range(2)) for _ in range(cfg.L)]
    feeds = models.gpt_step_feeds(cfg, params, toks, 20, caches)
    LW.w8a8(g, [feeds])
    (exe,) = Runner(g, RocmTarget(approx_f32=True)).executables("rocm")
    assert len(exe.program) == 1
    want, got = _both(g, exe, feeds)
    for a, b in zip(want, got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("d", [1, 7, 8, 15, 100, 128, 129, 136, 191, 192, 255, 256, 257, 263, 300, 384, 504, 511, 512, 513])
def test_layernorm_pairwise_order(lib, d):
    """NumPy's pairwise order at every depth of the split, bit for bit."""
    rng = np.random.default_rng(d)
    x = (rng.standard_normal((3, d)) * 10 + 3).astype(np.float32)
    gm, bt = rng.standard_normal(d).astype(np.float32), rng.standard_normal(d).astype(np.float32)
    want = G.layernorm([x, gm, bt], {"eps": 1e-5})
    dx, dg, db = T(x), T(gm), T(bt)
    y = empty((3, d), dx.dtype)
    L.check(lib.mr_layernorm_f32(dx.data_ptr(), 3, d, dg.data_ptr(), db.data_ptr(), 1e-5, 0, y.data_ptr(), None, 0, 1.0,
                                 stream()), "layernorm")
    sync()
    assert np.array_equal(y.cpu().numpy().view(np.uint32), np.asarray(want).view(np.uint32))
