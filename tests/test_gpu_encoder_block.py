"""GPU: the encoder block's two calls against the same block strung together from the single entry points (Linear, the fused
attention or its ops, LayerNorm, ReLU, add and their backward).  What the block's products do on the way into their results (ReLU,
residual, ReLU's gradient, a first contribution read from elsewhere) rounds where the separate op would, so the output and the
gradients are equal bit for bit, but for two things.  In 16 bits grad_x is one f32 sum rounded once where the single calls round four;
and where ReLU's gradient is cheap enough as a small product on its own, the plan differs from that of a product that adds
to its result, and with it the order of the sum.  These are bounded per element and in the norm.  The shapes reach the small, the split and
the tiled kernels, whole tiles and edges."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from helpers import rng
from gpu_util import announce, device

pytestmark = pytest.mark.gpu

from dfdx_amd import EncoderBlock, Rocm, View  # noqa: E402
from dfdx_amd.encoder import PARAMS  # noqa: E402


def by_ops(dev, dtype, p, x, go, H):
    B, S, d = x.shape
    D, scale = d // H, (d // H) ** -0.5
    zeros = lambda v: dev.zeros(dtype, v.shape)
    q, k, v = (dev.linear_forward(x, p["w" + n], p["b" + n]) for n in "qkv")
    heads = lambda t, *perm: View(t.storage, dtype, (B, S, H, D), (S * d, d, D, 1)).permute(*perm)
    qv, vv, kv, kt = heads(q, 0, 2, 1, 3), heads(v, 0, 2, 1, 3), heads(k, 0, 2, 1, 3), heads(k, 0, 2, 3, 1)
    fused = dev.attention_supported(dtype, D)
    if fused:
        tok, lse = dev.attention_forward(qv, kv, vv, scale)
    else:
        probs = dev.softmax_forward(dev.forward(qv, kt), scale)
        tokens = dev.forward(probs, vv)
        tok = dev.reshape_forward(tokens.permute(0, 2, 1, 3), (B, S, d))
    h1 = dev.add_forward(dev.linear_forward(tok, p["wo"], p["bo"]), x)
    n1 = dev.layer_norm_forward(h1, p["g1"], p["be1"])
    r1 = dev.relu_forward(dev.linear_forward(n1, p["w1"], p["b1"]))
    h2 = dev.add_forward(dev.linear_forward(r1, p["w2"], p["b2"]), n1)
    out = dev.layer_norm_forward(h2, p["g2"], p["be2"])
    g = {n: zeros(p[n]) for n in PARAMS}
    gh2, gn1, gr1, gf1, gh1, gx, gtok, gq, gk, gv = (zeros(t) for t in (x, x, r1, r1, x, x, x, x, x, x))
    dev.layer_norm_backward(h2, p["g2"], gh2, g["g2"], g["be2"], go)
    dev.linear_backward(r1, gr1, p["w2"], g["w2"], g["b2"], gh2)
    dev.relu_backward(r1, gf1, gr1)
    dev.add_backward(gn1, zeros(x), gh2)
    dev.linear_backward(n1, gn1, p["w1"], g["w1"], g["b1"], gf1)
    dev.layer_norm_backward(h1, p["g1"], gh1, g["g1"], g["be1"], gn1)
    dev.add_backward(gx, zeros(x), gh1)
    dev.linear_backward(tok, gtok, p["wo"], g["wo"], g["bo"], gh1)
    if fused:
        dev.attention_backward(qv, gq, kv, gk, vv, gv, scale, tok, gtok, lse)
    else:
        gtokens, gp, gs = zeros(tokens), zeros(probs), zeros(probs)
        dev.reshape_backward(tokens.permute(0, 2, 1, 3), gtokens, gtok)
        dev.backward(probs, gp, vv, gv, gtokens)
        dev.softmax_backward(probs, gs, gp, scale)
        dev.backward(qv, gq, kt, gk, gs)
    for n, gg in zip("qkv", (gq, gk, gv)):
        dev.linear_backward(x, gx, p["w" + n], g["w" + n], g["b" + n], gg)
    return out, g, gx


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("B,S,d,H,ff", [(1, 1, 64, 1, 64), (2, 33, 120, 3, 200), (3, 100, 256, 4, 1024), (1, 257, 512, 4, 2048), (4, 300, 1024, 16, 4096)])
def test_block_equals_its_ops(dtype, B, S, d, H, ff):
    dev = device()
    announce("encoder block", dtype, (B, S, d, H, ff))
    g = rng(d + S)
    up = lambda shape, s: dev.tensor(oracle.to_storage((g.standard_normal(int(np.prod(shape))) * s).astype(np.float32), dtype), dtype, shape)
    shapes = {n: (d, d) for n in ("wq", "wk", "wv", "wo")} | {"w1": (ff, d), "w2": (d, ff), "b1": (ff,)}
    p = {n: up(shapes.get(n, (d,)), 1.0 if n in ("g1", "g2") else 0.05) for n in PARAMS}
    x, go = up((B, S, d), 1.0), up((B, S, d), 1.0)
    block = EncoderBlock(dev, dtype, d, H, ff, p)
    out, saved = block.forward(x)
    grads, gx = block.backward(saved, go)
    want, wg, wgx = by_ops(dev, dtype, p, x, go, H)
    dev.synchronize()
    pairs = {"out": (out, want), "x": (gx, wgx)} | {n: (grads[n], wg[n]) for n in PARAMS}
    eps = {"f16": 2.0 ** -12, "bf16": 2.0 ** -9, "f32": 0.0}[dtype]
    behind_relu = ("wq", "bq", "wk", "bk", "wv", "bv", "wo", "bo", "g1", "be1", "w1", "b1")   # what ReLU's gradient reaches
    for n, (a, b) in pairs.items():
        a, b = (oracle.to_f64(dev.to_host(t), dtype)[:int(np.prod(b.shape))] for t in (a, b))
        if dtype == "f32" or not (n == "x" or (n in behind_relu and (B, S, d) == (3, 100, 256))):
            assert np.array_equal(a, b), (n, np.abs(a - b).max())
        elif n != "bk":   # a shift of all scores of a row: its gradient is the rounding of zero
            assert np.linalg.norm(a - b) <= 5 * (4e-6 + eps) * np.linalg.norm(b), (n, np.linalg.norm(a - b) / np.linalg.norm(b))
            # five roundings of sums that are twice the largest result at most, each half a unit in the last place (2 eps)
            assert np.abs(a - b).max() <= 20 * eps * np.abs(b).max(), (n, np.abs(a - b).max() / np.abs(b).max())
    assert saved["f1"].shape == (B, S, ff) and saved["probs"].shape == (B, H, S, S) and saved["tokens"].shape == (B, H, S, d // H)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("B,S,d,H", [(2, 64, 256, 4), (16, 128, 512, 8), (3, 100, 256, 4)])
def test_block_does_not_depend_on_where_its_parameters_lie(dtype, B, S, d, H):
    """The three projections run as one launch that walks from one matrix to the next by their distance: the same bits with
    the parameters in one buffer in reverse order (negative distances, gaps) as with each in its own."""
    dev, g, ff = device(), rng(d + S), 2 * d
    shapes = {n: (d, d) for n in ("wq", "wk", "wv", "wo")} | {"w1": (ff, d), "w2": (d, ff), "b1": (ff,)}
    host = {n: oracle.to_storage((g.standard_normal(int(np.prod(shapes.get(n, (d,))))) * 0.05 + (n in ("g1", "g2"))).astype(np.float32), dtype) for n in PARAMS}
    own = {n: dev.tensor(host[n], dtype, shapes.get(n, (d,))) for n in PARAMS}
    order, at, pos = list(PARAMS)[::-1], {}, 0
    for i, n in enumerate(order):
        at[n] = pos
        pos += host[n].size + 8 * (i % 3)
    flat = np.zeros(pos, dtype=host["wq"].dtype)
    for n in order:
        flat[at[n]:at[n] + host[n].size] = host[n]
    arena = dev.tensor(flat, dtype)
    one = {n: View(arena.storage[2 * at[n]:2 * (at[n] + host[n].size)], dtype, own[n].shape, own[n].strides) for n in PARAMS}
    x, go = (dev.tensor(oracle.to_storage(g.standard_normal(B * S * d).astype(np.float32), dtype), dtype, (B, S, d)) for _ in range(2))
    results = []
    for p in (own, one):
        block = EncoderBlock(dev, dtype, d, H, ff, p)
        out, saved = block.forward(x)
        grads, gx = block.backward(saved, go)
        results.append([dev.to_host(t) for t in (out, gx, *(grads[n] for n in PARAMS))])
    for a, b in zip(*results):
        assert np.array_equal(a.view(np.uint16), b.view(np.uint16))


@pytest.mark.parametrize("dtype", ["f16", "f32", "f64"])
@pytest.mark.parametrize("B,S", [(0, 5), (2, 0), (0, 0)])
def test_no_tokens(dtype, B, S):
    """An empty batch: an empty result, and gradients that are sums over nothing."""
    dev, d, ff, H = device(), 64, 128, 2
    announce("encoder block, no tokens", dtype, B, S)
    shapes = {n: (d, d) for n in ("wq", "wk", "wv", "wo")} | {"w1": (ff, d), "w2": (d, ff), "b1": (ff,)}
    p = {n: dev.zeros(dtype, shapes.get(n, (d,))) for n in PARAMS}
    block = EncoderBlock(dev, dtype, d, H, ff, p)
    out, saved = block.forward(dev.zeros(dtype, (B, S, d)))
    grads, gx = block.backward(saved, dev.zeros(dtype, (B, S, d)))
    dev.synchronize()
    assert out.shape == gx.shape == (B, S, d)
    for n in PARAMS:
        assert grads[n].shape == p[n].shape and not dev.to_host(grads[n]).any(), n


def a_block(dtype, B, S, d, H, ff, seed=3, **more):
    dev, g = device(), rng(seed)
    up = lambda shape, s: dev.tensor(oracle.to_storage((g.standard_normal(int(np.prod(shape))) * s).astype(np.float32), dtype), dtype, shape)
    shapes = {n: (d, d) for n in ("wq", "wk", "wv", "wo")} | {"w1": (ff, d), "w2": (d, ff), "b1": (ff,)}
    p = {n: up(shapes.get(n, (d,)), 1.0 if n in ("g1", "g2") else 0.05) for n in PARAMS}
    return EncoderBlock(dev, dtype, d, H, ff, p, **more), up((B, S, d), 1.0), up((B, S, d), 1.0)


KEPT = {"x", "qv", "kv", "vv", "probs", "tokens", "tok", "h1", "n1", "f1", "r1", "h2", "scale", "folded"}


@pytest.mark.parametrize("dtype,d,H", [("f16", 128, 2), ("bf16", 128, 2), ("f32", 128, 2), ("f64", 96, 2), ("f16", 96, 4), ("f32", 4, 1)])
@pytest.mark.parametrize("deferred", [True, False])
def test_backward_takes_any_dict_of_the_names(dtype, d, H, deferred):
    """A plain copy of what the forward returned goes through the single ops: the same gradients up to the roundings in between
    (the bound of test_block_equals_its_ops; the probabilities are rounded there)."""
    dev = device()
    B, S, ff = 2, 33, 2 * d
    announce("encoder block, plain dict", dtype, d, H, deferred)
    block, x, go = a_block(dtype, B, S, d, H, ff, deferred_zeros=deferred)
    _, saved = block.forward(x)
    want, wx = block.backward(saved, go)
    assert set(saved) == set(saved.keys()) == KEPT and len(saved) == len(KEPT) and all(n in saved for n in KEPT) and saved.get("nothing", 7) == 7
    plain = dict(saved)
    assert type(plain) is dict and set(plain) == KEPT and saved["tokens"].strides == (H * S * (d // H), S * (d // H), d // H, 1)
    got, gx = block.backward(plain, go)
    dev.synchronize()
    eps = {"f16": 2.0 ** -12, "bf16": 2.0 ** -9, "f32": 2.0 ** -24, "f64": 2.0 ** -53}[dtype]
    for n, a, b in [("x", gx, wx)] + [(n, got[n], want[n]) for n in PARAMS if n != "bk"]:
        a, b = (oracle.to_f64(dev.to_host(t), dtype)[:int(np.prod(b.shape))] for t in (a, b))
        # scores and probabilities rounded to the type on one side: two more roundings in front of the gradients of the attention
        assert np.linalg.norm(a - b) <= 20 * eps * np.linalg.norm(b) + 1e-6 * (dtype == "f32") * np.linalg.norm(b), (n, np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("how", ["replaced", "changed in place", "changed in the arena"])
def test_backward_uses_what_the_caller_put_there(how):
    """Zeros in the place of the ReLU's output (or of the probabilities) leave no gradient for what is behind it."""
    dev = device()
    block, x, go = a_block("f16", 2, 33, 128, 2, 256)
    announce("encoder block, saved values", how)
    _, saved = block.forward(x)
    if how == "replaced":
        saved["r1"] = dev.zeros("f16", saved["r1"].shape)
        none = ("w2", "w1", "b1")
    elif how == "changed in the arena":
        saved["r1"].storage.zero_()
        none = ("w2", "w1", "b1")
    else:
        saved["probs"].storage.zero_()
        none = ("wv", "bv", "wq", "bq", "wk")
    grads, _ = block.backward(saved, go)
    dev.synchronize()
    for n in PARAMS:
        if n != "bk":
            assert bool(dev.to_host(grads[n]).astype(np.float32).any()) == (n not in none), n


def test_no_stale_value_is_made():
    """f1 is not kept: asked for after its weights have changed, it is refused instead of made from other weights."""
    block, x, go = a_block("f16", 1, 9, 64, 1, 128)
    _, saved = block.forward(x)
    before = device().to_host(saved["f1"]).copy()
    _, late = block.forward(x)
    want, _ = block.backward(late, go)
    block.p["w1"].storage.zero_()
    with pytest.raises(RuntimeError):
        late["f1"]
    assert np.array_equal(device().to_host(saved["f1"]), before)
    assert set(late) == KEPT


def graph_nodes(run, stream):
    """Launches of `run`: the nodes of the graph it is captured into."""
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=stream):
        keep = run()
    with open("/proc/self/maps") as maps:
        hip = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    n = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    del keep
    return n.value


@pytest.mark.parametrize("shape,forward,backward", [((16, 128, 512, 8, 1024), 7, None), ((16, 512, 1024, 16, 4096), 7, 18)])
def test_three_projections_are_one_launch(shape, forward, backward):
    """Forward: the projections, the attention, three products and two LayerNorms.  Backward: two launches for each LayerNorm
    and for the attention, four input gradients (one for all projections) and four weight gradients with their combines."""
    block, x, go = a_block("bf16", *shape)
    announce("encoder block, launches", shape)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        own = Rocm(0)
        block = EncoderBlock(own, "bf16", *shape[2:], block.p)
        _, saved = block.forward(x)
        block.backward(saved, go)   # (the workspaces have their sizes before a capture)
        own.synchronize()
        assert graph_nodes(lambda: block.forward(x), stream) == forward
        assert backward is None or graph_nodes(lambda: block.backward(saved, go), stream) == backward
        own.synchronize()
    own.close()
