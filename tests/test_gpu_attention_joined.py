"""GPU: the fused attention's backward in one launch (few rows) against the two launches that more rows take: the same heads, by themselves
and at the front of a batch that fills the chip.  dQ and dV have the same bits; dK differs by the order of the f32 row sums of out * grad_out,
D terms, and so by a rounding of the result at most (twice eps of its largest value), and by what stays of the sums themselves where dS cancels."""
import numpy as np
import pytest
import torch

import oracle
from helpers import rng
from gpu_util import announce, device, launches
from test_gpu_attention_fused import reference
from test_gpu_encoder_block import graph_nodes

from dfdx_amd import Rocm, View

pytestmark = pytest.mark.gpu


def backward(dev, dtype, st, B, H, S, D, in_place=False):
    d = H * D
    q, k, v = (dev.tensor(t[:B * S * d], dtype, (B, H, S, D), (S * d, D, d, 1)) for t in st[:3])
    go = dev.tensor(st[3][:B * S * d], dtype, (B, S, d))
    out, lse = dev.attention_forward(q, k, v, D ** -0.5)
    gq, gk, gv = dev.zeros_many([go, go, go], deferred=True)
    if in_place:
        gv = View(v.storage, dtype, (B, S, d), (S * d, d, 1))   # dV is added to V where it lies
    dev.attention_backward(q, gq, k, gk, v, gv, D ** -0.5, out, go, lse)
    dev.synchronize()
    return [oracle.to_f64(dev.to_host(t), dtype) for t in (gq, gk, gv)]


def count(dtype, B, H, S, D):
    """Launches of the backward."""
    def prepare(dev):
        q, k, v, gq, gk, gv = (dev.zeros(dtype, (B, H, S, D)) for _ in range(6))
        go = dev.zeros(dtype, (B, S, H * D))
        out, lse = dev.attention_forward(q, k, v, D ** -0.5)
        return lambda: dev.attention_backward(q, gq, k, gk, v, gv, D ** -0.5, out, go, lse)
    return launches(prepare)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("H,S,D", [(2, 1, 64), (3, 63, 32), (2, 64, 64), (2, 65, 128), (2, 100, 64), (1, 129, 128), (4, 197, 64), (1, 257, 32)])
def test_one_launch_and_two_agree(dtype, H, S, D):
    dev, g = device(), rng(S * 11 + D)
    many = fills_the_chip(dev, H, S)
    n = many * S * H * D
    st = [oracle.to_storage(g.standard_normal(n) * w, dtype) for w in (2.0, 2.0, 1.0, 1.0)]
    announce("attention backward, joined", dtype, H, S, D, many)
    assert [count(dtype, B, H, S, D) for B in (1, many)] == [1, 2]
    few, all_ = backward(dev, dtype, st, 1, H, S, D), backward(dev, dtype, st, many, H, S, D)
    eps = 2.0 ** -11 if dtype == "f16" else 2.0 ** -8
    for name, a, b in zip(("dq", "dk", "dv"), few, all_):
        b = b[:a.size]
        if name == "dk":
            top = [np.abs(oracle.to_f64(t, dtype)).max() for t in st]   # q, k, v, grad_out
            floor = D * 2.0 ** -24 * D * top[2] * top[3] * D ** -0.5 * top[0]
            assert np.abs(a - b).max() <= 2 * eps * np.abs(b).max() + floor, np.abs(a - b).max()
        else:
            assert np.array_equal(a, b), name


def test_a_gradient_where_an_input_lies():
    """Two launches: every workgroup reads the rows of V that it writes, the queries' workgroups have read all of them before."""
    dev, g = device(), rng(5)
    H, S, D = 2, 130, 64
    st = [oracle.to_storage(g.standard_normal(S * H * D), "f16") for _ in range(4)]
    announce("attention backward, dV onto V")
    apart, onto = backward(dev, "f16", st, 1, H, S, D), backward(dev, "f16", st, 1, H, S, D, in_place=True)
    v = oracle.to_f64(st[2], "f16")
    assert np.array_equal(apart[0], onto[0])
    assert np.abs(onto[2] - (apart[2] + v)).max() <= 2.0 ** -10 * np.abs(apart[2] + v).max()


def fills_the_chip(dev, H, S):
    """Images whose workgroups, of both sides, are more than the chip has places for."""
    return -(-dev.device_info()["compute_units"] // (H * -(-S // 128))) + 1


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("shared", ["qkv", "qk", "qv", "kv"])
@pytest.mark.parametrize("deferred", [False, True])
@pytest.mark.parametrize("few", [True, False])
@pytest.mark.parametrize("H,S,D", [(2, 130, 64), (1, 40, 128)])
def test_a_gradient_that_operands_share(dtype, shared, deferred, few, H, S, D):
    """Self-attention on one tensor, and two operands' gradients in one buffer: their sum, few rows (which take one launch where nothing
    is shared) and many.  Each gradient is within eight eps of its largest value (test_gpu_attention_fused.py); what is added to is
    rounded in between, half an eps of the partial sum each time."""
    dev, g = device(), rng(len(shared) + S)
    B, d = (1 if few else fills_the_chip(dev, H, S)), H * D
    announce("attention backward, shared gradient", dtype, shared, deferred, (B, H, S, D))
    st = [oracle.to_storage(g.standard_normal(B * S * d) * w, dtype) for w in (2.0, 2.0, 1.0, 1.0)]
    if shared == "qkv":
        st[1] = st[2] = st[0]
    rows = [oracle.to_f64(t, dtype).reshape(B, S, H, D).swapaxes(1, 2) for t in st]
    want = dict(zip("qkv", reference(*rows, D ** -0.5)[1:]))
    x = {n: dev.tensor(t, dtype, (B, H, S, D), (S * d, D, d, 1)) for n, t in zip("qkv", st)}
    if shared == "qkv":
        x = dict.fromkeys("qkv", x["q"])
    go = dev.tensor(st[3], dtype, (B, S, d))
    out, lse = dev.attention_forward(x["q"], x["k"], x["v"], D ** -0.5)
    one, *others = dev.zeros_many([go] * (4 - len(shared)), deferred=deferred)
    grads = {n: one if n in shared else others[0] for n in "qkv"}
    dev.attention_backward(x["q"], grads["q"], x["k"], grads["k"], x["v"], grads["v"], D ** -0.5, out, go, lse)
    dev.synchronize()
    eps = 2.0 ** -11 if dtype == "f16" else 2.0 ** -8
    top = [np.abs(r).max() for r in rows]
    floor = D * 2.0 ** -24 * D * top[2] * top[3] * D ** -0.5 * max(top[:2])
    for names, buffer in ((shared, one), *((n, others[0]) for n in "qkv" if n not in shared)):
        ref = sum(want[n] for n in names).swapaxes(1, 2).reshape(-1)
        bound = sum(9 * eps * np.abs(want[n]).max() + floor for n in names)
        err = np.abs(oracle.to_f64(dev.to_host(buffer), dtype) - ref).max()
        assert err <= bound, (names, err, bound)


@pytest.mark.parametrize("layout,launches", [("apart", 1), ("packed rows", 1), ("packed heads", 1), ("one buffer", 2), ("half a row on", 2), ("one row on", 2)])
def test_launches(layout, launches):
    """Gradients whose spans interleave without meeting keep the one launch; where rows of dQ and dK meet it takes two."""
    dev, g = device(), rng(3)
    B, H, S, D = 2, 3, 70, 64
    d = H * D
    strides = {"packed rows": (S * 3 * d, D, 3 * d, 1), "packed heads": (S * 3 * d, 3 * D, 3 * d, 1)}.get(layout, (S * d, D, d, 1))
    step = {"apart": B * S * d, "packed rows": d, "packed heads": D, "one buffer": 0, "half a row on": D // 2, "one row on": d}[layout]
    announce("attention backward, launches", layout)
    x = oracle.to_storage(g.standard_normal(5 * B * S * d), "f16")
    torch_stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(torch_stream):
        own = Rocm(0)
        hold, grad = own.tensor(x, "f16"), own.zeros("f16", (x.size,))
        at = (0, step, 2 * step if "packed" in layout else 3 * B * S * d)
        q, k, v = (View(hold.storage, "f16", (B, H, S, D), strides, n) for n in at)
        gq, gk, gv = (View(grad.storage, "f16", (B, H, S, D), strides, n) for n in at)
        go = own.tensor(x[:B * S * d], "f16", (B, S, d))
        out, lse = own.attention_forward(q, k, v, D ** -0.5)
        run = lambda: own.attention_backward(q, gq, k, gk, v, gv, D ** -0.5, out, go, lse)
        run()   # (the workspace has its size before a capture)
        own.synchronize()
        assert graph_nodes(run, torch_stream) == launches
        own.synchronize()
    own.close()
