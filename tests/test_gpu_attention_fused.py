"""GPU: the fused attention entry points (softmax(scale * q.k^T).v without the score matrix) against a float64 evaluation of
the same formulas on the same rounded inputs, forward and the three gradients, at the edges of their tiles: 64 staged
rows, 32 rows per wave, 128 per workgroup.  Tolerance: the operands of the second products (probabilities, dS) and the
results are each rounded once to the element type, eps = 2^-11 (f16) or 2^-8 (bf16) of the largest value at most; the
sums run over 2 * S such terms, whose errors are independent, so eight eps of the tensor's largest value bound them."""
import numpy as np
import pytest

import oracle
from helpers import rng
from gpu_util import announce, device

pytestmark = pytest.mark.gpu

from dfdx_amd import View  # noqa: E402


def reference(q, k, v, g, scale):
    s = scale * q @ k.swapaxes(-1, -2)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    out = p @ v
    dp = g @ v.swapaxes(-1, -2)
    ds = p * (dp - (dp * p).sum(-1, keepdims=True))
    return out, scale * ds @ k, scale * ds.swapaxes(-1, -2) @ q, p.swapaxes(-1, -2) @ g


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("B,H,S,D", [(1, 1, 1, 64), (2, 3, 31, 32), (1, 2, 64, 64), (2, 2, 65, 128), (1, 3, 128, 32), (1, 2, 129, 64),
                                     (1, 1, 200, 128), (2, 1, 321, 64)])
def test_fused_attention(dtype, B, H, S, D):
    dev = device()
    announce("attention", dtype, (B, H, S, D))
    g = rng(S * 7 + D)
    d = H * D
    st = [oracle.to_storage(g.standard_normal(B * S * d) * w, dtype) for w in (2.0, 2.0, 1.0, 1.0)]   # token layout (B, S, H, D)
    qv, kv, vv, gv = (oracle.to_f64(t, dtype).reshape(B, S, H, D).swapaxes(1, 2) for t in st)
    scale = D ** -0.5
    want = reference(qv, kv, vv, gv, scale)
    q, k, v = (dev.tensor(t, dtype, (B, H, S, D), (S * d, D, d, 1)) for t in st[:3])
    go = dev.tensor(st[3], dtype, (B, S, d))
    out, lse = dev.attention_forward(q, k, v, scale)
    old = oracle.to_storage(g.standard_normal(B * S * d), dtype)   # dV is added to what is there; dQ, dK are declared zero
    gq, gk = dev.zeros_many([go, go], deferred=True)
    gvv = dev.tensor(old, dtype, (B, S, d))
    dev.attention_backward(q, gq, k, gk, v, gvv, scale, out, go, lse)
    again = dev.zeros(dtype, (B, S, d))
    dev.attention_backward(q, again, k, dev.zeros(dtype, (B, S, d)), v, dev.zeros(dtype, (B, S, d)), scale, out, go, lse)
    dev.synchronize()
    eps = 2.0 ** -11 if dtype == "f16" else 2.0 ** -8
    for name, got, ref, base in zip(("out", "dq", "dk", "dv"), (out, gq, gk, gvv), want, (0, 0, 0, oracle.to_f64(old, dtype))):
        ref = ref.swapaxes(1, 2).reshape(-1) + base
        err = np.abs(oracle.to_f64(dev.to_host(got), dtype) - ref).max()
        # dS subtracts two f32 sums of D products of v and g, each within D * 2^-24 of the sum of their magnitudes: where they
        # cancel (S = 1: the gradient is exactly zero) this much, times a value of q or k, is what stays
        floor = D * 2.0 ** -24 * D * np.abs(vv).max() * np.abs(gv).max() * scale * max(np.abs(qv).max(), np.abs(kv).max())
        assert err <= 8 * eps * np.abs(ref).max() + (floor if name in ("dq", "dk") else 0.0), (name, err, np.abs(ref).max())
    assert np.array_equal(dev.to_host(again), dev.to_host(gq)), "dQ: stored and added to zeros differ"


def test_fused_attention_refuses_what_it_does_not_take():
    from dfdx_amd import RocmError

    dev = device()
    for dtype, D in (("f32", 64), ("f16", 80)):
        x = dev.zeros(dtype, (1, 1, 4, D))
        with pytest.raises(RocmError):
            dev.attention_forward(x, x, x, 0.125)
        assert not dev.attention_supported(dtype, D)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("strides", [(0, 64, 128), (8192, 0, 128), (8192, 64, 56), (8192, 32, 128)],
                         ids=["one batch for all", "one head for all", "rows shorter than a head", "heads inside each other"])
def test_gradients_that_would_share_rows_are_refused(dtype, strides):
    """Views of q, k, v whose rows overlap are read by the forward (the same as on copies of them); their gradients would be
    added by several workgroups without order, and are refused with nothing written."""
    from dfdx_amd import RocmError
    from dfdx_amd.rocm import ERR_ALIASED_OUTPUT

    dev = device()
    B, H, S, D = 2, 2, 64, 64
    announce("attention, aliased", dtype, strides)
    g = rng(5)
    size = 1 + sum((n - 1) * s for n, s in zip((B, H, S, D), (*strides, 1)))
    st = [oracle.to_storage(g.standard_normal(size), dtype) for _ in range(3)]
    q, k, v = (dev.tensor(t, dtype, (B, H, S, D), (*strides, 1)) for t in st)
    flat = [np.lib.stride_tricks.as_strided(t, (B, H, S, D), [x * t.itemsize for x in (*strides, 1)]).copy().reshape(-1) for t in st]
    out, lse = dev.attention_forward(q, k, v, 0.125)
    same, _ = dev.attention_forward(*(dev.tensor(t, dtype, (B, H, S, D)) for t in flat), 0.125)
    assert np.array_equal(dev.to_host(out), dev.to_host(same))
    grads = [dev.tensor(np.zeros_like(st[0]), dtype) for _ in range(3)]
    with pytest.raises(RocmError) as err:
        dev.attention_backward(q, grads[0], k, grads[1], v, grads[2], 0.125, out, out, lse)
    assert err.value.code == ERR_ALIASED_OUTPUT
    assert all(not dev.to_host(t).any() for t in grads)


def test_results_that_would_share_rows_are_refused():
    dev = device()
    announce("attention, aliased result")
    B, H, S, D = 2, 2, 16, 64
    x = dev.zeros("f16", (B, H, S, D))
    from dfdx_amd.rocm import DTYPES, ERR_ALIASED_OUTPUT, _i64s

    for strides in ((0, D, H * D), (S * H * D, 0, H * D), (S * H * D, D, D)):
        rc = dev._f.attention_forward(dev.ctx, DTYPES["f16"], B, H, S, D, x.ptr, x.ptr, x.ptr, _i64s(x.strides[:3]), 0.125, x.ptr, _i64s(strides), None)
        assert rc == ERR_ALIASED_OUTPUT, strides


@pytest.mark.parametrize("wrong", ["grad_out", "lse", "small gradient", "strides of v"])
def test_backward_looks_at_its_arguments(wrong):
    dev = device()
    B, H, S, D = 1, 2, 16, 64
    x, rows = dev.zeros("f16", (B, H, S, D)), dev.zeros("f16", (B, S, H * D))
    lse = dev.zeros("f32", (B, H, S))
    v, go, gv = x, rows, dev.zeros("f16", (B, H, S, D))
    if wrong == "grad_out":
        go = dev.zeros("f16", (B, H, S, D))
    elif wrong == "lse":
        lse = dev.zeros("f16", (B, H, S))
    elif wrong == "small gradient":
        gv = dev.zeros("f16", (B, 1, S, D))
    else:
        v = dev.zeros("f16", (B, S, H, D)).permute(0, 2, 1, 3)
    with pytest.raises(AssertionError):
        dev.attention_backward(x, dev.zeros("f16", (B, H, S, D)), x, dev.zeros("f16", (B, H, S, D)), v, gv, 0.125, rows, go, lse)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("case,S", [("last value", 65), ("last value", 200), ("first tile of keys", 130), ("first tile of keys", 64 + 17), ("last key", 65),
                                    ("last gradient", 65), ("last gradient", 127)])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_infinities_reach_what_depends_on_them_and_nothing_else(dtype, case, S, D):
    """The kernels work in tiles of 64 rows: what fills a tile up, and what a row's maximum starts from, may not meet an infinity.
    Infinities and NaN as in the float64 formulas, finite values within the tolerance above (with one rounding of the largest finite one)."""
    dev = device()
    announce("attention, infinities", dtype, case, S, D)
    B, H = 1, 2
    d = H * D
    g = rng(S + D)
    st = [oracle.to_storage(np.abs(g.standard_normal(B * S * d)) * w, dtype) for w in (0.5, 0.5, 1.0, 1.0)]
    at = lambda t, rows: t.reshape(S, d)[rows, 3:4]   # one column of the first head
    inf = oracle.to_storage(np.array([np.inf]), dtype)[0]
    minus = oracle.to_storage(np.array([-np.inf]), dtype)[0]
    if case == "last value":
        at(st[2], slice(S - 1, S))[:] = inf
    elif case == "first tile of keys":
        at(st[1], slice(0, 64))[:] = minus     # (the queries are positive: scores of -infinity)
    elif case == "last key":
        at(st[1], slice(S - 1, S))[:] = minus
    else:
        at(st[3], slice(S - 1, S))[:] = inf
    qv, kv, vv, gv = (oracle.to_f64(t, dtype).reshape(B, S, H, D).swapaxes(1, 2) for t in st)
    scale = D ** -0.5
    with np.errstate(invalid="ignore"):
        want = reference(qv, kv, vv, gv, scale)
    q, k, v = (dev.tensor(t, dtype, (B, H, S, D), (S * d, D, d, 1)) for t in st[:3])
    go = dev.tensor(st[3], dtype, (B, S, d))
    out, lse = dev.attention_forward(q, k, v, scale)
    grads = dev.zeros_many([go, go, go], deferred=True)
    dev.attention_backward(q, grads[0], k, grads[1], v, grads[2], scale, out, go, lse)
    eps = 2.0 ** -11 if dtype == "f16" else 2.0 ** -8
    for name, got, ref in zip(("out", "dq", "dk", "dv"), (out, *grads), want):
        if case == "last value" and name != "out":
            continue   # (the gradients of an infinite result: out * grad_out and grad_out . v differ in which of them are NaN)
        ref = ref.swapaxes(1, 2).reshape(-1)
        got = oracle.to_f64(dev.to_host(got), dtype)
        assert np.array_equal(np.isnan(got), np.isnan(ref)), (name, np.isnan(got).sum(), np.isnan(ref).sum())
        assert np.array_equal(got[np.isinf(got)], ref[np.isinf(ref)]) and np.array_equal(np.isinf(got), np.isinf(ref)), name
        ok = np.isfinite(ref)
        assert ok.any() or name != "out"
        most = lambda t: np.abs(t[np.isfinite(t)]).max()
        floor = D * 2.0 ** -24 * D * most(vv) * most(gv) * scale * max(most(qv), most(kv))   # as in test_fused_attention
        if ok.any():
            err = np.abs(got[ok] - ref[ok]).max()
            assert err <= 8 * eps * np.abs(ref[ok]).max() + floor * (name in ("dq", "dk")), (name, err)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("S,D", [(65, 64), (130, 32), (33, 128)])
@pytest.mark.parametrize("layout", ["heads in front", "one of three in a row", "padded rows"])
def test_strides_and_offsets(dtype, S, D, layout):
    """Views of other strides than the token layout, offsets of whole 16-byte pieces included: the same sums in the same order, so
    the bits of contiguous tokens, and nothing written between the rows of a gradient."""
    dev = device()
    B, H = 2, 3
    announce("attention, strides", dtype, S, D, layout)
    d = H * D
    strides, offset, size = {"heads in front": ((H * S * D, S * D, D), 0, B * S * d), "one of three in a row": ((S * 3 * d, D, 3 * d), d, B * S * 3 * d),
                             "padded rows": ((S * (d + 16), D, d + 16), 8, B * S * (d + 16) + 8)}[layout]
    g = rng(S + D)
    at = offset + sum(np.arange(n).reshape([-1 if i == j else 1 for j in range(4)]) * s for i, (n, s) in enumerate(zip((B, H, S, D), (*strides, 1))))
    tokens = [oracle.to_storage(g.standard_normal(B * S * d), dtype) for _ in range(4)]
    spread = []
    for t in tokens[:3]:
        u = np.zeros(size, t.dtype)
        u[at] = t.reshape(B, S, H, D).swapaxes(1, 2)
        spread.append(u)
    token = (S * d, D, d, 1)
    go = dev.tensor(tokens[3], dtype, (B, S, d))

    def both(storages, st, off):
        q, k, v = (View(dev.tensor(t, dtype).storage, dtype, (B, H, S, D), st, off) for t in storages)
        out, lse = dev.attention_forward(q, k, v, D ** -0.5)
        grads = [View(dev.zeros(dtype, (len(storages[0]),)).storage, dtype, (B, H, S, D), st, off) for _ in range(3)]
        dev.attention_backward(q, grads[0], k, grads[1], v, grads[2], D ** -0.5, out, go, lse)
        return dev.to_host(out), [dev.to_host(View(t.storage, dtype, (), ())) for t in grads]

    out, grads = both(spread, (*strides, 1), offset)
    want, wgrads = both(tokens[:3], token, 0)
    assert np.array_equal(out.view(np.uint16), want.view(np.uint16))
    for a, b in zip(grads, wgrads):
        assert np.array_equal(a[at].view(np.uint16), b.reshape(B, S, H, D).swapaxes(1, 2).view(np.uint16))
        a[at] = 0
        assert not a.any()


@pytest.mark.parametrize("wrong", ["address", "row stride", "scale", "result's address"])
def test_what_the_pieces_of_16_bytes_cannot_walk_is_refused(wrong):
    from dfdx_amd import RocmError
    from dfdx_amd.rocm import DTYPES, _i64s

    dev = device()
    B, H, S, D = 1, 2, 16, 64
    room = dev.zeros("f16", (B, S, H * (D + 8) + 64))
    strides = (S * H * D, D, H * D + (4 if wrong == "row stride" else 0))
    x = View(room.storage, "f16", (B, H, S, D), (*strides, 1), 1 if wrong == "address" else 0)
    scale, out = 0.0 if wrong == "scale" else 0.125, dev.zeros("f16", (B, S, H * D + 8))
    rc = dev._f.attention_forward(dev.ctx, DTYPES["f16"], B, H, S, D, x.ptr, x.ptr, x.ptr, _i64s(strides), scale,
                                  out.ptr + (2 if wrong == "result's address" else 0), _i64s((S * H * D, D, H * D)), None)
    assert rc == -2   # DFDX_ROCM_ERR_UNSUPPORTED
    if wrong != "result's address":
        with pytest.raises(RocmError):
            dev.attention_forward(x, x, x, scale)
