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
