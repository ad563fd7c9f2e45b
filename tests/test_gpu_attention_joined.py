"""GPU: the fused attention's backward in one launch (few rows) against the two launches that more rows take: the same heads, by themselves
and at the front of a batch that fills the chip.  dQ and dV have the same bits; dK differs by the order of the f32 row sums of out * grad_out,
D terms, and so by a rounding of the result at most (twice eps of its largest value), and by what stays of the sums themselves where dS cancels."""
import numpy as np
import pytest

import oracle
from helpers import rng
from gpu_util import announce, device

from dfdx_amd import View

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


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("H,S,D", [(2, 1, 64), (3, 63, 32), (2, 64, 64), (2, 65, 128), (2, 100, 64), (1, 129, 128), (4, 197, 64), (1, 257, 32)])
def test_one_launch_and_two_agree(dtype, H, S, D):
    dev, g = device(), rng(S * 11 + D)
    many = -(-dev.device_info()["compute_units"] // (H * -(-S // 128))) + 1   # images whose workgroups fill the chip more than once
    n = many * S * H * D
    st = [oracle.to_storage(g.standard_normal(n) * w, dtype) for w in (2.0, 2.0, 1.0, 1.0)]
    announce("attention backward, joined", dtype, H, S, D, many)
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
