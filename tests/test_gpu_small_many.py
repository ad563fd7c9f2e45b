"""Two or three small products in one launch (launch_small_many of gemm_small.hip): the bits of separate launches, whatever the waves
and passes of each, and one behind the other where they share a result."""
import numpy as np
import pytest

import oracle
from gpu_util import announce, device
from helpers import rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "f64"])
@pytest.mark.parametrize("rows,i,o", [(64, 512, 256), (17, 33, 5), (1, 40, 24), (130, 16, 300), (20, 232, 978), (48, 2100, 40), (400, 31, 30)])
def test_backward_of_a_small_linear_layer(dtype, rows, i, o):
    """1 to 16 waves and one pass or more on either side.  Whole numbers below 2^11: the sums are exact, one rounding each."""
    dev, g = device(), rng(rows + i + o)
    announce("small pair", dtype, rows, i, o)
    x, w, go = (oracle.to_storage(g.integers(-2, 3, size=s).astype(np.float64), dtype) for s in ((rows, i), (o, i), (rows, o)))
    dx, dw, dgo = (dev.tensor(t, dtype) for t in (x, w, go))
    X, W, G = (oracle.to_f64(t, dtype).reshape(t.shape) for t in (x, w, go))
    host = lambda t, shape: oracle.to_f64(dev.to_host(t), dtype)[:int(np.prod(shape))].reshape(shape)
    rounded = lambda v: oracle.to_f64(oracle.to_storage(v, dtype), dtype).reshape(v.shape)
    gx, gw, gb = dev.zeros_many([dx, dw, dev.zeros(dtype, (o,))], deferred=True)
    before = [np.zeros(s) for s in ((rows, i), (o, i), (o,))]
    for _ in range(2):   # into fresh gradients, then onto them
        dev.linear_backward(dx, gx, dw, gw, gb, dgo)
        want = [rounded(b + v) for b, v in zip(before, (G @ W, G.T @ X, G.sum(axis=0)))]
        for got, v in zip((gx, gw, gb), want):
            np.testing.assert_array_equal(host(got, v.shape), v)
        before = want
    # the separate calls that one launch stands for
    sx, sw = dev.zeros(dtype, (rows, i)), dev.zeros(dtype, (o, i))
    x2, go2 = (dev.tensor(oracle.to_storage(g.standard_normal(s), dtype), dtype) for s in ((rows, i), (rows, o)))
    dev.gemm(dev.gemm_desc(dtype, rows, o, i, go2.ptr, (o, 1), dw.ptr, (i, 1), sx.ptr, (i, 1), accumulate=True))
    dev.gemm(dev.gemm_desc(dtype, i, rows, o, x2.ptr, (1, i), go2.ptr, (o, 1), sw.ptr, (1, i), accumulate=True))
    jx, jw = dev.zeros(dtype, (rows, i)), dev.zeros(dtype, (o, i))
    wt = dw.permute(1, 0)
    dev.backward(x2, jx, wt, jw.permute(1, 0), go2)
    if "small" in dev.gemm_plan(dev.gemm_desc(dtype, i, rows, o, x2.ptr, (1, i), go2.ptr, (o, 1), sw.ptr, (1, i), accumulate=True))[2] and dtype in ("f32", "f64"):
        np.testing.assert_array_equal(host(jx, (rows, i)), host(sx, (rows, i)))
        np.testing.assert_array_equal(host(jw, (o, i)), host(sw, (o, i)))


@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_one_buffer_for_both_gradients(dtype):
    """x . x: the second product adds to what the first has stored."""
    dev, g, n = device(), rng(5), 40
    announce("small pair, one gradient", dtype)
    x, go = (g.integers(-3, 4, size=(n, n)).astype(np.float64) for _ in range(2))
    dx, dgo = (dev.tensor(oracle.to_storage(t, dtype), dtype) for t in (x, go))
    gx = dev.zeros_like_storage(dx)
    dev.backward(dx, gx, dx, gx, dgo)
    np.testing.assert_array_equal(oracle.to_f64(dev.to_host(gx), dtype).reshape(n, n), go @ x.T + x.T @ go)
