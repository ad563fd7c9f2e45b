"""Two or three small products in one launch (launch_small_many of gemm_small.hip): the bits of separate launches, whatever the waves
and passes of each, and one behind the other where they share a result."""
import numpy as np
import pytest

import oracle
from dfdx_amd.rocm import ITEMSIZE
import test_gpu_encoder_block
from gpu_util import announce, device, launches
from helpers import rng

pytestmark = pytest.mark.gpu


def joined(dev, dtype, rows, i, o):
    """Do both products run on the small-product kernel by themselves?  (Those of the 16-bit types with an extent off the grid of eight: the
    others may be one launch of the ring tiles.)"""
    p = dev.zeros(dtype, (8,)).ptr
    descs = (dev.gemm_desc(dtype, rows, o, i, p, (o, 1), p, (i, 1), p, (i, 1), accumulate=True),
             dev.gemm_desc(dtype, i, rows, o, p, (1, i), p, (o, 1), p, (1, i), accumulate=True))
    return (ITEMSIZE[dtype] > 2 or i % 8 or o % 8) and all("_small_" in dev.gemm_plan(d)[2] for d in descs)


@pytest.mark.parametrize("dtype,rows,i,o", [
    ("f32", 64, 512, 256), ("f32", 48, 2100, 40), ("f64", 20, 232, 978), ("f16", 130, 16, 300), ("bf16", 17, 33, 5), ("f16", 130, 33, 1000),
    ("bf16", 2100, 17, 24),   # 16 waves and one
])
def test_launches(dtype, rows, i, o):
    """Both gradients and the bias gradient: one launch."""
    announce("small pair, launches", dtype, rows, i, o)
    assert joined(device(), dtype, rows, i, o)

    def prepare(dev):
        x, w, go = (dev.zeros(dtype, s) for s in ((rows, i), (o, i), (rows, o)))
        gx, gw, gb = (dev.zeros(dtype, s) for s in ((rows, i), (o, i), (o,)))
        return lambda: dev.linear_backward(x, gx, w, gw, gb, go)
    assert launches(prepare) == 1


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
def test_three_projections(dtype):
    """The forward of a block whose projections are small products: they are one launch, behind it the attention of heads of 40 (its two products
    with the softmax between them, and the reshape), three products (f32: ReLU and two additions apart) and two LayerNorms; the bits
    of the separate calls."""
    B, S, d, H, ff = 2, 33, 120, 3, 200
    announce("small three", dtype)
    block, x, go = test_gpu_encoder_block.a_block(dtype, B, S, d, H, ff)

    def prepare(dev):
        own = type(block)(dev, dtype, d, H, ff, block.p)
        return lambda: own.forward(x)
    assert launches(prepare) == (13 if dtype == "f32" else 10)
    test_gpu_encoder_block.test_block_equals_its_ops(dtype, B, S, d, H, ff)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "f64"])
@pytest.mark.parametrize("rows,i,o", [(64, 512, 256), (17, 33, 5), (1, 40, 24), (130, 16, 300), (20, 232, 978), (48, 2100, 40), (400, 31, 30),
                                      (130, 33, 1000), (2100, 17, 24)])
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
    if joined(dev, dtype, rows, i, o):
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
