"""The 16-bit tiles behind a ring of LDS stages (gemm_mfma16_ring.hip): edges of tiles, partial last k tiles, contractions
shorter and longer than the ring, batches, and the row sums that ride along."""
import numpy as np
import pytest

import oracle
from dfdx_amd.rocm import KERNEL_AUTO, KERNEL_MFMA
from gpu_util import announce, device, launches
from helpers import assert_within, rng
from test_gpu_gemm import run_case

pytestmark = pytest.mark.gpu
TILES = 5


def ring_ids():
    dev = device()
    plan = lambda v: dev.gemm_plan(dev.gemm_desc("f16", 256, 256, 256, 256, (256, 1), 512, (256, 1), 1024, (256, 1), kernel=KERNEL_MFMA, variant=v))[2]
    ids = [v for v in range(1, dev.mfma_variant_count("f16")) if "_ring_" in plan(v)]
    assert len(ids) == TILES
    return ids


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("tile", range(TILES))
@pytest.mark.parametrize("m,n", [(64, 64), (128, 128), (65, 67), (200, 264), (1, 136), (8, 9)])
@pytest.mark.parametrize("k", [8, 64, 72, 184, 256, 320, 456])
def test_operands_along_k(dtype, tile, m, n, k):
    """1 to 8 k tiles (3 or 4 are in flight), the last one whole or partial; columns of C off the grid of eight."""
    assert "_ring_" in run_case(dtype, m, k, n, "nt", m > 64, KERNEL_MFMA, ring_ids()[tile], bias=n % 8 == 0, seed=m + k)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("tile", range(TILES))
@pytest.mark.parametrize("layout,k", [("tn", 1), ("tn", 63), ("tn", 65), ("tn", 259), ("tn", 449), ("nn", 24), ("nn", 328), ("tt", 136)])
@pytest.mark.parametrize("splits", [1, 2])
def test_operands_across_k(dtype, tile, layout, k, splits):
    """The transposing reads: any length of the contraction where both operands lie across it, whole pieces of eight else."""
    run_case(dtype, 136, k, 72, layout, True, KERNEL_MFMA, ring_ids()[tile], split_k=splits, pads=(8, 8, 8), seed=k)
    run_case(dtype, 72, k, 200, layout, False, KERNEL_MFMA, ring_ids()[tile], split_k=splits, bias=True, c_colmajor=False, seed=k + 1)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("reduce", [False, True])
@pytest.mark.parametrize("k", [40, 64, 137])
def test_batches(dtype, reduce, k):
    """Batches side by side and summed over (the k loop then restarts in every batch, behind a partial tile)."""
    dev, g = device(), rng(71 + k)
    b1, b2, m, n = 2, 3, 72, 80
    a = oracle.to_storage(g.standard_normal(b1 * b2 * k * m), dtype)
    b = oracle.to_storage(g.standard_normal(b1 * b2 * k * n), dtype)
    A = oracle.to_f64(a, dtype).reshape(b1 * b2, k, m).transpose(0, 2, 1)
    B = oracle.to_f64(b, dtype).reshape(b1 * b2, k, n)
    want = A @ B
    if reduce:
        want = want.sum(axis=0, keepdims=True)
    da, db = dev.tensor(a, dtype), dev.tensor(b, dtype)
    for variant in ring_ids():
        announce("ring batches", dtype, reduce, k, variant)
        c = dev.zeros(dtype, (want.shape[0], m, n))
        d = dev.gemm_desc(dtype, m, k, n, da.ptr, (1, m), db.ptr, (n, 1), c.ptr, (n, 1), batch=(b1, b2), a_batch=(b2 * k * m, k * m),
                          b_batch=(b2 * k * n, k * n), c_batch=(0, 0) if reduce else (b2 * m * n, m * n), reduce_batch=reduce,
                          kernel=KERNEL_MFMA, variant=variant)
        dev.gemm(d)
        got = oracle.to_f64(dev.to_host(c), dtype).reshape(want.shape)
        ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
        assert_within(dtype, k * (b1 * b2 if reduce else 1), got, want, A, B, extra=ulp * float(np.abs(want).max()), what="ring batches")


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rows,i,o", [(100, 256, 256), (263, 136, 520), (529, 768, 384), (1344, 768, 768), (2001, 64, 72)])
def test_bias_gradient_rides_along(dtype, rows, i, o):
    """Linear's backward on rows that are no multiple of 64: the sums of small whole numbers are exact in f32, so the bias gradient
    has the one rounding of its result; both gradients against float64."""
    dev, g = device(), rng(rows)
    announce("ring row sums", dtype, rows, i, o)
    x, w = (oracle.to_storage(g.standard_normal(s), dtype) for s in ((rows, i), (o, i)))
    go = oracle.to_storage(g.integers(-4, 5, size=(rows, o)).astype(np.float64), dtype)
    dx, dw, dgo = dev.tensor(x, dtype), dev.tensor(w, dtype), dev.tensor(go, dtype)
    gx, gw, gb = dev.zeros_like_storage(dx), dev.zeros_like_storage(dw), dev.zeros(dtype, (o,))
    dev.linear_backward(dx, gx, dw, gw, gb, dgo)
    X, W, G = oracle.to_f64(x, dtype), oracle.to_f64(w, dtype), oracle.to_f64(go, dtype)
    host = lambda t, shape: oracle.to_f64(dev.to_host(t), dtype).reshape(shape)
    want = oracle.to_f64(oracle.to_storage(G.sum(axis=0), dtype), dtype)
    np.testing.assert_array_equal(host(gb, (o,)), want)
    ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
    assert_within(dtype, rows, host(gw, (o, i)), G.T @ X, G, X, extra=ulp * float(np.abs(G.T @ X).max()), what="weight")
    assert_within(dtype, o, host(gx, (rows, i)), G @ W, G, W, extra=ulp * float(np.abs(G @ W).max()), what="input")


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rows,i,o", [(400, 256, 1024), (96, 128, 128), (529, 768, 768), (1344, 768, 1536), (1344, 768, 3072)])
def test_two_products_of_a_backward_pass(dtype, rows, i, o):
    """Launches of both gradients together, of few work items and of more than the chip has places for, into fresh and into
    accumulated gradients."""
    dev, g = device(), rng(rows + o)
    announce("ring pair", dtype, rows, i, o)
    x, w, go = (oracle.to_storage(g.standard_normal(s), dtype) for s in ((rows, i), (i, o), (rows, o)))
    dx, dw, dgo = dev.tensor(x, dtype), dev.tensor(w, dtype), dev.tensor(go, dtype)
    X, W, G = oracle.to_f64(x, dtype), oracle.to_f64(w, dtype), oracle.to_f64(go, dtype)
    ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
    gx, gw = dev.zeros_many([dx, dw], deferred=True)
    for times in (1, 2):
        dev.backward(dx, gx, dw, gw, dgo)
        for got, a, b, what in ((gx, G, W.T, "lhs"), (gw, X.T, G, "rhs")):
            want = times * (a @ b)
            assert_within(dtype, a.shape[1], oracle.to_f64(dev.to_host(got), dtype).reshape(want.shape), want, a, b,
                          extra=2 * times * ulp * float(np.abs(want).max()), what=what)

    def prepare(own):
        x, w, go, gx, gw = (own.zeros(dtype, s) for s in ((rows, i), (i, o), (rows, o), (rows, i), (i, o)))
        return lambda: own.backward(x, gx, w, gw, go)
    assert launches(prepare) == 1


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("batch,m,k,n,expected", [
    (39, 448, 80, 448, 1), (43, 256, 256, 256, 1), (25, 200, 136, 264, 1),   # more work items than the chip has places for
    (54, 512, 80, 512, 2), (77, 320, 128, 320, 2),                           # no tile whose second round is worth it
])
def test_batches_of_a_backward_pass(dtype, batch, m, k, n, expected):
    """The right operand stored along k, as attention's keys are."""
    dev, g = device(), rng(batch + m)
    announce("ring pair, batches", dtype, batch, m, k, n)
    x, wt, go = (oracle.to_storage(g.standard_normal(s), dtype) for s in ((batch, m, k), (batch, n, k), (batch, m, n)))
    shapes = ((batch, m, k), (batch, n, k), (batch, m, n), (batch, m, k), (batch, n, k))
    turned = lambda t: t.permute(0, 2, 1)
    dx, dw, dgo = dev.tensor(x, dtype), dev.tensor(wt, dtype), dev.tensor(go, dtype)
    gx, gw = dev.zeros_many([dx, dw], deferred=True)
    dev.backward(dx, gx, turned(dw), turned(gw), dgo)
    X, W, G = oracle.to_f64(x, dtype), oracle.to_f64(wt, dtype), oracle.to_f64(go, dtype)
    ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
    for got, a, b, what in ((gx, G, W, "lhs"), (gw, G.transpose(0, 2, 1), X, "rhs")):
        want = a @ b
        assert_within(dtype, a.shape[2], oracle.to_f64(dev.to_host(got), dtype)[:want.size].reshape(want.shape), want, a, b,
                      extra=ulp * float(np.abs(want).max()), what=what)

    def prepare(own):
        x, w, go, gx, gw = (own.zeros(dtype, s) for s in shapes)
        return lambda: own.backward(x, gx, turned(w), turned(gw), go)
    assert launches(prepare) == expected


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("n", [128, 384])
def test_a_gradient_that_both_products_add_to(dtype, n):
    """x . x: both gradients go to one buffer, one behind the other."""
    dev, g = device(), rng(n)
    announce("ring pair, one gradient", dtype, n)
    x, go = (oracle.to_storage(g.standard_normal((n, n)), dtype) for _ in range(2))
    dx, dgo = dev.tensor(x, dtype), dev.tensor(go, dtype)
    X, G = oracle.to_f64(x, dtype), oracle.to_f64(go, dtype)
    gx = dev.zeros_like_storage(dx)
    dev.backward(dx, gx, dx, gx, dgo)
    want = G @ X.T + X.T @ G
    ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]

    def prepare(own, shared):
        x, go, gx, gy = (own.zeros(dtype, (n, n)) for _ in range(4))
        return lambda: own.backward(x, gx, x, gx if shared else gy, go)
    assert [launches(lambda own: prepare(own, shared)) for shared in (True, False)] == [2, 1]
    assert_within(dtype, 2 * n, oracle.to_f64(dev.to_host(gx), dtype).reshape(n, n), want, X, G, extra=2 * ulp * float(np.abs(want).max()), what="sum")


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("m,k,n,want", [
    (2048, 64, 367, "mfma16_64x64x64_w2x2"), (520, 128, 1001, "mfma16_64x64x64_w2x2"), (8, 16384, 257, "gemv_rows"),
    (1000, 8192, 63, "mfma16_ring_64x64x64_w2x2_s4_splitk10"), (300, 2048, 1025, "ring"),
])
def test_results_off_the_grid_have_rivals(dtype, m, k, n, want):
    """Whole k tiles and a C that only the ring takes of the LDS-DMA kernels: the other families are weighed too."""
    dev = device()
    name = dev.gemm_plan(dev.gemm_desc(dtype, m, k, n, 256, (k, 1), 512, (1, k), 1024, (n, 1)))[2]
    assert want == name or (want == "ring" and "_ring_" in name and "_realigned" not in name), name


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("m,k,n,layout,accumulate,want", [
    (7040, 64, 512, "nn", False, "_dma_128x128"), (512, 256, 5248, "tn", False, "_dma_128x128"),   # many stores behind a few k tiles
    (7040, 64, 512, "nn", True, "_ring_"), (1152, 64, 640, "nn", False, "_ring_"), (7040, 512, 512, "nn", False, "_ring_"),
    (512, 208, 200, "tn", False, "_small_"), (104, 64, 384, "tn", False, "_small_"), (256, 96, 1971, "nt", False, "_small_"),   # short contractions
    (512, 288, 200, "tn", False, "_ring_"), (512, 208, 200, "tn", True, "_ring_"),
])
def test_where_the_ring_has_rivals(dtype, m, k, n, layout, accumulate, want):
    assert want in run_case(dtype, m, k, n, layout, accumulate, KERNEL_AUTO, 0, seed=m + n)
