"""One to sixteen vectors against a matrix stored along k, rows anywhere (the rows form of gemv_multi.hip): steps that are whole,
partial or missing, rows off the 16-byte grid, outputs past the last sixteen, k slices."""
import numpy as np
import pytest

import oracle
from dfdx_amd.rocm import KERNEL_AUTO, KERNEL_GEMV
from gpu_util import announce, device
from helpers import assert_within, rng
from test_gpu_gemm import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,k,n", [(2, 1061, 2050), (1, 1063, 1601), (8, 2531, 4099), (16, 1999, 1040), (5, 5001, 517), (13, 12289, 600)])
@pytest.mark.parametrize("pads", [(0, 0, 0), (3, 5, 1)])
def test_rows_off_the_grid(dtype, rows, k, n, pads):
    """Either operand as the matrix; bias, both beta, column-major C; the longest ones in k slices."""
    assert run_case(dtype, rows, k, n, "nt", False, KERNEL_AUTO, 0, bias=True, pads=pads, seed=k) == "gemv_rows"
    assert run_case(dtype, n, k, rows, "nt", True, KERNEL_AUTO, 0, pads=pads, seed=k + 1) == "gemv_rows"
    run_case(dtype, rows, k, n, "nt", True, KERNEL_AUTO, 0, c_colmajor=True, pads=pads, seed=k + 2)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,k,n", [(12, 6077, 218), (16, 5493, 453), (13, 14271, 151), (2, 7680, 250), (9, 15104, 130), (3, 3071, 128), (3, 3073, 129),
                                      (7, 2559, 257), (7, 2561, 1087), (16, 8190, 1024)])
@pytest.mark.parametrize("pads", [(0, 0, 0), (3, 5, 1)])
def test_few_outputs_of_long_rows(dtype, rows, k, n, pads):
    """Up to sixteen k slices of four waves and more, rows on the 16-byte grid instead of the lines; at the lengths where either begins."""
    for m_, n_, acc in ((rows, n, False), (n, rows, True)):
        assert run_case(dtype, m_, k, n_, "nt", acc, KERNEL_GEMV, 5, pads=pads, seed=k + acc) == "gemv_rows"


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("k", [1024, 1024 + 1, 1024 + 31, 1024 + 32, 1024 + 63, 4096 - 7])
@pytest.mark.parametrize("n", [2056, 200])
def test_what_lies_behind_the_contraction_counts_for_nothing(dtype, k, n):
    """Rows with a gap of NaN behind each: the partial step takes zeros in their place."""
    dev, g = device(), rng(k)
    rows, gap = 4, 9
    announce("gemv rows gaps", dtype, k)
    x, w = (oracle.to_storage(np.concatenate([g.standard_normal((r, k)), np.full((r, gap), np.nan)], axis=1), dtype) for r in (rows, n))
    dx, dw, dc = dev.tensor(x, dtype), dev.tensor(w, dtype), dev.zeros(dtype, (rows, n))
    dev.gemm(dev.gemm_desc(dtype, rows, k, n, dx.ptr, (k + gap, 1), dw.ptr, (1, k + gap), dc.ptr, (n, 1)))
    X, W = (oracle.to_f64(t, dtype).reshape(-1, k + gap)[:, :k] for t in (x, w))
    want = X @ W.T
    ulp = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
    assert_within(dtype, k, oracle.to_f64(dev.to_host(dc), dtype).reshape(want.shape), want, X, W, extra=ulp * float(np.abs(want).max()), what="rows")


def chains(a, b, n):
    """a . b^T in f32 as n interleaved chains of fused multiply-adds whose sums meet in pairs."""
    pad = ((0, 0), (0, -a.shape[1] % n))
    a, b = np.pad(a, pad).astype(np.float64), np.pad(b, pad).astype(np.float64)
    part = np.zeros((a.shape[0], b.shape[0], n), np.float32)
    for s in range(0, a.shape[1], n):
        part = (part + a[:, None, s:s + n] * b[None, :, s:s + n]).astype(np.float32)
    while n > 1:
        n //= 2
        part = part[..., :n] + part[..., n:]
    return part[..., 0]


@pytest.mark.parametrize("k", [435, 771, 1219, 3071])
def test_f32_sums_are_short_chains(k):
    """No further from float64 than 32 chains (the norm of 8320 independent errors is known to 1 %, the rest of the 15 % is for waves
    that have a step more than others)."""
    dev, g, rows, n = device(), rng(k), 16, 520
    announce("gemv rows, f32 sums", k)
    x, w = g.standard_normal((rows, k)).astype(np.float32), (g.uniform(-1.0, 1.0, (n, k)) * k ** -0.5).astype(np.float32)
    dx, dw, dc = dev.tensor(x, "f32"), dev.tensor(w, "f32"), dev.zeros("f32", (rows, n))
    desc = dev.gemm_desc("f32", rows, k, n, dx.ptr, (k, 1), dw.ptr, (1, k), dc.ptr, (n, 1))
    assert dev.gemm_plan(desc)[2] == "gemv_rows"
    dev.gemm(desc)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    far = lambda got: np.linalg.norm(got - want)
    assert far(dev.to_host(dc).reshape(rows, n)) <= 1.15 * far(chains(x, w, 32))


@pytest.mark.parametrize("dtype,rows,k,n", [("f16", 16, 4096, 4096), ("f16", 4, 4093, 4091), ("f32", 4, 4093, 1091), ("f16", 8, 4096, 4096)])
def test_the_kernel_that_a_plan_names_can_be_asked_for(dtype, rows, k, n):
    """By the id that the plan reports; without one the vector-ALU form comes first, where there is one."""
    dev = device()
    plan = lambda *how: dev.gemm_plan(dev.gemm_desc(dtype, rows, k, n, 256, (k, 1), 512, (1, k), 1024, (n, 1), kernel=how[0], variant=how[1]))
    assert plan(*plan(KERNEL_AUTO, 0)[:2]) == plan(KERNEL_AUTO, 0)
    kernel, variant, name = plan(KERNEL_GEMV, 5)
    assert (kernel, variant, name) == (KERNEL_GEMV, 5, "gemv_rows")
    assert plan(kernel, 0)[2] == ("gemv_multi" if k % 8 == 0 and rows <= 8 else "gemv_rows")
    if n < 2000:
        assert run_case(dtype, rows, k, n, "nt", True, kernel, variant, seed=k) == "gemv_rows"


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rows,k,n,pad,want", [
    (16, 10304, 4355, 0, "_ring_"), (8, 8960, 7680, 0, "_ring_"), (12, 5376, 4438, 0, "_ring_"),   # rows on the grid of a large matrix
    (16, 10304, 4355, 4, "gemv_rows"), (16, 10301, 4355, 0, "gemv_rows"), (8, 2048, 2744, 0, "gemv_rows"),
    (2, 12920, 12288, 0, "gemv_multi"), (8, 16768, 11008, 0, "gemv_multi"), (16, 16768, 11008, 0, "_ring_"),   # beyond the caches
])
def test_rivals_on_large_matrices(dtype, rows, k, n, pad, want):
    dev = device()
    name = dev.gemm_plan(dev.gemm_desc(dtype, rows, k, n, 256, (k + pad, 1), 512, (1, k + pad), 1024, (n, 1)))[2]
    announce("gemv rows, rivals", dtype, rows, k, n, pad, name)
    assert want in name, name
