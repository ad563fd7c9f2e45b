"""16-bit products cut behind their last full round of tiles (plan_tail of gemm_mfma16_dma.hip): what is left goes to the ring tiles,
along the rows or the columns of C, with everything that belongs to an element of C."""
import numpy as np
import pytest
import torch

import oracle
import test_gpu_encoder_block
from gpu_util import announce, device
from dfdx_amd import Rocm
from dfdx_amd.rocm import KERNEL_MFMA
from helpers import rng

pytestmark = pytest.mark.gpu
K = 1152   # long enough for a round of tiles that a second launch undercuts


def tiles(dev, dtype, name):
    """Ids of the tiles whose names have `name` in them."""
    p = dev.zeros(dtype, (8,)).ptr
    plan = lambda v: dev.gemm_plan(dev.gemm_desc(dtype, 256, 256, 256, p, (256, 1), p, (256, 1), p, (256, 1), kernel=KERNEL_MFMA, variant=v))[2]
    return [v for v in range(1, dev.mfma_variant_count(dtype)) if name in plan(v)]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("m,n,layout,pad,copied", [
    (65792, 256, "nn", 0, False),    # only rows can be cut: 257 tiles one above the other
    (66000, 248, "nt", 8, False),    # 258, the last ones partial in either direction
    (66001, 256, "nn", 0, False),
    (256, 65792, "tn", 0, False),    # only columns can
    (200, 66304, "nn", 8, False),
    (256, 66001, "nt", 0, True),     # the last column off the grid
    (4352, 4100, "tn", 0, True),     # 17 rows of 17 tiles, a copy of one operand
    (4400, 4097, "nt", 3, True),     # of both
    (4225, 4000, "tn", 0, True),
])
def test_cut_products_have_the_bits_of_whole_ones(dtype, m, n, layout, pad, copied):
    """257 - 306 tiles (more than there are compute units).  Against a tile that the call asks for, which is not cut and sums in the same
    order; where no such tile takes the operands, against the sums, which are exact in f32 (multiples of 1/64)."""
    dev, g = device(), rng(m + n)
    at, bt = layout[0] == "t", layout[1] == "t"
    la, lb = (m if at else K) + pad, (K if bt else n) + pad
    ldc = n + pad
    a = oracle.to_storage(g.integers(-8, 9, size=(K, la) if at else (m, la)).astype(np.float32) / 8, dtype)
    b = oracle.to_storage(g.integers(-8, 9, size=(n, lb) if bt else (K, lb)).astype(np.float32) / 8, dtype)
    c = oracle.to_storage(g.standard_normal((m, ldc), dtype=np.float32), dtype)
    bias = oracle.to_storage(g.standard_normal(n), dtype)
    da, db, dbias = dev.tensor(a, dtype), dev.tensor(b, dtype), dev.tensor(bias, dtype)
    tile = tiles(dev, dtype, "dma_128x128")[0]
    for accumulate in (False, True):
        got = []
        for forced in (0,) if copied else (0, tile):
            dc = dev.tensor(c, dtype)
            d = dev.gemm_desc(dtype, m, K, n, da.ptr, (1, la) if at else (la, 1), db.ptr, (1, lb) if bt else (lb, 1), dc.ptr, (ldc, 1),
                              accumulate=accumulate, bias=dbias.ptr, kernel=KERNEL_MFMA if forced else 0, variant=forced, no_split_k=True)
            name = dev.gemm_plan(d)[2]
            announce("gemm tail", dtype, m, n, layout, pad, accumulate, name)
            assert ("+ring" in name) == (not forced) and ("_realigned" in name) == (copied and not forced), name
            dev.gemm(d)
            got.append(oracle.to_f64(dev.to_host(dc), dtype).reshape(m, ldc))
        np.testing.assert_array_equal(got[0][:, n:], oracle.to_f64(c, dtype).reshape(m, ldc)[:, n:])
        if not copied:
            np.testing.assert_array_equal(*got)
            continue
        A, B = oracle.to_f64(a, dtype).reshape(a.shape), oracle.to_f64(b, dtype).reshape(b.shape)
        A, B = (A[:, :m].T if at else A[:, :K]), (B[:, :K].T if bt else B[:, :n])
        rows = np.r_[0:64, m - 600:m] if m > 600 else np.arange(m)
        want = A[rows] @ B + oracle.to_f64(bias, dtype) + (oracle.to_f64(c, dtype).reshape(m, ldc)[rows, :n] if accumulate else 0.0)
        ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]   # one rounding to the type, two additions in f32 before it
        np.testing.assert_allclose(got[0][rows, :n], want, rtol=1.01 * ulp, atol=ulp * 2.0 ** -10 + 2.0 ** -20)


@pytest.mark.parametrize("kernel,launches", [(0, 2), (KERNEL_MFMA, 1)])
def test_a_tile_that_is_asked_for_is_not_cut(kernel, launches):
    """The plan that names two kernels is two launches; the same tile by its id is one."""
    m, n = 4352, 4096
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        own = Rocm(0)
        a, b, c = own.zeros("f16", (m, K)), own.zeros("f16", (K, n)), own.zeros("f16", (m, n))
        variant = tiles(own, "f16", "dma_256x256")[0] if kernel else 0
        d = own.gemm_desc("f16", m, K, n, a.ptr, (K, 1), b.ptr, (n, 1), c.ptr, (n, 1), kernel=kernel, variant=variant, no_split_k=True)
        name = own.gemm_plan(d)[2]
        announce("gemm tail, launches", kernel, name)
        assert "dma_256x256" in name and ("+ring" in name) == (launches == 2)
        run = lambda: own.gemm(d)
        run()
        own.synchronize()
        assert test_gpu_encoder_block.graph_nodes(run, stream) == launches
        own.synchronize()
    own.close()


def test_what_rides_along_with_a_cut_product():
    """ReLU, its gradient, a residual: the block's products on 17 x 16 tiles against the single ops."""
    dev, p = device(), device().zeros("f16", (8,)).ptr
    rows, d, ff = 17 * 256, 1024, 4096
    for b in ((1, d), (ff, 1)):   # the first feed-forward product; the input gradient of the second one
        assert "+ring" in dev.gemm_plan(dev.gemm_desc("f16", rows, d, ff, p, (d, 1), p, b, p, (ff, 1)))[2]
    test_gpu_encoder_block.test_block_equals_its_ops("f16", 17, 256, d, 16, ff)
