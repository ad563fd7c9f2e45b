"""16-bit products cut behind their last full round of tiles (plan_tail of gemm_mfma16_dma.hip): what is left goes to the ring tiles,
along the rows or the columns of C, with everything that belongs to an element of C."""
import numpy as np
import pytest

import oracle
from gpu_util import announce, device
from dfdx_amd.rocm import KERNEL_MFMA
from helpers import rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("m,n", [(65792, 256), (66000, 248), (66001, 256), (256, 65792), (200, 66304), (256, 66001)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_cut_products_have_the_bits_of_whole_ones(dtype, m, n, layout):
    """257 - 259 tiles of 256 x 256 (more than there are compute units), the last ones partial, the last columns off the grid; bias
    and old values.  The 128 x 128 tiles, which are never cut, sum in the same order."""
    dev, g, k = device(), rng(m + n), 512
    announce("gemm tail", dtype, m, n, layout)
    at, bt = layout[0] == "t", layout[1] == "t"
    up = lambda v: (v + 7) // 8 * 8      # (operands stay on the 16-byte grid; C need not)
    la, lb = (up(m), up(n)) if not bt else (up(m), k)
    a = oracle.to_storage(g.integers(-8, 9, size=(k, la) if at else (m, k)).astype(np.float64) / 8, dtype)
    b = oracle.to_storage(g.integers(-8, 9, size=(n, k) if bt else (k, lb)).astype(np.float64) / 8, dtype)
    c = oracle.to_storage(g.standard_normal((m, n)), dtype)
    bias = oracle.to_storage(g.standard_normal(n), dtype)
    da, db, dbias = dev.tensor(a, dtype), dev.tensor(b, dtype), dev.tensor(bias, dtype)
    tile = next(v for v in range(1, dev.mfma_variant_count(dtype)) if "dma_128x128" in dev.gemm_plan(
        dev.gemm_desc(dtype, 256, 256, 256, da.ptr, (256, 1), db.ptr, (256, 1), da.ptr, (256, 1), kernel=KERNEL_MFMA, variant=v))[2])
    forcible = n % 8 == 0 and not (at and m % 8)
    for accumulate in (False, True):
        got = []
        for forced in (0, tile):
            dc = dev.tensor(c, dtype)
            d = dev.gemm_desc(dtype, m, k, n, da.ptr, (1, la) if at else (k, 1), db.ptr, (1, k) if bt else (lb, 1), dc.ptr, (n, 1),
                              accumulate=accumulate, bias=dbias.ptr, kernel=KERNEL_MFMA if forced and forcible else 0,
                              variant=forced if forcible else 0, no_split_k=True)
            dev.gemm(d)
            got.append(oracle.to_f64(dev.to_host(dc), dtype))
        np.testing.assert_array_equal(*got)
        if not forcible:  # the plan is the same on both sides: against the sums, which are exact in f32 (multiples of 1/64)
            A, B = oracle.to_f64(a, dtype).reshape(a.shape), oracle.to_f64(b, dtype).reshape(b.shape)
            A, B = (A.T[:m] if at else A), (B.T if bt else B[:, :n])
            rows = np.r_[0:64, m - 600:m] if m > 600 else np.arange(m)
            want = A[rows] @ B + oracle.to_f64(bias, dtype) + (oracle.to_f64(c, dtype).reshape(m, n)[rows] if accumulate else 0.0)
            ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]   # one rounding to the type, two additions in f32 before it
            np.testing.assert_allclose(got[0].reshape(m, n)[rows], want, rtol=1.01 * ulp, atol=ulp * 2.0 ** -10 + 2.0 ** -20)
