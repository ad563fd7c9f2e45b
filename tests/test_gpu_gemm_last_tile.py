"""Products of the 16-bit types whose contraction ends inside a k tile, with an operand on the 16-byte grid whose rows lie along
memory: its last k tile is copied next to zeros, the rest is read where it lies.  What lies behind the operand is NaN."""
import numpy as np
import pytest
import torch

import oracle
from helpers import assert_within, rng
from gpu_util import announce, device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("m,k,n,a_across,pad", [
    (2048, 1001, 2048, True, 0),     # both operands: their last tiles
    (2048, 2047, 2048, True, 24),    # 63 of 64 rows, rows wider than the matrix
    (2304, 1025, 2048, True, 8),     # one row
    (4352, 1100, 4096, True, 0),     # more than whole rounds of tiles: the rest on other tiles
    (2051, 3073, 2048, False, 16),   # A whole (off the grid), B's last tile
    (512, 20011, 1024, False, 0),    # split contraction, its last piece shorter
    (512, 20011, 1024, True, 0),
    (4096, 50, 4096, True, 0),       # nothing but the last tile
    (1024, 4113, 520, True, 0),      # 8-column remainders of a tile
])
@pytest.mark.parametrize("accumulate", [False, True])
def test_only_the_last_tile_is_copied(dtype, m, k, n, a_across, pad, accumulate):
    dev, g = device(), rng(m + k + n)

    def operand(rows, cols, ld):  # `rows` rows of `cols` values, NaN between and behind them
        t = np.full((rows + 70, ld), np.nan)
        t[:rows, :cols] = g.standard_normal((rows, cols))
        return oracle.to_storage(t.ravel(), dtype), ld

    a, lda = operand(k, m, m + pad) if a_across else operand(m, k, k)
    b, ldb = operand(k, n, n + pad)
    c = oracle.to_storage(g.standard_normal(m * n), dtype)
    da, db, dc = (dev.tensor(t, dtype) for t in (a, b, c))
    desc = dev.gemm_desc(dtype, m, k, n, da.ptr, (1, lda) if a_across else (lda, 1), db.ptr, (ldb, 1), dc.ptr, (n, 1), accumulate=accumulate)
    name = dev.gemm_plan(desc)[2]
    announce("last tile", dtype, m, k, n, a_across, pad, accumulate, name)
    dev.gemm(desc)
    got = oracle.to_f64(dev.to_host(dc), dtype).reshape(m, n)
    A = oracle.to_f64(a, dtype).reshape(-1, lda)[:k, :m].T if a_across else oracle.to_f64(a, dtype).reshape(-1, lda)[:m, :k]
    B = oracle.to_f64(b, dtype).reshape(-1, ldb)[:k, :n]
    old = oracle.to_f64(c, dtype).reshape(m, n) if accumulate else 0.0
    want = np.asarray((torch.from_numpy(np.ascontiguousarray(A)).cuda() @ torch.from_numpy(np.ascontiguousarray(B)).cuda()).cpu()) + old
    ulp = 2.0 ** (-11 if dtype == "f16" else -8)
    assert_within(dtype, k, got, want, A, B, extra=ulp * float(np.abs(want).max()))
