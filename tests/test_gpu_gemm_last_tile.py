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
@pytest.mark.parametrize("m,k,n,a_across,pad,plan", [
    (4096, 1001, 4096, True, 0, "dma_256x256x64_w2x4_realigned"),            # both operands: their last tiles
    (4096, 2047, 4096, True, 24, "dma_256x256x64_w2x4_realigned"),           # 63 of 64 rows, rows wider than the matrix
    (3080, 1025, 3072, True, 8, "dma_256x256x64_w2x4_realigned"),            # one row, partial tiles of C
    (4352, 1100, 4096, True, 0, "_realigned+ring"),                          # more than whole rounds of tiles: the rest on other tiles
    (2051, 3073, 2048, False, 16, "dma_256x128x64_w4x2_realigned"),          # A whole (off the grid), B's last tile
    (2048, 20011, 2048, False, 0, "dma_256x256x64_w2x4_realigned_splitk"),   # split contraction, its last piece shorter
    (2048, 20011, 2048, True, 0, "dma_256x256x64_w2x4_realigned_splitk"),
    (8192, 50, 4096, True, 0, "dma_256x256x64_w2x4_realigned"),              # nothing but the last tile
    (1024, 1025, 520, False, 0, "ring_64x64x64_w2x2_s4_dma_realigned"),      # the ring goes there too; 8-column remainders of a tile
    (512, 20011, 1024, False, 0, "ring_128x128x64_w2x4_s4_dma_realigned_splitk"),
    (2048, 1001, 2048, True, 0, "ring"),                                     # in place: the ring takes any k
    (2048, 2047, 2048, True, 24, "ring"),
    (2304, 1025, 2048, True, 8, ""),
    (512, 20011, 1024, True, 0, "ring"),
    (4096, 50, 4096, True, 0, ""),
    (1024, 4113, 520, True, 0, "ring"),
])
@pytest.mark.parametrize("accumulate", [False, True])
def test_only_the_last_tile_is_copied(dtype, m, k, n, a_across, pad, plan, accumulate):
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
    if not (k == 50 and accumulate):   # (so short a product that adds to C is not worth its copies)
        assert plan in name and ("_realigned" in name) == ("_realigned" in plan), name
    dev.gemm(desc)
    got = oracle.to_f64(dev.to_host(dc), dtype).reshape(m, n)
    A = oracle.to_f64(a, dtype).reshape(-1, lda)[:k, :m].T if a_across else oracle.to_f64(a, dtype).reshape(-1, lda)[:m, :k]
    B = oracle.to_f64(b, dtype).reshape(-1, ldb)[:k, :n]
    old = oracle.to_f64(c, dtype).reshape(m, n) if accumulate else 0.0
    want = np.asarray((torch.from_numpy(np.ascontiguousarray(A)).cuda() @ torch.from_numpy(np.ascontiguousarray(B)).cuda()).cpu()) + old
    ulp = 2.0 ** (-11 if dtype == "f16" else -8)
    assert_within(dtype, k, got, want, A, B, extra=ulp * float(np.abs(want).max()))
