"""The f32 tiles behind a ring of LDS stages (gemm_mfma32_ring.hip): edges of tiles, partial last k tiles, contractions shorter
and longer than the ring, operands on and off the 16-byte grid, batches, and what a captured stream gets."""
import numpy as np
import pytest

import oracle
from dfdx_amd.rocm import KERNEL_AUTO, KERNEL_MFMA
from gpu_util import announce, device
from helpers import assert_within, rng
from test_gpu_gemm import run_case

pytestmark = pytest.mark.gpu
STAGED, RING = 6, (9, 10)   # the register-staged 64 x 64 tile, and the 64 x 64 and 128 x 64 ones in front of the small-product kernel


@pytest.mark.parametrize("variant", RING)
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("m,n", [(64, 64), (128, 128), (65, 67), (200, 263), (1, 130), (7, 3)])
@pytest.mark.parametrize("k", [1, 31, 32, 33, 96, 128, 190, 292])
def test_tiles_and_tails(variant, layout, m, n, k):
    """1 to 10 k tiles (3 are in flight), the last one whole or partial; every pairing of operands on and off the grid."""
    pads = ((0, 0, 0), (4, 1, 3), (1, 4, 0))[(m + n + k) % 3]
    assert "_ring_" in run_case("f32", m, k, n, layout, k % 2 == 0, KERNEL_MFMA, variant, bias=m % 2 == 0, c_colmajor=n > 1 and k % 3 == 0, seed=m + k, pads=pads)


@pytest.mark.parametrize("variant", RING)
@pytest.mark.parametrize("layout", ["nt", "tn"])
@pytest.mark.parametrize("splits,k", [(2, 65), (4, 300), (5, 449)])
def test_pieces_of_the_contraction(variant, layout, splits, k):
    name = run_case("f32", 130, k, 75, layout, True, KERNEL_MFMA, variant, split_k=splits, bias=True, seed=k)
    assert name.endswith(f"_splitk{splits}")


@pytest.mark.parametrize("reduce", [False, True])
@pytest.mark.parametrize("k,n", [(32, 80), (40, 77), (129, 80)])
def test_batches_have_the_bits_of_the_staged_tile(reduce, k, n):
    """Batches side by side and summed over (the k loop restarts in every batch, behind a partial tile): the order of the sum, and
    so every bit, is that of the register-staged tile."""
    dev, g = device(), rng(71 + k)
    b1, b2, m = 2, 3, 72
    a, b = (oracle.to_storage(g.standard_normal(b1 * b2 * k * s), "f32") for s in (m, n))
    da, db = dev.tensor(a, "f32"), dev.tensor(b, "f32")
    A, B = (oracle.to_f64(t, "f32").reshape(b1 * b2, k, -1) for t in (a, b))
    want = A.transpose(0, 2, 1) @ B
    if reduce:
        want = want.sum(axis=0, keepdims=True)
    got = {}
    for variant in (STAGED, *RING):
        announce("f32 ring batches", reduce, k, n, variant)
        c = dev.zeros("f32", want.shape)
        dev.gemm(dev.gemm_desc("f32", m, k, n, da.ptr, (1, m), db.ptr, (n, 1), c.ptr, (n, 1), batch=(b1, b2), a_batch=(b2 * k * m, k * m),
                               b_batch=(b2 * k * n, k * n), c_batch=(0, 0) if reduce else (b2 * m * n, m * n), reduce_batch=reduce,
                               kernel=KERNEL_MFMA, variant=variant, no_split_k=True))
        got[variant] = dev.to_host(c)
    assert_within("f32", k * (b1 * b2 if reduce else 1), got[STAGED].reshape(want.shape), want, A, B, what="staged")
    for variant in RING:
        np.testing.assert_array_equal(got[variant], got[STAGED])


def test_infinities_stay_in_their_rows():
    """What lies beyond k is zero on both sides, and rows beyond the last repeat it: nothing meets an infinity that should not."""
    dev, m, k, n = device(), 67, 35, 66
    for layout in ("nt", "tn"):
        A, B = np.ones((m, k), np.float32), np.ones((k, n), np.float32)
        A[m - 1, k - 1] = np.inf
        a = np.ascontiguousarray(A if layout == "nt" else A.T)
        b = np.ascontiguousarray(B.T if layout == "nt" else B)
        da, db, c = dev.tensor(a, "f32"), dev.tensor(b, "f32"), dev.zeros("f32", (m, n))
        for variant in RING:
            announce("f32 ring infinities", layout, variant)
            dev.gemm(dev.gemm_desc("f32", m, k, n, da.ptr, (k, 1) if layout == "nt" else (1, m), db.ptr, (1, k) if layout == "nt" else (n, 1), c.ptr, (n, 1),
                                   kernel=KERNEL_MFMA, variant=variant))
            np.testing.assert_array_equal(dev.to_host(c).reshape(m, n), A @ B)


@pytest.mark.parametrize("m,k,n,layout,want", [
    (4096, 4096, 4096, "nt", "dma_256x256"), (136, 478, 6449, "nt", "_ring_64x64"), (1024, 1024, 1024, "nn", "_ring_64x64"),
    (164, 2955, 408, "nt", "_ring_64x64"), (64, 512, 256, "nt", "_small_"),
])
def test_plans(m, k, n, layout, want):
    a, b = ((k, 1), (1, k)) if layout == "nt" else ((k, 1), (n, 1))
    dev = device()
    assert want in dev.gemm_plan(dev.gemm_desc("f32", m, k, n, 256, a, 512, b, 1024, (n, 1), kernel=KERNEL_AUTO))[2]


@pytest.mark.parametrize("ld,tile", [(16777148, "_ring_64x64"), (16777152, "_64x64x32_w2x2")])
def test_rows_too_far_apart_for_the_ring(ld, tile):
    """64 rows of a k-contiguous operand (as many as a tile has, whatever m is) have to lie within 32 bits of bytes: beyond, the register-staged
    tile is planned."""
    import torch
    dev, (m, k, n) = device(), (5, 100, 72)
    gen = torch.Generator(device="cuda").manual_seed(ld)
    a = torch.zeros((m - 1) * ld + k, device="cuda")
    rows = a.as_strided((m, k), (ld, 1))
    rows.copy_(torch.randn(m, k, device="cuda", generator=gen))
    b, c = torch.randn(k, n, device="cuda", generator=gen), torch.zeros(m, n, device="cuda")
    desc = dev.gemm_desc("f32", m, k, n, a.data_ptr(), (ld, 1), b.data_ptr(), (n, 1), c.data_ptr(), (n, 1), kernel=KERNEL_MFMA, no_split_k=True)
    name = dev.gemm_plan(desc)[2]
    announce("f32, rows far apart", ld, name)
    assert tile in name and ("_ring_" in tile) == ("_ring_" in name), name
    dev.gemm(desc)
    dev.synchronize()
    A, B = rows.double().cpu().numpy(), b.double().cpu().numpy()
    assert_within("f32", k, c.double().cpu().numpy(), A @ B, A, B, what=name)


def test_captured_with_no_space_for_partial_sums():
    """A cold context: a product that is planned in pieces runs in one, and replays."""
    import torch
    from dfdx_amd import Rocm

    m, k, n, g = 704, 874, 512, rng(5)
    a, b = (oracle.to_storage(g.standard_normal(s), "f32") for s in ((m, k), (n, k)))
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        own = Rocm(0)
        da, db, c = own.tensor(a, "f32"), own.tensor(b, "f32"), own.zeros("f32", (m, n))
        desc = own.gemm_desc("f32", m, k, n, da.ptr, (k, 1), db.ptr, (1, k), c.ptr, (n, 1))
        assert "_ring_" in own.gemm_plan(desc)[2] and "splitk" in own.gemm_plan(desc)[2]
        announce("f32 ring captured")
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            own.gemm(desc)
        for _ in range(3):
            c.storage.fill_(255)
            graph.replay()
            stream.synchronize()
            A, B = oracle.to_f64(a, "f32").reshape(m, k), oracle.to_f64(b, "f32").reshape(n, k).T
            assert_within("f32", k, own.to_host(c).reshape(m, n), A @ B, A, B, what="replayed")
        del graph
        own.close()
