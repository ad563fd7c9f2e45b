"""GPU: the entry point that allocates nothing (`dfdx_rocm_gemm_noalloc`) against `dfdx_rocm_gemm`.

Both plan the same products; the difference is where the f32 partial sums of a split reduction, and the padded copies of
16-bit operands off the 16-byte grid, live (the library's fixed per-GPU scratch array instead of a context-owned buffer
that grows on demand), and that copies which do not fit are left out; the two results must be identical bit for bit -- and both within the stated tolerance of the oracle
(max|err| <= 2e-3*sqrt(K)*max|a|*max|b| for f16 / bf16, 1e-5*sqrt(K)*... for f32).  Every case makes two calls in a
row, the second on a smaller product, because all calls on a GPU share the one array and it keeps the last call's
contents.  Runs last (file name) so that a failure here cannot hide another test.
"""
import numpy as np
import pytest

import oracle
from helpers import assert_within, rng
from gpu_util import announce, device, make_operand, values

pytestmark = pytest.mark.gpu

from dfdx_amd import RocmError  # noqa: E402
from dfdx_amd.rocm import ERR_SCRATCH_TOO_SMALL, KERNEL_AUTO, NOALLOC_SCRATCH_BYTES  # noqa: E402


def both_entries(dtype, m, k, n, layout, accumulate, seed, split_k=0, expect_split=True, check_oracle=True):
    """One product through both entry points on identical inputs; returns nothing, asserts everything."""
    dev = device()
    g = rng(seed)
    at, bt = layout
    a, astr = make_operand(g, m, k, at, dtype, dist="uniform")
    b, bstr = make_operand(g, k, n, bt, dtype, dist="uniform")
    c, cstr = make_operand(g, m, n, False, dtype)
    da, db = dev.tensor(a, dtype), dev.tensor(b, dtype)
    dc_ref, dc_new = dev.tensor(c, dtype), dev.tensor(c, dtype)

    def desc(dc):
        return dev.gemm_desc(dtype, m, k, n, da.ptr, astr, db.ptr, bstr, dc.ptr, cstr, accumulate=accumulate,
                             kernel=KERNEL_AUTO, split_k=split_k)

    plan = dev.gemm_plan(desc(dc_new))[2]
    announce("gemm_noalloc", dtype, (m, k, n), layout, "acc" if accumulate else "ovw", "split_k", split_k, plan)
    if expect_split:
        assert "splitk" in plan or plan == "gemv", plan   # the case must exercise the scratch array
    dev.gemm_noalloc(desc(dc_new))
    dev.gemm(desc(dc_ref))
    dev.synchronize()
    got_st, ref_st = dev.to_host(dc_new), dev.to_host(dc_ref)
    assert np.array_equal(got_st.view(np.uint8), ref_st.view(np.uint8)), "noalloc entry differs from dfdx_rocm_gemm"
    if check_oracle:
        A, B = values(a, dtype, (m, k), astr), values(b, dtype, (k, n), bstr)
        c_or = c.copy()
        oracle.gemm(dtype, m, k, n, accumulate, a, astr, b, bstr, c_or, cstr)
        want = values(c_or, dtype, (m, n), cstr)
        ulp = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
        assert_within(dtype, k, values(got_st, dtype, (m, n), cstr), want, A, B,
                      extra=2 * ulp * float(np.max(np.abs(want))), what="noalloc vs oracle")


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_weight_gradient_shape_twice_second_smaller(dtype):
    # dW-shaped products (TN, beta = 1): few output tiles, long contraction -> the planner splits k
    both_entries(dtype, 512, 8192, 768, (True, False), True, seed=11)
    both_entries(dtype, 256, 4096, 384, (True, False), True, seed=12)


def test_f32_split_twice_second_smaller():
    both_entries("f32", 256, 4096, 512, (True, False), True, seed=21)
    both_entries("f32", 128, 4096, 384, (False, True), False, seed=22)


def test_forced_split_then_unsplit_then_sliced_vector_product():
    both_entries("f16", 1024, 4096, 1024, (False, False), False, seed=31, split_k=4)
    both_entries("f16", 256, 512, 256, (False, True), False, seed=32, expect_split=False)   # no scratch use at all
    # vec.mat with the k axis sliced over the grid: partial sums of the slices go through the same array
    both_entries("f16", 1, 16384, 4096, (False, False), False, seed=33)
    both_entries("f32", 1, 8192, 2048, (False, False), True, seed=34)


def test_full_size_scratch_and_refusal_beyond_it():
    dev = device()
    # config 3's weight gradient: 1024 x 1024 output, K = 16384, 8 splits = exactly the whole array
    both_entries("f16", 1024, 16384, 1024, (True, False), True, seed=41, split_k=8, check_oracle=False)
    # one split more than fits: refused before anything is launched, C untouched, and the ordinary entry still works
    m = n = 1024
    k = 16384
    g = rng(42)
    a, astr = make_operand(g, m, k, True, "f16", dist="uniform")
    b, bstr = make_operand(g, k, n, False, "f16", dist="uniform")
    c = np.full(m * n, 3.0, np.float16)
    da, db, dc = dev.tensor(a, "f16"), dev.tensor(b, "f16"), dev.tensor(c, "f16")
    desc = dev.gemm_desc("f16", m, k, n, da.ptr, astr, db.ptr, bstr, dc.ptr, (n, 1), accumulate=True, split_k=9)
    assert 9 * m * n * 4 > NOALLOC_SCRATCH_BYTES
    announce("gemm_noalloc refusal", dev.gemm_plan(desc)[2])
    with pytest.raises(RocmError) as err:
        dev.gemm_noalloc(desc)
    assert err.value.code == ERR_SCRATCH_TOO_SMALL and "scratch" in str(err.value)
    dev.synchronize()
    assert np.array_equal(dev.to_host(dc), c)
    dev.gemm(desc)
    dev.synchronize()
    assert not np.array_equal(dev.to_host(dc), c)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("m,k,n,layout,accumulate,copies", [
    (2305, 1024, 2051, (False, True), False, "none"),      # only C is off the grid: no space needed
    (2049, 1153, 1031, (False, False), False, "fit"),
    (4095, 4095, 4097, (False, False), True, "too large"), # 67 MB of copies
    (8193, 2049, 2047, (False, True), False, "too large"),
    (261, 6795, 871, (True, False), True, "fit"),          # split contraction
    (361, 2469, 4606, (False, False), False, "fit"),
    (1023, 9001, 1021, (True, False), True, "too large"),  # split contraction
])
def test_operands_off_the_grid(dtype, m, k, n, layout, accumulate, copies):
    """The same bits with the copies in the array, with none, and with the operands read where they lie because the copies do not fit."""
    dev = device()
    at, bt = layout
    sizes = [x * 64 * -(-y // 64) * 2 for x, y in ((m, k), (n, k))] if k % 64 else [0]
    assert copies == "none" or (sum(sizes) > NOALLOC_SCRATCH_BYTES) == (copies == "too large")
    desc = dev.gemm_desc(dtype, m, k, n, 256, (1, m) if at else (k, 1), 512, (1, k) if bt else (n, 1), 1024, (n, 1), accumulate=accumulate)
    plan = dev.gemm_plan(desc)[2]
    assert "_realigned" in plan, plan
    both_entries(dtype, m, k, n, layout, accumulate, seed=m + k, expect_split=False, check_oracle=m * k * n < 1 << 33)


@pytest.mark.parametrize("dtype,m,k,n,layout,accumulate", [
    ("f16", 512, 5056, 4416, (True, False), True), ("bf16", 1344, 4416, 4032, (True, False), True), ("bf16", 6400, 5568, 896, (False, True), False),
    ("f16", 1472, 4224, 3968, (False, False), False), ("bf16", 1472, 12160, 2624, (False, False), False),
])
def test_pieces_of_large_tiles_fit(dtype, m, k, n, layout, accumulate):
    """Products that 256 x 192 tiles would take in pieces of 42 to 47 MB, and other tiles in less."""
    both_entries(dtype, m, k, n, layout, accumulate, seed=m + k, expect_split=False, check_oracle=False)


@pytest.mark.parametrize("m,k,n,at", [(2049, 1153, 1031, False), (261, 6795, 871, True), (2305, 1024, 2051, False)])
def test_captured_into_a_graph_with_a_cold_context(m, k, n, at):
    """A context that has no buffer yet allocates none while its stream is captured: the operands are read where they lie (a split
    needs its partial sums, so that context has run a small split product before), and every replay leaves the bits of the eager call."""
    import torch

    from dfdx_amd import Rocm

    dev, g, dtype = device(), rng(7), "f16"
    a, astr = make_operand(g, m, k, at, dtype, dist="uniform")
    b, bstr = make_operand(g, k, n, False, dtype, dist="uniform")
    da, db, want = dev.tensor(a, dtype), dev.tensor(b, dtype), dev.zeros(dtype, (m, n))
    desc = lambda d, c: d.gemm_desc(dtype, m, k, n, da.ptr, astr, db.ptr, bstr, c.ptr, (n, 1))
    name = dev.gemm_plan(desc(dev, want))[2]
    assert "_realigned" in name, name
    announce("captured", (m, k, n), name)
    dev.gemm(desc(dev, want))
    dev.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        own = Rocm(0)
        if "splitk" in name:   # 16 MB of partial sums, less than the copies need besides
            x = own.zeros("f32", (1024, 1024))
            own.gemm(own.gemm_desc("f32", 512, 1024, 1024, x.ptr, (1024, 1), x.ptr, (1024, 1), own.zeros("f32", (512, 1024)).ptr, (1024, 1), split_k=8, kernel=2, variant=4))
        out = own.zeros(dtype, (m, n))
        own.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            own.gemm(desc(own, out))
        for _ in range(3):
            out.storage.fill_(0x55)
            graph.replay()
            own.synchronize()
            assert np.array_equal(own.to_host(out).view(np.uint16), dev.to_host(want).view(np.uint16))
    own.close()


@pytest.mark.parametrize("dtype,m,k,n,at,plan", [("f16", 12, 6077, 218, False, "gemv_rows"), ("f32", 3, 9001, 300, False, "gemv_rows"),
                                                 ("bf16", 8, 2496, 384, True, "_ring_64x64x64_w2x2_s4_splitk"), ("f16", 16, 10304, 1091, False, "_ring_64x64x64_w2x2_s4_splitk")])
def test_a_cold_context_captures_in_one_piece(dtype, m, k, n, at, plan):
    """Slices of the contraction on kernels that took such products from others without partial sums: where there is no space for the sums and
    none can be had, one piece."""
    import torch

    from dfdx_amd import Rocm

    dev, g = device(), rng(k)
    a, astr = make_operand(g, m, k, at, dtype)
    b, bstr = make_operand(g, k, n, not at, dtype)
    da, db = dev.tensor(a, dtype), dev.tensor(b, dtype)
    desc = lambda d, c: d.gemm_desc(dtype, m, k, n, da.ptr, astr, db.ptr, bstr, c.ptr, (n, 1))
    name = dev.gemm_plan(desc(dev, da))[2]
    announce("captured, cold", dtype, (m, k, n), name)
    assert plan in name, name
    dev.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        own = Rocm(0)
        out = own.zeros(dtype, (m, n))
        own.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            own.gemm(desc(own, out))
        A, B = values(a, dtype, (m, k), astr), values(b, dtype, (k, n), bstr)
        want = A @ B
        ulp = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
        for _ in range(3):
            out.storage.fill_(0x55)
            graph.replay()
            own.synchronize()
            assert_within(dtype, k, oracle.to_f64(own.to_host(out), dtype).reshape(m, n), want, A, B, extra=ulp * float(np.abs(want).max()), what=name)
    own.close()


@pytest.mark.parametrize("m,k,n,variant", [(704, 874, 512, 0), (512, 1024, 512, 4), (512, 1024, 512, 7)])
def test_pieces_that_were_asked_for_are_not_dropped(m, k, n, variant):
    """f32 in three pieces because the caller says so: captured with no space it is refused, not run in another order."""
    import torch

    from dfdx_amd import Rocm

    dev, g = device(), rng(k)
    a, astr = make_operand(g, m, k, False, "f32")
    b, bstr = make_operand(g, k, n, True, "f32")
    da, db, want = dev.tensor(a, "f32"), dev.tensor(b, "f32"), dev.zeros("f32", (m, n))
    desc = lambda d, c, **kw: d.gemm_desc("f32", m, k, n, da.ptr, astr, db.ptr, bstr, c.ptr, (n, 1), kernel=2, variant=variant, **kw)
    name = dev.gemm_plan(desc(dev, want, split_k=3))[2]
    announce("captured, cold, pieces asked for", (m, k, n), name)
    assert "splitk3" in name, name
    dev.gemm(desc(dev, want, split_k=3))
    dev.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        own = Rocm(0)
        out, other = own.zeros("f32", (m, n)), own.zeros("f32", (m, n))
        own.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            with pytest.raises(RocmError) as err:
                own.gemm(desc(own, out, split_k=3))
            own.gemm(desc(own, other, no_split_k=True))
        assert err.value.code == ERR_SCRATCH_TOO_SMALL
        for _ in range(3):
            graph.replay()
            own.synchronize()
            assert not own.to_host(out).any() and own.to_host(other).any()
        own.gemm(desc(own, out, split_k=3))   # outside a capture the space is had
        own.synchronize()
        assert np.array_equal(own.to_host(out).view(np.uint32), dev.to_host(want).view(np.uint32))
        del graph
    own.close()


@pytest.mark.parametrize("dtype,m,k,n", [("f16", 12, 6077, 218), ("f32", 16, 7744, 1100), ("bf16", 1090, 7177, 16), ("f16", 16, 10304, 1091)])
def test_few_rows_in_slices(dtype, m, k, n):
    """The partial sums of up to sixteen slices, or of the ring tiles' pieces, of one to sixteen rows fit the array."""
    name = device().gemm_plan(device().gemm_desc(dtype, m, k, n, 256, (k, 1), 512, (1, k), 1024, (n, 1)))[2]
    assert "gemv_rows" in name or "_ring_" in name, name
    both_entries(dtype, m, k, n, (False, True), True, seed=k, expect_split=False)
