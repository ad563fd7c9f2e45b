"""Products of the 16-bit types whose operands are copied onto the 16-byte grid for the LDS-DMA kernels: odd extents in each
place, contractions that end inside a k tile, a C at any address, padded leading dimensions, batches, shared operands."""
import threading

import numpy as np
import pytest
import torch

import oracle
from helpers import assert_within, rng
from gpu_util import announce, device

from dfdx_amd import Rocm, View
from dfdx_amd.rocm import KERNEL_AUTO
from test_gpu_gemm import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("m,k,n,layout,pads", [
    (2049, 1153, 1031, "nn", (0, 0, 0)),     # every extent odd, both copies
    (2047, 1217, 2049, "nt", (1, 3, 1)),     # odd leading dimensions
    (1025, 2111, 1279, "tn", (0, 5, 3)),     # A across k: zero rows behind the last
    (2305, 1024, 2051, "nt", (0, 0, 0)),     # no copy at all: only C is off the grid
    (2048, 1001, 2048, "nn", (0, 0, 0)),     # only the contraction is off the k tile
    (261, 6795, 871, "tn", (0, 0, 0)),       # split contraction
    (16384, 2048, 50, "tn", (0, 0, 0)),      # narrow output: the 64-column tile
])
@pytest.mark.parametrize("accumulate,bias,colmajor", [(False, True, False), (True, False, False), (True, False, True), (False, True, True)])
def test_operands_off_the_grid(dtype, m, k, n, layout, pads, accumulate, bias, colmajor):
    name = run_case(dtype, m, k, n, layout, accumulate, KERNEL_AUTO, 0, bias=bias, c_colmajor=colmajor, pads=pads, seed=m + k)
    if not colmajor:
        assert "_dma_" in name and "_realigned" in name, name


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("shift", [0, 1])
def test_batches_and_addresses_off_the_grid(dtype, shared, shift):
    """A batch whose matrices start anywhere, one operand shared by all of them, every pointer `shift` elements off."""
    dev, g = device(), rng(91)
    nb, m, k, n = 3, 2049, 1027, 2051
    a = oracle.to_storage(g.standard_normal(shift + nb * m * k), dtype)
    b = oracle.to_storage(g.standard_normal(shift + (1 if shared else nb) * k * n), dtype)
    c = oracle.to_storage(g.standard_normal(shift + nb * m * n + 8), dtype)
    da, db, dc = (dev.tensor(t, dtype) for t in (a, b, c))
    desc = dev.gemm_desc(dtype, m, k, n, da.ptr + 2 * shift, (k, 1), db.ptr + 2 * shift, (n, 1), dc.ptr + 2 * shift, (n, 1), accumulate=True,
                         batch=(nb, 1), a_batch=(m * k, 0), b_batch=(0 if shared else k * n, 0), c_batch=(m * n, 0))
    name = dev.gemm_plan(desc)[2]
    announce("realigned batch", dtype, shared, shift, name)
    assert "_realigned" in name, name
    dev.gemm(desc)
    got = oracle.to_f64(dev.to_host(dc), dtype)
    A = oracle.to_f64(a, dtype)[shift:].reshape(nb, m, k)
    B = oracle.to_f64(b, dtype)[shift:].reshape(-1, k, n)
    C = oracle.to_f64(c, dtype)
    assert np.array_equal(got[:shift], C[:shift]) and np.array_equal(got[shift + nb * m * n:], C[shift + nb * m * n:])
    ulp = 2.0 ** (-11 if dtype == "f16" else -8)
    for i in range(nb):
        Bi = B[0 if shared else i]
        want = A[i] @ Bi + C[shift + i * m * n: shift + (i + 1) * m * n].reshape(m, n)
        assert_within(dtype, k, got[shift + i * m * n: shift + (i + 1) * m * n].reshape(m, n), want, A[i], Bi, extra=ulp * float(np.abs(want).max()))


def test_infinities_stay_in_their_row_and_column():
    """The zeros that pad a copy meet zeros only: an infinite value in the last place of A reaches its row and nothing else."""
    dev = device()
    m, k, n, dtype = 2049, 1153, 1031, "f16"
    a = torch.randn(m, k, device="cuda").half()
    b = torch.rand(k, n, device="cuda").half() + 0.5
    a[m - 1, k - 1] = float("inf")
    view = lambda t: View(t.view(torch.uint8).reshape(-1), dtype, tuple(t.shape), tuple(t.stride()))
    y = dev.forward(view(a), view(b)).storage.view(torch.float16).reshape(m, n)
    assert bool(torch.isfinite(y[:-1]).all()) and bool((y[-1] == float("inf")).all())


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rows,cols", [(2048, 50257), (3, 129), (77, 1001), (512, 135)])
def test_bias_gradient_of_odd_rows(dtype, rows, cols):
    """Column sums of rows off the 16-byte grid; f32 sums, one rounding: half an ulp of the result and rows * 2^-24 of the sum of magnitudes."""
    dev = device()
    t = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.randn(rows, cols, device="cuda").to(t)
    old = torch.randn(cols, device="cuda").to(t)
    gb = old.clone()
    view = lambda t_: View(t_.view(torch.uint8).reshape(-1), dtype, tuple(t_.shape), tuple(t_.stride()))
    dev.bias_backward(view(g), view(gb))
    want = g.double().sum(0) + old.double()
    bound = want.abs() * 2.0 ** (-11 if dtype == "f16" else -8) + (g.double().abs().sum(0) + old.double().abs()) * rows * 2.0 ** -24 + 1e-7
    assert bool(((gb.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rows,inp,out", [(2048, 1024, 3001), (2113, 1024, 2112), (1500, 1111, 3333)])
def test_backward_products_share_one_copy_of_grad_out(dtype, rows, inp, out):
    """Both products of a backward call read grad_out; off the grid it is copied once for both, in Linear, the plain product and the
    broadcast one.  Against the two products as single calls, each with its own copies: the same kernels, the same bits."""
    dev = device()
    t = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    view = lambda t_: View(t_.view(torch.uint8).reshape(-1), dtype, tuple(t_.shape), tuple(t_.stride()))
    rnd = lambda *s: torch.randn(*s, device="cuda").to(t)
    x, w, b, g = rnd(rows, inp), rnd(out, inp) / 32, rnd(out), rnd(rows, out)
    wt = view(w).permute(1, 0)
    flat = lambda v: v.storage.view(t)
    gx, gw = torch.zeros_like(x), torch.zeros_like(w)
    for d in (dev.gemm_desc(dtype, rows, out, inp, g.data_ptr(), (out, 1), w.data_ptr(), (inp, 1), gx.data_ptr(), (inp, 1), accumulate=True),
              dev.gemm_desc(dtype, inp, rows, out, x.data_ptr(), (1, inp), g.data_ptr(), (out, 1), gw.data_ptr(), (1, inp), accumulate=True)):
        name = dev.gemm_plan(d)[2]
        announce("shared copy", dtype, rows, inp, out, name)
        assert "_realigned" in name or out == 2112, name   # (2112 columns are whole k tiles: only one product needs a copy)
        dev.gemm(d)
    for fresh in (True, False):
        ox, ow, ob = view(torch.zeros_like(x)), view(torch.zeros_like(w)), view(torch.zeros_like(b))
        if fresh:
            ox, ow, ob = dev.zeros_many([view(x), view(w), view(b)], deferred=True)
        dev.linear_backward(view(x), ox, view(w), ow, ob, view(g))
        dev.settle_zeros()
        assert torch.equal(flat(ox), gx.view(-1)) and torch.equal(flat(ow), gw.view(-1))
        assert torch.allclose(flat(ob).double(), g.double().sum(0), rtol=2.0 ** -7 if dtype == "bf16" else 2.0 ** -10, atol=1e-2)
        px, pw = view(torch.zeros_like(x)), view(torch.zeros_like(w)).permute(1, 0)
        dev.backward(view(x), px, wt, pw, view(g))
        assert torch.equal(flat(px), gx.view(-1)) and torch.equal(pw.storage.view(t), gw.view(-1))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rows,inp,out", [(2048, 1024, 3001), (2113, 1024, 2112), (1537, 1024, 1367), (513, 1024, 50257)])
def test_bias_gradient_taken_on_the_way_into_the_copy(dtype, rows, inp, out):
    """Column sums that ride on the copy of grad_out, added to an old gradient and stored into a fresh one, at ragged rows, ragged
    columns and both; f32 sums, one rounding: half an ulp of the result and rows * 2^-24 of the sum of magnitudes."""
    dev = device()
    t = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    view = lambda t_: View(t_.view(torch.uint8).reshape(-1), dtype, tuple(t_.shape), tuple(t_.stride()))
    rnd = lambda *s: torch.randn(*s, device="cuda").to(t)
    x, w, old, g = rnd(rows, inp), rnd(out, inp) / 32, rnd(out), rnd(rows, out)
    for start in (old, None):
        ox, ow, ob = dev.zeros_many([view(x), view(w), view(old)], deferred=True)
        if start is not None:
            ob = view(old.clone())
        dev.linear_backward(view(x), ox, view(w), ow, ob, view(g))
        dev.settle_zeros()
        before = old.double() if start is not None else torch.zeros_like(old).double()
        want = g.double().sum(0) + before
        bound = want.abs() * 2.0 ** (-11 if dtype == "f16" else -8) + (g.double().abs().sum(0) + before.abs()) * rows * 2.0 ** -24 + 1e-7
        assert bool(((ob.storage.view(t).double() - want).abs() <= bound).all())


def linear_operands(rows, inp, out):
    view = lambda t: View(t.view(torch.uint8).reshape(-1), "f16", tuple(t.shape), tuple(t.stride()))
    rnd = lambda *s: torch.randn(*s, device="cuda").half()
    return [view(t) for t in (rnd(rows, inp), rnd(out, inp) / 32, rnd(out), rnd(rows, out))]


def linear_gradients(dev, x, w, b, g):
    grads = dev.zeros_many([x, w, b], deferred=True)
    dev.linear_backward(x, grads[0], w, grads[1], grads[2], g)
    dev.settle_zeros()
    return grads


def test_the_shared_copy_has_its_space_once():
    """grad_out (4096 x 20001) is copied into one buffer; the input gradient's own space holds the weight's copy (41 MB) and partial sums
    (at most 64 MB), and no second copy of grad_out (164 MB)."""
    operands = linear_operands(4096, 1024, 20001)
    linear_gradients(device(), *operands)
    torch.cuda.synchronize()
    announce("space of a shared copy")
    own = Rocm(0)   # a context without buffers
    grads = own.zeros_many(operands[:3], deferred=True)
    own.synchronize()
    before = torch.cuda.mem_get_info()[0]
    own.linear_backward(operands[0], grads[0], operands[1], grads[1], grads[2], operands[3])
    own.synchronize()
    taken = before - torch.cuda.mem_get_info()[0]
    own.close()
    assert 160 << 20 < taken < 300 << 20, taken >> 20


def test_shared_copy_without_room_for_it():
    """On a stream that is being captured the context allocates nothing: each product reads its operands where they lie, with the same
    bits; the bias gradient is summed by itself (f32 sums, one rounding)."""
    dev = device()
    operands = linear_operands(2048, 1024, 3001)
    want = [dev.to_host(t).copy() for t in linear_gradients(dev, *operands)]
    announce("shared copy, captured")
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        own = Rocm(0)
        own.bias_backward(operands[3], own.zeros("f16", (3001,)))   # (room for the sums, 16 rows of them, and no more)
        grads = [own.zeros("f16", t.shape) for t in operands[:3]]
        own.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            own.linear_backward(operands[0], grads[0], operands[1], grads[1], grads[2], operands[3])
        for _ in range(3):
            for t in grads:
                t.storage.zero_()
            graph.replay()
            own.synchronize()
            got = [own.to_host(t) for t in grads]
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
            assert np.abs(got[2].astype(np.float64) - want[2].astype(np.float64)).max() <= 2.0 ** -10 * np.abs(want[2].astype(np.float64)).max()
    own.close()


def test_shared_copies_of_two_threads():
    """The copy of grad_out lives in the context's buffer until both products have been launched: calls of other threads stay out."""
    dev = device()
    announce("shared copy, threads")
    jobs = [linear_operands(2048 + 64 * t, 512, 2001 + 2 * t) for t in range(3)]
    want = [[dev.to_host(t).copy() for t in linear_gradients(dev, *j)] for j in jobs]
    got, errors = [[] for _ in jobs], []

    def worker(i):
        try:
            for _ in range(8):
                got[i].append([dev.to_host(t).copy() for t in linear_gradients(dev, *jobs[i])])
        except Exception as e:  # surfaced in the main thread
            errors.append(e)

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for runs, ref in zip(got, want):
        assert len(runs) == 8 and all(np.array_equal(a, b) for run in runs for a, b in zip(run, ref))


def test_copies_are_bounded():
    """Two gigabytes of copies at most; beyond, and at leading dimensions that the copies need not, the operands are read where they lie."""
    dev = device()
    plan = lambda m, k, n: dev.gemm_plan(dev.gemm_desc("f16", m, k, n, 256, (k, 1), 512, (n, 1), 1024, (n, 1)))[2]   # (no launch)
    assert "_realigned" in plan(20001, 20001, 20001) and "_realigned" not in plan(30001, 30001, 30001)


def test_rising_sizes_do_not_leave_a_buffer_behind_at_every_step():
    """Linear backward with a wide odd output and ever more rows, nothing synchronized through the library: the buffers grow by half of
    themselves at least (copies of grad_out: 82, 123 and 185 MB; without that, 17 of 82 to 164 MB, and as many workspaces)."""
    rows, out = 4096, 20001
    x, w, b, g = linear_operands(rows, 1024, out)
    part = lambda v, n: View(v.storage[:2 * n * v.shape[1]], v.dtype, (n, v.shape[1]), v.strides)
    announce("rising sizes")
    own = Rocm(0)
    gx, gw, gb = (own.zeros("f16", v.shape) for v in (x, w, b))
    own.synchronize()
    before = torch.cuda.mem_get_info()[0]
    for n in range(2048, rows + 1, 128):
        own.linear_backward(part(x, n), part(gx, n), w, gw, gb, part(g, n))
    torch.cuda.synchronize()
    taken = before - torch.cuda.mem_get_info()[0]
    own.close()
    assert taken < 1000 << 20, taken >> 20
