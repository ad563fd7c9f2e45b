"""Convolutions of images with one or three channels against float64: ends of tiles and bands, every filter size and stride,
channel counts around the blocks of 32 and 64, gradients stored and added, infinities."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from gpu_util import announce, device

from dfdx_amd import View

pytestmark = pytest.mark.gpu

TYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
EPS = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def view(t, dtype):
    return View(t.view(torch.uint8).reshape(-1), dtype, tuple(t.shape), tuple(t.stride()))


def reference(x, w, g, stride):
    """Output, gradients and, for the bounds, the sums of magnitudes behind each value; float64 on the CPU."""
    def conv(a, b, c):
        a, b = a.clone().requires_grad_(), b.clone().requires_grad_()
        y = F.conv2d(a, b, stride=stride, padding=w.shape[-1] // 2)
        return (y.detach(), *torch.autograd.grad(y, (a, b), c))
    x, w, g = (t.double().cpu() for t in (x, w, g))
    return conv(x, w, g), conv(x.abs(), w.abs(), g.abs())


def check(what, got, want, mag, terms, dtype, old=None):
    # one rounding of the result, f32 sums in any order of `terms` products, the rounding to nothing below the type's normals
    want = want + (old.double().cpu() if old is not None else 0)
    bound = EPS[dtype] * want.abs() + (mag + want.abs()) * terms * 2.0 ** -24 + 2.0 ** -24
    bad = (got.double().cpu() - want).abs() > bound
    assert not bool(bad.any()), (what, int(bad.sum()), float((got.double().cpu() - want).abs().max()))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("batch,cin,cout,h,w,k,stride", [
    (2, 3, 64, 32, 224, 7, 2),
    (3, 3, 64, 37, 48, 7, 2),      # odd height: a cell row cut in half, a last band of few rows
    (1, 1, 70, 18, 272, 7, 2),     # a second group of 64 channels in the forward (the backward goes through the patch matrix), 136 cells
    (2, 3, 33, 16, 32, 5, 2),
    (2, 1, 16, 9, 16, 3, 2),
    (2, 3, 64, 21, 40, 3, 1),
    (1, 3, 130, 16, 72, 3, 1),     # (so does the backward of this one)
    (2, 3, 24, 13, 64, 5, 1),
    (1, 1, 10, 28, 32, 5, 1),
    (1, 3, 32, 10, 24, 7, 1),      # (the backward of this one goes through the patch matrix)
    (40, 3, 8, 8, 16, 3, 2),
])
def test_against_float64(dtype, batch, cin, cout, h, w, k, stride):
    dev = device()
    announce("conv few", dtype, batch, cin, cout, h, w, k, stride)
    gen = torch.Generator(device="cuda").manual_seed(h * w + k)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, f = rnd(batch, cin, h, w).to(TYPES[dtype]), (rnd(cout, cin, k, k) / (cin * k * k) ** 0.5).to(TYPES[dtype])
    ho, wo = (h - 1) // stride + 1, (w - 1) // stride + 1
    g = rnd(batch, cout, ho, wo).to(TYPES[dtype])
    how = dict(stride=stride, padding=k // 2)
    (y, gx, gw), (my, mgx, mgw) = reference(x, f, g, stride)
    got = dev.conv2d_forward(view(x, dtype), view(f, dtype), **how)
    check("out", got.storage.view(TYPES[dtype]).reshape(y.shape), y, my, cin * k * k, dtype)
    general = (k == 7 and stride == 1) or cout > 64   # the general form rounds every tap's share of the image gradient
    for fresh in (True, False):
        ox, ow = rnd(*x.shape).to(TYPES[dtype]), rnd(*f.shape).to(TYPES[dtype])
        gi, gf = view(ox.clone(), dtype), view(ow.clone(), dtype)
        if fresh:
            gi, gf = dev.zeros_many([view(x, dtype), view(f, dtype)], deferred=True)
        dev.conv2d_backward(view(x, dtype), gi, view(f, dtype), gf, view(g, dtype), **how)
        dev.settle_zeros()
        if not general:
            check("grad_img", gi.storage.view(TYPES[dtype]).reshape(x.shape), gx, mgx, cout * k * k, dtype, None if fresh else ox)
        check("grad_filters", gf.storage.view(TYPES[dtype]).reshape(f.shape), gw, mgw, batch * ho * wo, dtype, None if fresh else ow)


@pytest.mark.parametrize("stride,k", [(2, 7), (1, 3)])
def test_infinities_reach_what_reads_them_and_nothing_else(stride, k):
    dev, dtype = device(), "f16"
    x = torch.randn(1, 3, 32, 96, device="cuda").half()
    f = (torch.randn(64, 3, k, k, device="cuda") / 12).half()
    y = dev.conv2d_forward(view(x, dtype), view(f, dtype), stride=stride, padding=k // 2)
    x[0, 1, 9, 40] = float("inf")
    bad = dev.conv2d_forward(view(x, dtype), view(f, dtype), stride=stride, padding=k // 2)
    a, b = (t.storage.view(torch.float16).reshape(t.shape) for t in (y, bad))
    reach = F.conv2d((~torch.isfinite(x)).float().sum(1, keepdim=True).cpu(), torch.ones(1, 1, k, k), stride=stride, padding=k // 2).cuda() > 0
    assert bool((~torch.isfinite(b)).any()) and torch.equal(torch.where(reach, 0, a), torch.where(reach, 0, b))
    x[0, 1, 9, 40] = 0.5
    g = torch.randn(*y.shape, device="cuda").half()
    grads = []
    for value in (None, float("nan")):
        if value is not None:
            g[0, 5, 3, 17] = value
        gi, gf = dev.zeros_many([view(x, dtype), view(f, dtype)], deferred=True)
        dev.conv2d_backward(view(x, dtype), gi, view(f, dtype), gf, view(g, dtype), stride=stride, padding=k // 2)
        dev.settle_zeros()
        grads.append((gi.storage.view(torch.float16).reshape(x.shape).clone(), gf.storage.view(torch.float16).reshape(f.shape).clone()))
    hit = torch.zeros(1, 1, *y.shape[2:])
    hit[0, 0, 3, 17] = 1
    pads = (x.shape[2] - ((y.shape[2] - 1) * stride - 2 * (k // 2) + k), x.shape[3] - ((y.shape[3] - 1) * stride - 2 * (k // 2) + k))
    reach = F.conv_transpose2d(hit, torch.ones(1, 1, k, k), stride=stride, padding=k // 2, output_padding=pads).cuda() > 0
    (a, fa), (b, fb) = grads
    assert bool(torch.isnan(b[:, :, 0]).any() or torch.isnan(b).any()) and bool(torch.isnan(torch.where(reach, b, float("nan"))).all())
    assert bool(torch.isfinite(torch.where(reach, 0, b)).all())
    assert torch.allclose(torch.where(reach, 0, a).float(), torch.where(reach, 0, b).float(), rtol=2e-3, atol=2e-3)
    other = torch.arange(64) != 5
    assert torch.equal(fa[other], fb[other]) and bool(torch.isnan(fb[5]).all())


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("k,stride,hw", [(7, 2, (37, 48)), (5, 2, (18, 32)), (3, 2, (9, 16)), (5, 1, (13, 64)), (3, 1, (21, 40))])
@pytest.mark.parametrize("where", ["filter", "gradient", "corner", "both"])
def test_image_gradient_of_infinities(dtype, k, stride, hw, where):
    """An infinite filter value or gradient: infinities and NaN where the sums over a pixel's taps have them (and not where a tap
    lies outside of the output), and the other pixels within the bound of finite values."""
    dev, (batch, cin, cout), pad = device(), (2, 3, 40), k // 2
    h, w = hw
    announce("conv few, infinities", dtype, k, stride, where)
    gen = torch.Generator(device="cuda").manual_seed(k)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    x, f = rnd(batch, cin, h, w).to(TYPES[dtype]), (rnd(cout, cin, k, k) / 10).to(TYPES[dtype])
    ho, wo = (h - 1) // stride + 1, (w - 1) // stride + 1
    g = rnd(batch, cout, ho, wo).to(TYPES[dtype])
    if where in ("filter", "both"):
        f[35, 1, 0, k - 1] = float("inf")
    if where in ("gradient", "both"):
        g[1, 7, ho // 2, wo // 2] = float("-inf")
    if where == "corner":
        g[0, 39, 0, 0], g[1, 0, ho - 1, wo - 1] = float("inf"), float("-inf")
    gi, gf = dev.zeros_many([view(x, dtype), view(f, dtype)], deferred=True)
    dev.conv2d_backward(view(x, dtype), gi, view(f, dtype), gf, view(g, dtype), stride=stride, padding=pad)
    dev.settle_zeros()
    got = gi.storage.view(TYPES[dtype]).reshape(x.shape).double().cpu()
    want, mag = torch.zeros(x.shape, dtype=torch.float64), torch.zeros(x.shape, dtype=torch.float64)
    f64, g64 = f.double().cpu(), g.double().cpu()
    for k1 in range(k):   # tap by tap, over the outputs that a tap reads from inside of the image
        rows = [o for o in range(ho) if 0 <= o * stride + k1 - pad < h]
        for k2 in range(k):
            cols = [o for o in range(wo) if 0 <= o * stride + k2 - pad < w]
            part = g64[:, :, rows][:, :, :, cols]
            y, z = rows[0] * stride + k1 - pad, cols[0] * stride + k2 - pad
            at = (slice(None), slice(None), slice(y, y + (len(rows) - 1) * stride + 1, stride), slice(z, z + (len(cols) - 1) * stride + 1, stride))
            want[at] += torch.stack([(f64[None, :, c, k1, k2, None, None] * part).sum(1) for c in range(cin)], 1)
            mag[at] += torch.stack([(f64[None, :, c, k1, k2, None, None] * part).abs().sum(1) for c in range(cin)], 1)
    finite = torch.isfinite(want)
    assert bool((~finite).any()) and bool(finite.any())
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
    check("grad_img", got[finite], want[finite], mag[finite], cout * k * k, dtype)


def test_an_infinite_filter_does_not_stall_the_step():
    """A step whose values have overflowed is worth nothing and has to end all the same: within four times a finite one's time."""
    dev, dtype = device(), "f16"
    x, f, g = torch.randn(16, 3, 224, 224, device="cuda").half(), torch.randn(64, 3, 7, 7, device="cuda").half(), torch.randn(16, 64, 112, 112, device="cuda").half()
    gi, gf = dev.zeros(dtype, x.shape), dev.zeros(dtype, f.shape)

    def best():
        times = []
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            dev.conv2d_backward(view(x, dtype), gi, view(f, dtype), gf, view(g, dtype), stride=2, padding=3)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    announce("conv few, time of an infinite filter")
    finite = best()
    f[3, 1, 2, 2] = float("inf")
    assert best() < 4 * finite + 0.1
