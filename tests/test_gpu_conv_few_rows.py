"""The image gradient of strided first layers by rows of cells (conv_few.hip): ends of tiles of 16 columns and of groups of four
rows, one to four chunks of 16 channels, both tile counts, more groups than workgroups walk at once, and what infinities reach."""
import pytest
import torch

from gpu_util import announce, device
from test_gpu_conv_few_channels import TYPES, check, reference, view

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("batch,cin,cout,h,w,k", [
    (1, 3, 64, 9, 224, 7), (1, 3, 17, 6, 128, 7), (2, 1, 40, 7, 144, 7),      # 112, 64 and 72 columns of grad_out
    (1, 3, 48, 8, 208, 5), (3, 1, 16, 2, 16, 5), (1, 3, 64, 33, 112, 3), (2, 3, 5, 1, 192, 3),
])
def test_sizes(dtype, batch, cin, cout, h, w, k):
    dev, gen = device(), torch.Generator(device="cuda").manual_seed(w + k)
    announce("conv few rows", dtype, batch, cin, cout, h, w, k)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen).to(TYPES[dtype])
    x, f, g = rnd(batch, cin, h, w), rnd(cout, cin, k, k) / 8, rnd(batch, cout, (h + 1) // 2, w // 2)
    (_, gx, _), (_, mgx, _) = reference(x, f, g, 2)
    for fresh in (True, False):
        old = rnd(*x.shape)
        gi, gf = dev.zeros_many([view(x, dtype), view(f, dtype)], deferred=True) if fresh else (view(old.clone(), dtype), view(torch.zeros_like(f), dtype))
        dev.conv2d_backward(view(x, dtype), gi, view(f, dtype), gf, view(g, dtype), stride=2, padding=k // 2)
        dev.settle_zeros()
        check("grad_img", gi.storage.view(TYPES[dtype]).reshape(x.shape), gx, mgx, cout * k * k, dtype, None if fresh else old)


@pytest.mark.parametrize("k", [3, 5, 7])
@pytest.mark.parametrize("w,col", [(224, 0), (224, 15), (224, 16), (224, 111), (96, 47)])
def test_an_infinity_at_an_edge(k, w, col):
    """Only the pixels with a tap at it, and the finite ones as they are without it."""
    dev, dtype, h, cout, row = device(), "f16", 14, 33, 4
    announce("conv few rows, infinity", k, w, col)
    gen = torch.Generator(device="cuda").manual_seed(col)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen).to(TYPES[dtype])
    x, f, g = rnd(2, 3, h, w), rnd(cout, 3, k, k) / 8, rnd(2, cout, h // 2, w // 2)
    g[1, 20, row, col] = 0
    results = []
    for value in (0.0, float("inf")):
        g[1, 20, row, col] = value
        gi, gf = dev.zeros_many([view(x, dtype), view(f, dtype)], deferred=True)
        dev.conv2d_backward(view(x, dtype), gi, view(f, dtype), gf, view(g, dtype), stride=2, padding=k // 2)
        dev.settle_zeros()
        results.append(gi.storage.view(TYPES[dtype]).reshape(x.shape).clone())
    reach = torch.zeros(2, 3, h, w, dtype=torch.bool, device="cuda")
    y, z = 2 * row - k // 2, 2 * col - k // 2
    reach[1, :, max(0, y):min(h, y + k), max(0, z):min(w, z + k)] = True
    assert torch.equal(~torch.isfinite(results[1]), reach)
    # (formed again position by position: the sums in another order, of cout * k * k terms of 8 at the most behind an f16 rounding)
    a, b = (torch.where(reach, 0, r).float() for r in results)
    assert bool(((a - b).abs() <= 2.0 ** -10 * a.abs() + cout * k * k * 8 * 2.0 ** -24).all())


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("batch,cin,cout,h,w,k", [(1100, 3, 16, 8, 32, 7), (1100, 3, 64, 7, 32, 3), (1100, 3, 10, 8, 160, 3), (700, 3, 64, 14, 144, 5)])
def test_several_groups_a_workgroup(dtype, batch, cin, cout, h, w, k):
    """Two workgroups a compute unit walk what is more than 512 groups: the next group's rows on their way under this one's sums."""
    dev, gen = device(), torch.Generator(device="cuda").manual_seed(cout + k)
    announce("conv few rows, walked", dtype, batch, cin, cout, h, w, k)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen).to(TYPES[dtype])
    x, f, g = rnd(batch, cin, h, w), rnd(cout, cin, k, k) / 8, rnd(batch, cout, (h + 1) // 2, w // 2)
    assert batch * -(-g.shape[2] // 4) > 1024
    image = lambda f, g: torch.nn.grad.conv2d_input(x.shape, f.double().cpu(), g.double().cpu(), stride=2, padding=k // 2)
    want, mag = image(f, g), image(f.abs(), g.abs())
    for fresh in (True, False):
        old = rnd(*x.shape)
        gi, gf = dev.zeros_many([view(x, dtype), view(f, dtype)], deferred=True) if fresh else (view(old.clone(), dtype), view(torch.zeros_like(f), dtype))
        dev.conv2d_backward(view(x, dtype), gi, view(f, dtype), gf, view(g, dtype), stride=2, padding=k // 2)
        dev.settle_zeros()
        check("grad_img", gi.storage.view(TYPES[dtype]).reshape(x.shape), want, mag, cout * k * k, dtype, None if fresh else old)


@pytest.mark.parametrize("cout,w", [(16, 32), (64, 32), (16, 160), (64, 160)])
def test_an_infinity_in_an_early_group(cout, w):
    """The groups that a workgroup walks behind one that it has formed again are what they are without it, bit for bit."""
    dev, dtype, batch, h, k = device(), "f16", 1100, 8, 7
    announce("conv few rows, infinity early", cout, w)
    gen = torch.Generator(device="cuda").manual_seed(w)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen).to(TYPES[dtype])
    x, f, g = rnd(batch, 3, h, w), rnd(cout, 3, k, k) / 8, rnd(batch, cout, h // 2, w // 2)
    images = [0, 1, 77, 300, 511, 512, 600]   # one group of four rows each
    results = []
    for value in (0.0, float("inf")):
        g[images, cout - 1, 2, w // 2 - 1] = value
        gi, gf = dev.zeros_many([view(x, dtype), view(f, dtype)], deferred=True)
        dev.conv2d_backward(view(x, dtype), gi, view(f, dtype), gf, view(g, dtype), stride=2, padding=k // 2)
        dev.settle_zeros()
        results.append(gi.storage.view(TYPES[dtype]).reshape(x.shape).clone())
    others = torch.ones(batch, dtype=torch.bool, device="cuda")
    others[images] = False
    assert torch.equal(results[0][others], results[1][others]) and bool(torch.isfinite(results[0]).all())
    assert bool((~torch.isfinite(results[1][images])).flatten(1).any(1).all())
