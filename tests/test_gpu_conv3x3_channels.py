"""3 x 3 unit-stride convolutions whose channel counts are no whole blocks of the band kernels (conv3x3.hip, conv3x3_wgrad.hip):
the last block of outputs and the last chunk of inputs are partial."""
import numpy as np
import pytest

import oracle
from gpu_util import announce, device, launches
from helpers import rng

pytestmark = pytest.mark.gpu
EPS = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def correlate(img, fil):
    """out[b][o][y][x] = sum of fil[o][c][ky][kx] * img[b][c][y + ky - 1][x + kx - 1] in 64 bits."""
    pad = np.pad(img, ((0, 0), (0, 0), (1, 1), (1, 1)))
    h, w = img.shape[2:]
    return sum(np.einsum("oc,bcyx->boyx", fil[:, :, ky, kx], pad[:, :, ky:ky + h, kx:kx + w]) for ky in range(3) for kx in range(3))


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("cin,cout", [(16, 16), (24, 64), (32, 96), (64, 32), (96, 48), (40, 136), (72, 200), (16, 80)])
@pytest.mark.parametrize("batch,h,w", [(3, 16, 16), (2, 18, 30), (3, 18, 20)])
def test_channels_that_are_no_whole_blocks(dtype, cin, cout, batch, h, w):
    """Forward, image and filter gradients (fresh and accumulated) of whole numbers that every type holds: sums below 2^24 are exact
    in f32 whatever their order, so each result has the one rounding of its type."""
    dev, g = device(), rng(cin * cout + w)
    announce("conv3x3 channels", dtype, cin, cout, batch, h, w)
    img, fil, go = (g.integers(-3, 4, size=s).astype(np.float64) for s in ((batch, cin, h, w), (cout, cin, 3, 3), (batch, cout, h, w)))
    dimg, dfil, dgo = (dev.tensor(oracle.to_storage(t, dtype), dtype) for t in (img, fil, go))
    host = lambda t, shape: oracle.to_f64(dev.to_host(t), dtype).reshape(shape)
    rounded = lambda v: oracle.to_f64(oracle.to_storage(v, dtype), dtype).reshape(v.shape)
    out = dev.conv2d_forward(dimg, dfil, stride=1, padding=1)
    np.testing.assert_array_equal(host(out, go.shape), rounded(correlate(img, fil)))
    want_img = correlate(go, fil[:, :, ::-1, ::-1].transpose(1, 0, 2, 3))
    pad = np.pad(img, ((0, 0), (0, 0), (1, 1), (1, 1)))
    want_fil = np.stack([np.stack([np.einsum("boyx,bcyx->oc", go, pad[:, :, ky:ky + h, kx:kx + w]) for kx in range(3)], -1) for ky in range(3)], -2)
    gi, gf = dev.zeros_many([dimg, dfil], deferred=True)
    dev.conv2d_backward(dimg, gi, dfil, gf, dgo, stride=1, padding=1)
    first_img, first_fil = rounded(want_img), rounded(want_fil)
    np.testing.assert_array_equal(host(gi, img.shape), first_img)
    np.testing.assert_array_equal(host(gf, fil.shape), first_fil)
    dev.conv2d_backward(dimg, gi, dfil, gf, dgo, stride=1, padding=1)  # onto what is there: rounded once more
    np.testing.assert_array_equal(host(gi, img.shape), rounded(first_img + want_img))
    np.testing.assert_array_equal(host(gf, fil.shape), rounded(first_fil + want_fil))


@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_filter_gradient_where_the_filters_lie(dtype):
    """Added to the filters in place: the image gradient has been formed from them before.  Whole numbers, as above."""
    dev, g = device(), rng(61)
    announce("conv3x3, filter gradient onto the filters", dtype)
    img, fil, go = (g.integers(-3, 4, size=s).astype(np.float64) for s in ((2, 64, 16, 16), (64, 64, 3, 3), (2, 64, 16, 16)))
    dimg, dfil, dgo = (dev.tensor(oracle.to_storage(t, dtype), dtype) for t in (img, fil, go))
    apart_img, apart_fil = dev.zeros_many([dimg, dfil], deferred=True)
    dev.conv2d_backward(dimg, apart_img, dfil, apart_fil, dgo, stride=1, padding=1)
    onto_img = dev.zeros(dtype, img.shape)
    want = oracle.to_f64(dev.to_host(apart_fil), dtype) + fil.reshape(-1)
    dev.conv2d_backward(dimg, onto_img, dfil, dfil, dgo, stride=1, padding=1)
    np.testing.assert_array_equal(dev.to_host(onto_img), dev.to_host(apart_img))
    ulp = 0.0 if dtype == "f32" else 2.0 ** -11   # the sum is rounded once more beside the one that stands alone
    assert np.abs(oracle.to_f64(dev.to_host(dfil), dtype) - want).max() <= 2 * ulp * np.abs(want).max()


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("batch,cin,cout,hw,forward", [(8, 16, 64, 32, 1), (8, 24, 96, 32, 1), (8, 16, 96, 56, 2), (8, 32, 64, 32, 2), (3, 16, 64, 20, 2)])
def test_little_to_do_is_one_launch(dtype, batch, cin, cout, hw, forward):
    """Half a chunk of channels: the band kernel, behind the launch that lays the filters, only where there is enough to do."""
    announce("conv3x3, launches", dtype, batch, cin, cout, hw)

    def prepare(dev):
        img, fil = dev.zeros(dtype, (batch, cin, hw, hw)), dev.zeros(dtype, (cout, cin, 3, 3))
        return lambda: dev.conv2d_forward(img, fil, stride=1, padding=1)
    assert launches(prepare) == forward


@pytest.mark.parametrize("batch,cin,cout,hw,band", [(4, 48, 512, 32, False), (4, 128, 512, 32, False), (8, 64, 256, 14, False), (1, 16, 128, 32, False),
                                                    (2, 16, 128, 32, True), (8, 64, 256, 96, True), (64, 32, 256, 20, True)])
def test_many_output_channels_and_few_pixels(batch, cin, cout, hw, band):
    """Backward: three launches with the band kernels (shares of the filter gradient, their sums beside the filters, the image gradient);
    with the patch matrix of the image there are the patches, two products and the fold."""
    announce("conv3x3 backward, launches", batch, cin, cout, hw)

    def prepare(dev):
        img, fil, go = (dev.zeros("f16", s) for s in ((batch, cin, hw, hw), (cout, cin, 3, 3), (batch, cout, hw, hw)))
        gi, gf = (dev.zeros("f16", t.shape) for t in (img, fil))
        return lambda: dev.conv2d_backward(img, gi, fil, gf, go, stride=1, padding=1)
    assert (launches(prepare) <= 3) == band
