"""Infinite activations in the last row and column of images that end inside an 8 x 32 tile: they reach the
weight gradient through the taps that see them and through no other (the tile's pixels past the image have a
zero output gradient, and zero times infinity is not zero).  Values that stay finite are compared with float64
at the 1e-5 of the weight gradient's other tests."""
import pytest
import torch

from ctreconstruction_amd import _native as N
from ctreconstruction_amd import prior as PR
from tests.test_gpu_wgrad import _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w", [(1, 1), (7, 31), (9, 33), (8, 40), (12, 32), (17, 64), (30, 45), (33, 95)])
@pytest.mark.parametrize("cin,cout", [(64, 64), (3, 64), (17, 33)])
def test_infinities_at_the_image_edge_stay_in_their_taps(h, w, cin, cout):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    gen = torch.Generator().manual_seed(h * w + cin)
    x = torch.randn((2, h, w, cin), generator=gen).to(torch.bfloat16)
    g = torch.randn((2, h, w, cout), generator=gen).to(torch.bfloat16)
    x[0, h - 1, w // 2, 0] = float("inf")
    x[1, h // 2, w - 1, 1] = float("inf")
    rw, rb = _reference(x, g)
    gw, gb = PR.conv3x3_wgrad(x.cuda(), g.cuda())
    gw, gb = gw.cpu().double(), gb.cpu().double()
    # at most the taps that read a pixel of the last row (ky = 1, 2) or column (kx = 1, 2)
    finite = torch.isfinite(rw)
    assert finite[:, 0, :, 0].all() and finite[:, :, 0, 1].all()
    assert torch.equal(torch.isfinite(gw), finite)
    assert (gw - rw)[finite].abs().max() <= 1e-5 * rw[finite].abs().max().clamp_min(1.0)
    assert (gb - rb).abs().max() <= 1e-5 * rb.abs().max().clamp_min(1.0)
