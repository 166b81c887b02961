"""The convolution's weight and bias gradients where the tiling can go wrong: images around the
8 x 32 pixel tile, channel counts around the 16-channel blocks (vectorised and element loads, the
row-split kernel for at most 16 input channels), more tiles than workgroups, a bias left out.

The operands are exact in bfloat16 and the sums are FP32: with P pixels the error of a sum of P
products is at most P ulp and about sqrt(P) ulp of the sum of magnitudes, so 1e-5 of the largest
gradient (as for the other shapes) leaves room at these sizes."""
import pytest
import torch

from ctreconstruction_amd import _native as N
from ctreconstruction_amd import prior as PR

pytestmark = pytest.mark.gpu


def _reference(x, g):
    n, h, w, cin = x.shape
    pad = torch.nn.functional.pad(x.double(), (0, 0, 1, 1, 1, 1))
    go = g.double().reshape(-1, g.shape[-1])
    gw = torch.stack([torch.stack([go.t() @ pad[:, a:a + h, b:b + w].reshape(-1, cin) for b in range(3)], 1)
                      for a in range(3)], 1)
    return gw, go.sum(0)


@pytest.mark.parametrize("n,h,w", [(1, 1, 1), (2, 7, 31), (1, 8, 32), (3, 9, 33), (1, 16, 64), (5, 30, 45), (40, 33, 97)])
@pytest.mark.parametrize("cin,cout", [(64, 64), (3, 64), (64, 1), (16, 16), (17, 33), (48, 24), (1, 1)])
def test_weight_gradient_tiles_match_float64(n, h, w, cin, cout):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    gen = torch.Generator().manual_seed(n * h + w + cin)
    x = torch.randn((n, h, w, cin), generator=gen).to(torch.bfloat16)
    g = torch.randn((n, h, w, cout), generator=gen).to(torch.bfloat16)
    rw, rb = _reference(x, g)
    gw, gb = PR.conv3x3_wgrad(x.cuda(), g.cuda())
    assert (gw.cpu().double() - rw).abs().max() <= 1e-5 * rw.abs().max().clamp_min(1.0)
    assert (gb.cpu().double() - rb).abs().max() <= 1e-5 * rb.abs().max().clamp_min(1.0)
    gw2, none = PR.conv3x3_wgrad(x.cuda(), g.cuda(), with_bias=False)
    assert none is None and torch.equal(gw2, gw)


@pytest.mark.parametrize("cin,cout", [(64, 64), (3, 64), (64, 1), (17, 33)])
def test_combined_backward_equals_its_parts(cin, cout):
    """The same kernels on the same operands: bit-identical; the input gradient may be left out."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    gen = torch.Generator().manual_seed(cin)
    x = torch.randn((2, 19, 37, cin), generator=gen).to(torch.bfloat16).cuda()
    g = torch.randn((2, 19, 37, cout), generator=gen).to(torch.bfloat16).cuda()
    w = torch.randn((cout, 3, 3, cin), generator=gen).to(torch.bfloat16).cuda()
    gx, gw, gb = PR.conv3x3_backward(x, w, g)
    assert torch.equal(gx, PR.conv3x3_forward(g, PR.flip_transpose(w)))
    rw, rb = PR.conv3x3_wgrad(x, g)
    assert torch.equal(gw, rw) and torch.equal(gb, rb)
    none, gw, gb = PR.conv3x3_backward(x, w, g, input_grad=False)
    assert none is None and torch.equal(gw, rw) and torch.equal(gb, rb)
