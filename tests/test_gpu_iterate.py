"""The one-pass residual and update kernels against the torch expressions on the CPU: the same FP32
operations in the same order with correctly rounded divisions, so the results are equal bit for bit
(a negative zero counts as zero).  Sizes on both sides of the 4-wide form and of a 1024-value block,
addresses off 16 bytes, zero weights, infinities and NaN."""
import pytest
import torch

from ctreconstruction_amd import _native as N
from ctreconstruction_amd import ScanGeometry
from ctreconstruction_amd import iterative as IT
from tests.conftest import make_params

pytestmark = pytest.mark.gpu


def _inputs(shape, batch, offset, seed=0):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    gen = torch.Generator().manual_seed(seed)
    n = torch.Size(shape).numel()
    full = batch + shape
    a, b = torch.randn(full, generator=gen), torch.randn(full, generator=gen)
    w = torch.rand(shape, generator=gen)
    w.view(-1)[::3] = 0
    for t in (a, b):
        t.view(-1)[n // 2] = float("nan")
        t.view(-1)[n // 3] = float("-inf")
        t.view(-1)[n // 4] = -0.0

    def device(t):      # a contiguous tensor `offset` floats off the allocation's alignment
        buf = torch.empty(t.numel() + 8, device="cuda")
        out = buf[offset:offset + t.numel()].view(t.shape)
        return out.copy_(t)
    return (a, b, w), tuple(device(t) for t in (a, b, w))


SHAPES = [((1, 1, 1), ()), ((1, 1, 4), ()), ((3, 5, 7), ()), ((2, 16, 32), (3,)), ((4, 16, 16), ()), ((5, 11, 20), (2,)),
          ((3, 7, 9), (2, 2))]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape,batch", SHAPES)
def test_residual_equals_the_expressions(shape, batch, offset):
    cpu, gpu = _inputs(shape, batch, offset)
    for weighted in (True, False):
        ref, got = IT._residual(*cpu, weighted, 1e-6), IT._residual(*gpu, weighted, 1e-6)
        assert IT._elementwise(*gpu) and got.shape == ref.shape
        assert torch.equal(got.cpu().nan_to_num(nan=7e30), ref.nan_to_num(nan=7e30))


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape,batch", SHAPES)
def test_update_equals_the_expressions(shape, batch, offset):
    cpu, gpu = _inputs(shape, batch, offset, 1)
    for masked in (True, False):
        for nonneg in (True, False):
            ref = IT._update(*cpu, -0.5, 1e-6, masked, nonneg)
            got = IT._update(*gpu, -0.5, 1e-6, masked, nonneg)
            assert torch.equal(got.cpu().nan_to_num(nan=7e30), ref.nan_to_num(nan=7e30))


def test_other_forms_keep_the_expressions():
    (a, b, w), (ga, gb, gw) = _inputs((4, 6, 8), (), 0)
    batch = torch.stack([a, b])
    for x, y in ((batch, b), (a.double(), b)):
        ref, got = IT._residual(x, y, w, True), IT._residual(x.cuda(), y.cuda(), gw, True)
        assert got.dtype == ref.dtype and torch.equal(got.cpu().nan_to_num(nan=7e30), ref.nan_to_num(nan=7e30))
    assert not IT._elementwise(ga.transpose(0, 1), gb.transpose(0, 1), gw.transpose(0, 1).contiguous())
    assert not IT._elementwise(ga, gb, gw, torch.tensor(0.5))
    assert not IT._elementwise(ga.requires_grad_(True), gb, gw)


def test_one_volume_for_a_batch_of_projections():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    geom = ScanGeometry(make_params(NumberOfImage=[16, 16, 8], NumberOfViews=6, NumberOfDetectorPixels=[32, 24]))
    gen = torch.Generator().manual_seed(2)
    p, x0 = torch.rand(geom.proj_shape, generator=gen).cuda(), torch.rand(geom.vol_shape, generator=gen).cuda()
    # the data term of two equal scans has twice the gradient of one: doubling is exact in FP32
    two = IT.sart(torch.stack([p, p]), geom, 1, relaxation=0.25, x0=x0)
    one = IT.sart(p, geom, 1, relaxation=0.5, x0=x0)
    assert two.shape == one.shape and torch.allclose(two, one, rtol=0, atol=1e-6)
