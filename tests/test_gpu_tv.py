"""The total-variation kernels against the torch expressions they stand in for, evaluated in float64,
where the tiling can go wrong: axes from the smallest (3) over the 64 x 4 x 16 tile's edges, batches,
flat volumes (norm below eps), one and several steps.

The kernels and the float64 reference start from the same float32 volume.  A difference of two
neighbours is exact to an ulp of the difference's operands (values up to 1: 6e-8), |D| >= sqrt(eps),
so each of the gradient's terms is good to about 4 * 6e-8 / sqrt(1e-7) = 8e-4 of its bound 1 in the
worst voxel; relative to the gradient's norm, which sums thousands of such terms, 2e-5 bounds the
2-norm of the error.  A step of size s adds s times that."""
import pytest
import torch

from ctreconstruction_amd import _native as N
from ctreconstruction_amd import iterative as IT

pytestmark = pytest.mark.gpu


def _volume(shape, seed=0):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    gen = torch.Generator().manual_seed(seed)
    return torch.rand(shape, generator=gen).cuda()


def _exact(x, eps=1e-7):
    return IT._normalise_pad(IT._tv_terms(x.double(), eps), eps)


@pytest.mark.parametrize("shape", [(3, 3, 3), (4, 5, 6), (16, 4, 64), (17, 5, 65), (18, 9, 66), (33, 31, 130), (2, 20, 7, 70),
                                   (2, 3, 5, 6, 9)])
def test_gradient_matches_float64(shape):
    x = _volume(shape)
    got, ref = IT.tv_gradient(x), _exact(x)
    assert got.shape == x.shape
    assert (got.double() - ref).norm() <= 2e-5 * ref.norm()
    border = got.clone()
    border[..., 1:-1, 1:-1, 1:-1] = 0
    assert torch.count_nonzero(border) == 0


@pytest.mark.parametrize("steps", [1, 2, 5])
@pytest.mark.parametrize("shape", [(5, 6, 7), (3, 17, 20, 65)])
def test_descent_matches_float64(shape, steps):
    x = _volume(shape, 1)
    step = torch.linspace(0.1, 0.3, x[..., 0, 0, 0].numel()).cuda().reshape(x.shape[:-3] + (1, 1, 1))
    ref = x.double()
    for _ in range(steps):
        ref = ref - step.double() * _exact(ref)
    before = x.clone()
    got = IT._tv_descent(x, step, steps, 1e-7)
    assert torch.equal(x, before)  # the input is left alone
    moved = (ref - x.double()).norm()
    assert (got.double() - ref).norm() <= 1e-4 * moved + 1e-7 * x.double().norm()


def test_flat_volume_has_no_gradient():
    x = _volume((2, 8, 8, 8)).mul_(0).add_(0.3)
    assert torch.count_nonzero(IT.tv_gradient(x)) == 0
    assert torch.equal(IT._tv_descent(x, torch.ones(2, 1, 1, 1, device="cuda"), 3, 1e-7), x)


def test_what_the_kernels_do_not_take_goes_to_torch():
    x = _volume((6, 7, 8))
    ref = _exact(x)
    for y in (x.double(), x.cpu(), x.permute(2, 0, 1).contiguous().permute(1, 2, 0), x.clone().requires_grad_(True)):
        assert not IT._on_tv_kernels(y, 1e-7)
        assert (IT.tv_gradient(y).detach().double().to(ref.device) - ref).norm() <= 2e-5 * ref.norm()
    mapped = torch.func.vmap(IT.tv_gradient)(x[None])
    assert (mapped[0].double() - ref).norm() <= 2e-5 * ref.norm()
    _, tangent = torch.func.jvp(IT.tv_gradient, (x,), (torch.ones_like(x),))
    assert tangent.abs().max() <= 1e-3  # a constant shift changes nothing
