"""Values of the total-variation eps that are not positive normal float32 numbers: Python's go to the torch
expressions, the C entries refuse them."""
import ctypes

import pytest
import torch

from ctreconstruction_amd import _native as N
from ctreconstruction_amd import iterative as IT


@pytest.mark.parametrize("eps", [1e-40, 1e-45, 1e-50, 0.0, -1e-7])
def test_the_c_entries_refuse_an_eps_below_the_normal_floats(eps):
    lib = N.lib()
    buf = ctypes.create_string_buffer(1 << 16)   # never read: the arguments are refused first
    at = lambda k: ctypes.c_void_p(ctypes.addressof(buf) + k)  # noqa: E731
    nbytes = lib.ctr_tv_workspace_bytes(1, 4, 4, 4, 2)
    assert 0 < nbytes <= 1 << 14
    assert lib.ctr_tv_gradient(at(0), at(1 << 12), 1, 4, 4, 4, eps, at(1 << 14), nbytes, None) == N.CTR_ERR_INVALID
    assert lib.ctr_tv_descent(at(0), at(1 << 12), at(1 << 13), 1, 4, 4, 4, eps, 2, at(1 << 14), nbytes,
                              None) == N.CTR_ERR_INVALID


@pytest.mark.gpu
@pytest.mark.parametrize("eps", [1e-40, 1e-45, 1e-50])
def test_tiny_eps_is_computed_by_torch(eps):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    x = torch.rand((2, 6, 7, 9), generator=torch.Generator().manual_seed(0)).cuda()
    x[:, :, :, :4] = 0.25   # flat: |D| is sqrt(eps) there
    step = torch.full((2, 1, 1, 1), 0.1, device="cuda")
    ref = IT._normalise_pad(IT._tv_terms(x, eps), eps)
    assert torch.isfinite(ref).all() == (eps >= 1e-45)   # at eps = 0 a flat voxel is 0 / 0
    assert not IT._on_tv_kernels(x, eps) and IT._on_tv_kernels(x, 1e-37)
    assert torch.equal(IT.tv_gradient(x, eps).nan_to_num(nan=7.0), ref.nan_to_num(nan=7.0))
    assert torch.equal(IT._tv_descent(x, step, 1, eps).nan_to_num(nan=7.0), (x - step * ref).nan_to_num(nan=7.0))


@pytest.mark.gpu
def test_an_eps_tensor_is_differentiable_and_goes_to_torch():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    x = torch.rand((6, 7, 9), generator=torch.Generator().manual_seed(1)).cuda()
    eps = torch.tensor(1e-3, device="cuda", requires_grad=True)
    y = IT.tv_gradient(x, eps)
    (g,) = torch.autograd.grad(y.square().mean() + y.abs().mean(), eps)
    assert torch.isfinite(g)
