"""Which calls the total-variation, residual and update kernels take: anything that watches torch's work on a
tensor keeps the torch expressions, a default device does not, and so does a torch that cannot tell."""
import pytest
import torch
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

import ctreconstruction_amd as ctr
from ctreconstruction_amd import _native as N
from ctreconstruction_amd import iterative as IT
from tests.conftest import make_params

PRIVATE = [(torch.overrides, "_get_current_function_mode_stack"), (torch.utils._python_dispatch, "_get_current_dispatch_mode"),
           (torch._C._functorch, "is_functorch_wrapped_tensor")]


class FunctionMode(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class DispatchMode(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_what_counts_as_observed():
    x = torch.zeros(3)
    assert not IT._observed(x)
    with torch.device("cpu"):
        assert not IT._observed(x)
        with FunctionMode():
            assert IT._observed(x)
    for mode in (FunctionMode(), DispatchMode()):
        with mode:
            assert IT._observed(x)
    seen = []
    torch.func.vmap(lambda t: (seen.append(IT._observed(t)), t)[1])(torch.zeros(2, 3))
    with forward_ad.dual_level():
        seen.append(IT._observed(forward_ad.make_dual(x, torch.ones(3))))
        assert not IT._observed(x)
    torch.jit.trace(lambda t: (seen.append(IT._observed(t)), t + 1)[1], (x,), check_trace=False)
    assert seen == [True, True, True]
    assert not IT._observed(x)


@pytest.mark.parametrize("owner,name", PRIVATE, ids=[n for _, n in PRIVATE])
def test_a_torch_without_a_private_name_keeps_the_expressions(owner, name, monkeypatch):
    x = torch.zeros(3)
    monkeypatch.delattr(owner, name)
    assert IT._observed(x)


def _scan():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    geom = ctr.ScanGeometry(make_params(NumberOfImage=[24, 20, 16], NumberOfViews=10, NumberOfDetectorPixels=[40, 30]))
    return geom, torch.rand(geom.proj_shape, generator=torch.Generator().manual_seed(0)).cuda()


@pytest.mark.gpu
def test_a_default_device_keeps_the_kernels(monkeypatch):
    geom, proj = _scan()
    x0 = torch.zeros(geom.vol_shape, device="cuda")
    ref = IT.asd_pocs(proj, geom, n_outer=1, na=1, ng=3, x0=x0)
    calls, plain = [], IT._plain
    monkeypatch.setattr(IT, "_plain", lambda *t: calls.append(plain(*t)) or calls[-1])
    torch.set_default_device("cuda")
    try:
        got = IT.asd_pocs(proj, geom, n_outer=1, na=1, ng=3, x0=x0)
    finally:
        torch.set_default_device(None)
    assert calls and all(calls) and torch.equal(got, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("owner,name", PRIVATE, ids=[n for _, n in PRIVATE])
def test_iterations_run_without_a_private_name(owner, name, monkeypatch):
    geom, proj = _scan()
    x0 = torch.zeros(geom.vol_shape, device="cuda")
    ref = IT.sart(proj, geom, 2, nonneg=True), IT.asd_pocs(proj, geom, n_outer=1, na=1, ng=3, x0=x0)
    monkeypatch.delattr(owner, name)
    got = IT.sart(proj, geom, 2, nonneg=True), IT.asd_pocs(proj, geom, n_outer=1, na=1, ng=3, x0=x0)
    monkeypatch.undo()
    # the elementwise kernels equal the expressions bit for bit; the TV steps to float32 rounding
    assert torch.equal(got[0], ref[0])
    assert (got[1] - ref[1]).norm() <= 1e-5 * ref[1].norm()
