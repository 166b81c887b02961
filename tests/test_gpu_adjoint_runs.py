"""The matched adjoint of scans whose detector windows (16 bytes per view and 16 x 16 column tile) would take
more than 1 GiB goes through the views in runs: the workspace stays bounded, no size is refused for it, and the
result is the sum over the runs, for one scan, a batch and an accumulating call.

Tolerance 1e-4 of the peak, as for every operator: a voxel is the sum of 65535 terms in another order, in chains
of about 13 000, each with a rounding of 6e-8 of the sum so far."""
import ctypes

import pytest
import torch

import ctreconstruction_amd as ctr
from ctreconstruction_amd import _native as N
from ctreconstruction_amd import projector as P
from ctreconstruction_amd.autograd import adjoint_batch
from tests.conftest import make_params

TOL = 1e-4


def test_the_windows_of_a_large_slice_are_bounded():
    geom = ctr.ScanGeometry(make_params(NumberOfImage=[8192, 8192, 1], ImagePixelSpacing=[0.02] * 3, NumberOfViews=8,
                                        NumberOfDetectorPixels=[64, 1]))
    g = geom.ctypes_struct()
    g.n_views = 8192
    nbytes = N.lib().ctr_dd_backproject_workspace_bytes(ctypes.byref(g), N.BP_MODES["adjoint"])
    assert 0 < nbytes < 1.25 * (1 << 30)


@pytest.mark.gpu
def test_runs_of_views_add_up():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    views, n = 65535, 528
    assert ((n + 15) // 16) ** 2 * views > 1 << 26
    geom = ctr.ScanGeometry(make_params(NumberOfImage=[n, n, 1], NumberOfViews=views, NumberOfDetectorPixels=[16, 1],
                                        DetectorPixelSize=[26.0, 2.0]))
    gen = torch.Generator().manual_seed(0)
    y = torch.rand((2,) + tuple(geom.proj_shape), generator=gen).cuda()
    half = [list(range(0, 40000)), list(range(40000, views))]   # one run each
    ref = [sum(P.dd_adjoint(p[h].contiguous(), geom.with_views(h)).double() for h in half) for p in y]
    peak = ref[0].abs().max()
    got = P.dd_adjoint(y[0], geom)
    assert (got - ref[0]).abs().max() <= TOL * peak
    both = adjoint_batch(y, geom)
    for b in range(2):
        assert (both[b] - ref[b]).abs().max() <= TOL * peak
    base = torch.full_like(got, float(peak))
    P.dd_backproject(y[0], geom, mode="adjoint", out=base, accumulate=True)
    assert (base - peak - ref[0]).abs().max() <= 2 * TOL * peak
