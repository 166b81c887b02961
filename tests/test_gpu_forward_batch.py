"""A batch of volumes projected by one launch equals the volumes projected one by one: the same
sums per volume, except that slabs may be shared out differently (FP64 partial sums in another order,
below an FP32 rounding or two of the result; 1e-6 of the peak bounds them).  Detectors of a few rows
and of several row blocks, odd column counts, a view of z slabs, batches over several launches."""
import numpy as np
import pytest
import torch

import ctreconstruction_amd as ctr
from ctreconstruction_amd import _native as N
from ctreconstruction_amd import projector as P
from ctreconstruction_amd.autograd import adjoint_batch, forward_batch
from tests.conftest import make_params

pytestmark = pytest.mark.gpu


def _case(n, det, views, batch, **kw):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    p = make_params(NumberOfImage=n, NumberOfDetectorPixels=det, NumberOfViews=views, StartAngle=0.1,
                    EndAngle=0.1 + 2 * np.pi, **kw)
    geom = ctr.ScanGeometry(p)
    gen = torch.Generator().manual_seed(3)
    return geom, torch.rand((batch,) + tuple(geom.vol_shape), generator=gen).cuda()


@pytest.mark.parametrize("n,det,views,batch", [
    ([9, 10, 7], [14, 1], 5, 3), ([9, 10, 1], [15, 3], 4, 2), ([9, 10, 7], [14, 5], 5, 1), ([20, 17, 33], [37, 70], 7, 5),
    ([64, 64, 20], [80, 130], 24, 4)])
def test_batch_equals_single_volumes(n, det, views, batch):
    geom, vols = _case(n, det, views, batch)
    got = forward_batch(vols, geom)
    for b in range(batch):
        ref = ctr.dd_forward(vols[b], geom)
        assert (got[b] - ref).abs().max() <= 1e-6 * ref.abs().max()


def test_z_slab_views():
    geom, vols = _case([12, 12, 6], [16, 12], 3, 3, SourceInit=[0, 300.0, 320.0], DetectorInit=[0, -300.0, -320.0])
    got = forward_batch(vols, geom)
    for b in range(3):
        assert torch.equal(got[b], ctr.dd_forward(vols[b], geom))


def test_several_launches(monkeypatch):
    geom, vols = _case([9, 10, 7], [14, 70], 5, 5)
    whole = forward_batch(vols, geom)
    monkeypatch.setattr(P, "_FORWARD_TABLES", 0)
    assert (forward_batch(vols, geom) - whole).abs().max() <= 1e-6 * whole.abs().max()
    assert forward_batch(vols[:0], geom).shape == (0,) + tuple(geom.proj_shape)


@pytest.mark.parametrize("n,det,views,batch", [([9, 10, 1], [15, 3], 4, 2), ([20, 17, 33], [37, 70], 9, 5),
                                               ([64, 64, 20], [80, 130], 24, 4)])
def test_adjoint_batch_equals_single_scans(n, det, views, batch, monkeypatch):
    """The view splits differ with the batch: FP32 sums of at most `views` terms in another order."""
    geom, _ = _case(n, det, views, 1)
    proj = torch.rand((batch,) + tuple(geom.proj_shape), generator=torch.Generator().manual_seed(4)).cuda()
    got = adjoint_batch(proj, geom)
    for b in range(batch):
        ref = P.dd_adjoint(proj[b], geom)
        assert (got[b] - ref).abs().max() <= 2e-6 * ref.abs().max()
    monkeypatch.setattr(P, "_ADJOINT_TABLES", 4 * 2 * proj[0].numel())      # two scans to a launch
    assert (adjoint_batch(proj, geom) - got).abs().max() <= 2e-6 * got.abs().max()
    assert adjoint_batch(proj[:0], geom).shape == (0,) + tuple(geom.vol_shape)
