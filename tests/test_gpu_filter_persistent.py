"""Every row of the launches that run as persistent workgroups (2048 and 4096 points, from four rounds of the
resident workgroups on) against the float64 oracle: both halves of each length, an odd last row, the first row
count that is persistent, a whole number of rounds, rows of several views, in place, and the mirrored rows of the
pixel-driven filter.  The output starts as NaN, so that a row left out shows.

Tolerance 1e-4 of the peak against float64, as for every operator; the rows are random, so another row's values
are off by the peak itself."""
import numpy as np
import pytest
import torch

import ctreconstruction_amd as ctr
from ctreconstruction_amd import _native as N
from ctreconstruction_amd import pixel_fdk as PF
from oracle import dd_oracle as O
from oracle import pixel_oracle as PO
from tests.conftest import make_cone_params, make_params

pytestmark = pytest.mark.gpu

TOL = 1e-4


def _rows(shape, seed):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    return np.random.default_rng(seed).random(shape).astype(np.float32)


# resident: 1024 workgroups of two rows at 2048 points, 512 at 4096
@pytest.mark.parametrize("nu,views,nv", [(1000, 1, 8301), (1024, 3, 2801), (514, 1, 8191), (1025, 1, 8193), (1025, 2, 5120),
                                         (1500, 1, 4203), (2048, 1, 4096), (2049, 1, 4095), (2049, 3, 1501)])
def test_every_row_matches_the_oracle(nu, views, nv):
    x = _rows((views, nv, nu), nu + nv)
    p = make_params(NumberOfDetectorPixels=[nu, nv], NumberOfViews=views, FilterType="shepp-logan")
    geom = ctr.ScanGeometry(p)
    ref = O.filter_projections(O.Geometry(p), x)
    xd = torch.from_numpy(x).cuda()
    out = ctr.fdk_filter(xd, geom, out=torch.full_like(xd, float("nan")))
    assert np.abs(out.cpu().numpy() - ref).max() <= TOL * np.abs(ref).max()
    assert torch.equal(ctr.fdk_filter(xd, geom, out=xd), out)


@pytest.mark.parametrize("nu,views,nv", [(1000, 3, 2801), (2049, 2, 2101)])
def test_every_mirrored_row_matches_the_oracle(nu, views, nv):
    x = _rows((views, nv, nu), nu)
    prm = make_cone_params(DetectorWidth=nu, DetectorHeight=nv, NumberOfViews=views)
    ref = PO.filter_projections(PO.PixelGeometry(prm), x)
    xd = torch.from_numpy(x).cuda()
    out = PF.pixel_filter(xd, PF.PixelScan(prm), out=torch.full_like(xd, float("nan"))).cpu().numpy()
    assert np.abs(out - ref).max() <= TOL * np.abs(ref).max()
