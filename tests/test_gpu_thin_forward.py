"""The forward projector of detectors with few rows (lane = column): every row count it takes and
the first it leaves, one and several slices, footprints over one to many cells, columns off the
volume, column counts around a wavefront, z-slab views among the others.

Tolerance 1e-4 of the peak against the oracle, as for every operator."""
import numpy as np
import pytest
import torch

import ctreconstruction_amd as ctr
from ctreconstruction_amd import _native as N
from oracle import dd_oracle as O
from tests.conftest import make_params

pytestmark = pytest.mark.gpu

TOL = 1e-4


def _check(p):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    g = O.Geometry(p)
    vol = np.random.default_rng(3).random((g.nz, g.ny, g.nx)).astype(np.float32)
    ref = O.forward_project(g, vol)
    out = ctr.dd_forward(torch.from_numpy(vol).to("cuda:0"), ctr.ScanGeometry(p)).cpu().numpy()
    assert np.abs(out - ref).max() <= TOL * np.abs(ref).max()


@pytest.mark.parametrize("nv", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("nz", [1, 2, 9])
@pytest.mark.parametrize("shape", ["Flat", "Curved"])
def test_row_counts_match_the_oracle(nv, nz, shape):
    _check(make_params(NumberOfImage=[19, 23, nz], NumberOfDetectorPixels=[70, nv], DetectorPixelSize=[0.6, 0.8],
                       NumberOfViews=9, StartAngle=0.1, EndAngle=0.1 + 2 * np.pi, DetectorShape=shape,
                       DetectorOffset=[0.0 if shape == "Curved" else 0.4, 0.2]))


# cells from a fifth of a voxel to six voxels wide; 1 to 129 columns
@pytest.mark.parametrize("nu,cell", [(1, 30.0), (63, 0.15), (64, 0.7), (65, 1.4), (129, 2.4), (12, 4.5)])
@pytest.mark.parametrize("nz", [1, 5])
def test_footprints_match_the_oracle(nu, cell, nz):
    _check(make_params(NumberOfImage=[21, 18, nz], NumberOfDetectorPixels=[nu, 2 if nz > 1 else 1],
                       DetectorPixelSize=[cell, 1.1], NumberOfViews=7, StartAngle=0.05, EndAngle=0.05 + 2 * np.pi))


def test_z_slab_views_are_left_to_their_kernel():
    _check(make_params(SourceInit=[0, 300.0, 320.0], DetectorInit=[0, -300.0, -320.0], NumberOfImage=[12, 12, 6],
                       NumberOfDetectorPixels=[20, 3], NumberOfViews=4))
