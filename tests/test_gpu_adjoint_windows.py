"""The matched adjoint's LDS windows and view splits against the oracle's exact transpose, where they
can go wrong: window sizes at the edges of the work shapes and past the last one (gathered from
global memory), short z chunks, columns and rows off the detector.

Tolerance 1e-4 of the peak, as for every operator."""
import numpy as np
import pytest
import torch

import ctreconstruction_amd as ctr
from ctreconstruction_amd import _native as N
from oracle import dd_oracle as O
from tests.conftest import make_params

pytestmark = pytest.mark.gpu

TOL = 1e-4


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    return torch.device("cuda:0")


def _check(dev, p):
    g = O.Geometry(p)
    geom = ctr.ScanGeometry(p)
    y = np.random.default_rng(11).random((g.nview, g.nv, g.nu)).astype(np.float32)
    ref = O.forward_adjoint(g, y)
    out = ctr.dd_backproject(torch.from_numpy(y).to(dev), geom, mode="adjoint")
    peak = np.abs(ref).max()
    assert np.abs(out.cpu().numpy() - ref).max() <= TOL * peak
    # into a buffer that is not 16-byte aligned, scaled and added
    base = torch.full((out.numel() + 1,), 2.0 * float(peak), device=dev)
    odd = base[1:].view(geom.vol_shape)
    ctr.dd_backproject(torch.from_numpy(y).to(dev), geom, mode="adjoint", scale=-0.5, out=odd, accumulate=True)
    assert np.abs(odd.cpu().numpy() - (2.0 * peak - 0.5 * ref)).max() <= 2 * TOL * peak


# detector cells per voxel: windows well inside, at the edges of the shapes, and too large
@pytest.mark.parametrize("cells", [0.4, 1.0, 1.45, 2.1, 4.2, 9.0])
@pytest.mark.parametrize("nz", [5, 17, 40])
@pytest.mark.parametrize("shape", ["Flat", "Curved"])
def test_windows_match_the_oracle(dev, cells, nz, shape):
    cell = 0.75 / cells  # 0.5 mm voxels
    _check(dev, make_params(NumberOfImage=[18, 17, nz], NumberOfViews=5, StartAngle=0.3, EndAngle=0.3 + 2 * np.pi,
                            NumberOfDetectorPixels=[int(20 / cell), int((nz + 4) * 0.75 / cell) + 2],
                            DetectorPixelSize=[cell, cell], DetectorShape=shape))


# a single view, an odd number, and splits whose last share is one view; a detector that the volume
# overhangs in both directions; a helix; a near source
@pytest.mark.parametrize("views", [1, 5, 13, 41])
@pytest.mark.parametrize("kind", ["overhang", "helix", "near", "slice"])
def test_view_splits_match_the_oracle(dev, views, kind):
    kw = {"overhang": dict(NumberOfDetectorPixels=[17, 11]),
          "helix": dict(Pitch=0.5, EndAngle=4 * np.pi, NumberOfDetectorPixels=[40, 20]),
          "near": dict(SourceInit=[0, 60.0, 0], DetectorInit=[0, -40.0, 0], NumberOfDetectorPixels=[40, 60]),
          "slice": dict(NumberOfImage=[24, 20, 1], NumberOfDetectorPixels=[40, 1])}[kind]
    base = dict(NumberOfImage=[20, 19, 34], NumberOfViews=views, StartAngle=0.2, EndAngle=0.2 + 2 * np.pi)
    _check(dev, make_params(**{**base, **kw}))
