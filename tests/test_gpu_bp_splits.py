"""The FDK backprojection's view splits: small volumes share their views out to several workgroups
per tile, whose partial volumes a second kernel adds up.

Tolerance 1e-4 of the peak against the oracle, as for every operator (the splits only change the
order of FP32 sums of at most a few hundred terms: under 1e-6 of the peak on top)."""
import ctypes

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


# (image, views): one split, the first with two, a last split of one view, sizes that the reduction
# reads one float at a time (17 * 19 * 9 is odd) and a slice (the single pass)
@pytest.mark.parametrize("image,views", [([16, 16, 40], 7), ([16, 16, 40], 8), ([17, 19, 9], 37),
                                         ([33, 18, 34], 50), ([20, 24, 1], 61)])
@pytest.mark.parametrize("mode,zero_tol", [("ref", 0.0), ("edge", 0.0), ("ref", 1e-5)])
def test_split_views_match_the_oracle(dev, image, views, mode, zero_tol):
    det = [44, 1] if image[2] == 1 else [44, 46]
    p = make_params(NumberOfImage=image, NumberOfDetectorPixels=det, NumberOfViews=views, StartAngle=0.1,
                    EndAngle=0.1 + 2 * np.pi)
    g = O.Geometry(p)
    geom = ctr.ScanGeometry(p)
    q = np.random.default_rng(views).random((g.nview, g.nv, g.nu)).astype(np.float32)
    ref = O.backproject(g, q, mode, zero_tol=zero_tol if zero_tol > 0 else None)
    qd = torch.from_numpy(q).to(dev)
    out = ctr.dd_backproject(qd, geom, mode=mode, zero_tol=zero_tol)
    peak = np.abs(ref).max()
    assert np.abs(out.cpu().numpy() - ref).max() <= TOL * peak
    # added to a volume, and into a buffer that is not 16-byte aligned: the same sums
    base = torch.full((out.numel() + 1,), 0.5 * float(peak), device=dev)
    odd = base[1:].view(geom.vol_shape)
    ctr.dd_backproject(qd, geom, mode=mode, zero_tol=zero_tol, out=odd, accumulate=True)
    assert float(base[0]) == np.float32(0.5 * peak)
    assert np.abs(odd.cpu().numpy() - (ref + 0.5 * peak)).max() <= 2 * TOL * peak


def test_workspace_covers_the_splits(dev):
    """The query counts the partial volumes, and a workspace one byte short is refused."""
    geom = ctr.ScanGeometry(make_params(NumberOfViews=64))
    g = geom.ctypes_struct()
    lib = N.lib()
    need = lib.ctr_dd_backproject_workspace_bytes(ctypes.byref(g), 0)
    assert need >= 64 * 64 + 16 * geom.nx * geom.ny * geom.nz * 4
    dummy = ctypes.c_void_p(16)  # never dereferenced: the size check fails first
    assert lib.ctr_dd_backproject(ctypes.byref(g), dummy, dummy, dummy, dummy, 0, 1.0, 0.0, 0, dummy, need - 1,
                                  None) == N.CTR_ERR_WORKSPACE


def _check(dev, p, mode="ref", tol=TOL):
    g = O.Geometry(p)
    geom = ctr.ScanGeometry(p)
    q = np.random.default_rng(5).random((g.nview, g.nv, g.nu)).astype(np.float32)
    ref = O.backproject(g, q, mode)
    qd = torch.from_numpy(q).to(dev)
    peak = np.abs(ref).max()
    two = ctr.dd_backproject(qd, geom, mode=mode).cpu().numpy()
    one = ctr.dd_backproject(qd, geom, mode=mode, zero_tol=-1.0).cpu().numpy()
    assert np.abs(two - ref).max() <= tol * peak
    assert np.abs(one - ref).max() <= tol * peak


# detector cells per voxel (at the magnification of 1.5): below, at and above the edges of the work
# shapes (about 1, 1.4, 2 and 4), and beyond the last one (gathers from global memory)
@pytest.mark.parametrize("cells", [0.5, 0.95, 1.05, 1.12, 1.35, 1.45, 1.95, 2.1, 3.9, 4.3, 7.0])
@pytest.mark.parametrize("nz", [7, 17, 40])
def test_every_work_shape_matches_the_oracle(dev, cells, nz):
    cell = 0.75 / cells  # 0.5 mm voxels
    _check(dev, make_params(NumberOfImage=[18, 17, nz], NumberOfViews=5, StartAngle=0.3, EndAngle=0.3 + 2 * np.pi,
                            NumberOfDetectorPixels=[int(30 / cell), int((nz + 4) * 0.75 / cell) + 2],
                            DetectorPixelSize=[cell, cell]))


# sub-chunks that straddle the source height (at voxel centres and edges, and moving along a helix),
# that the detector cuts, and that hold fewer voxels than their shape's; coarse voxels (no series)
@pytest.mark.parametrize("nz", [1, 2, 15, 16, 24, 25, 31, 33, 48])
@pytest.mark.parametrize("kind", ["centred", "shifted", "helix", "cut", "coarse_curved"])
def test_ragged_and_straddling_sub_chunks_match_the_oracle(dev, nz, kind):
    kw = {"centred": {}, "shifted": dict(ReconCenter=[0.4, -0.3, 0.25 * nz + 0.13]),
          "helix": dict(Pitch=0.4, EndAngle=4 * np.pi, NumberOfViews=9),
          "cut": dict(NumberOfDetectorPixels=[22, 12]),
          "coarse_curved": dict(ImagePixelSpacing=[3.0, 3.0, 3.0], DetectorPixelSize=[5.0, 5.0],
                                DetectorShape="Curved", NumberOfDetectorPixels=[40, 30])}[kind]
    base = dict(NumberOfImage=[19, 18, nz], NumberOfViews=5, NumberOfDetectorPixels=[26, 44], StartAngle=0.2,
                EndAngle=0.2 + 2 * np.pi)
    _check(dev, make_params(**{**base, **kw}), "edge" if kind == "cut" else "ref")


# a single slice has a kernel of its own: one and several detector rows, cells from a fifth of a
# pixel to three pixels wide, slices off the source height, both grids, weight zeroing
@pytest.mark.parametrize("nv,cell", [(1, 0.15), (1, 0.7), (3, 0.5), (7, 0.1), (2, 2.0)])
@pytest.mark.parametrize("shape", ["Flat", "Curved"])
@pytest.mark.parametrize("zc", [0.0, 0.3])
def test_single_slice_matches_the_oracle(dev, nv, cell, shape, zc):
    p = make_params(NumberOfImage=[21, 34, 1], ReconCenter=[0.2, -0.1, zc], NumberOfViews=23, StartAngle=0.1,
                    EndAngle=0.1 + 2 * np.pi, NumberOfDetectorPixels=[int(24 / cell), nv],
                    DetectorPixelSize=[cell, 0.6], DetectorShape=shape)
    for mode in ("ref", "edge"):
        _check(dev, p, mode)
    g = O.Geometry(p)
    q = np.random.default_rng(8).random((g.nview, g.nv, g.nu)).astype(np.float32)
    ref = O.backproject(g, q, "ref", zero_tol=1e-5)
    out = ctr.dd_backproject(torch.from_numpy(q).to(dev), ctr.ScanGeometry(p), zero_tol=1e-5).cpu().numpy()
    assert np.abs(out - ref).max() <= TOL * np.abs(ref).max()


# the pixel-driven backprojection's view splits: one split, two, a last split of one view; volumes
# whose size the reduction reads one float at a time; a buffer that is not 16-byte aligned, added to.
# Voxels whose sample lies within 2e-3 cells of the detector's edge in a view are left out, as in the
# other tests of this operator (either side of the reference's bounds test is right for them).
@pytest.mark.parametrize("views,size", [(4, (24, 24, 24)), (8, (24, 24, 24)), (37, (17, 19, 9)), (33, (20, 18, 40))])
def test_pixel_view_splits_match_the_oracle(dev, views, size):
    from ctreconstruction_amd import pixel_fdk as PF
    from oracle import pixel_oracle as PO
    from tests.conftest import make_cone_params
    prm = make_cone_params(NumberOfViews=views, ReconX=size[0], ReconY=size[1], ReconZ=size[2])
    g = PO.PixelGeometry(prm)
    q = np.random.default_rng(views).random((views, g.nv, g.nu)).astype(np.float32)
    ref = PO.backproject(g, q)
    keep = PO.edge_margin(g) > 2e-3
    peak = np.abs(ref).max()
    scan = PF.PixelScan(prm)
    qd = torch.from_numpy(q).to(dev)
    out = PF.pixel_backproject(qd, scan).cpu().numpy()
    assert np.abs(out - ref)[keep].max() <= TOL * peak
    base = torch.full((out.size + 1,), 0.5 * float(peak), device=dev)
    odd = base[1:].view(scan.vol_shape)
    PF.pixel_backproject(qd, scan, out=odd, accumulate=True)
    assert np.abs(odd.cpu().numpy() - (ref + 0.5 * peak))[keep].max() <= 2 * TOL * peak


# the pixel-driven backprojection with and without the per-sample row test: detectors that see all of
# the volume, cut it at both ends, and miss most of it, with both z extents of a work-item
@pytest.mark.parametrize("nv", [6, 20, 40, 120])
@pytest.mark.parametrize("nz,pitch", [(33, 0.8), (70, 0.8), (40, 0.2)])
def test_pixel_row_test_matches_the_oracle(dev, nv, nz, pitch):
    from ctreconstruction_amd import pixel_fdk as PF
    from oracle import pixel_oracle as PO
    from tests.conftest import make_cone_params
    prm = make_cone_params(NumberOfViews=7, ReconX=18, ReconY=17, ReconZ=nz, DetectorHeight=nv, DetectorPixelHeight=pitch)
    g = PO.PixelGeometry(prm)
    q = np.random.default_rng(nv).random((7, g.nv, g.nu)).astype(np.float32)
    ref = PO.backproject(g, q)
    keep = PO.edge_margin(g) > 2e-3
    out = PF.pixel_backproject(torch.from_numpy(q).to(dev), PF.PixelScan(prm)).cpu().numpy()
    assert np.abs(out - ref)[keep].max() <= TOL * np.abs(ref).max()
