"""Scans whose preparation takes more workgroups than a launch's x extent holds (2^32 - 1 threads, 16777215
workgroups of 256): a slice of over 23 000^2 voxels, a single row of over 8000 columns at 65535 views.  The part
that the last workgroups prepare is compared with the same part as a small scan of its own."""
import ctypes

import pytest
import torch

import ctreconstruction_amd as ctr
from ctreconstruction_amd import _native as N
from ctreconstruction_amd import projector as P
from tests.conftest import make_params


def _gpu(gigabytes):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    if torch.cuda.mem_get_info()[0] < gigabytes << 30:
        pytest.skip("not enough free GPU memory")


@pytest.mark.gpu
def test_forward_projection_of_a_very_large_slice():
    _gpu(40)
    n, m, d = 23200, 96, 0.01
    assert (n + 31) // 32 * n > (2 ** 32 - 1) // 256
    half = 0.5 * (n - 1) * d
    corner = [half - 0.5 * (m - 1) * d, -half + 0.5 * (m - 1) * d]   # centre of the last columns and rows
    u = 1500.0 * corner[0] / (1000.0 - corner[1])                    # where the source at (0, 1000) projects it
    det = dict(NumberOfDetectorPixels=[64, 1], DetectorPixelSize=[0.05, 0.05], DetectorOffset=[u, 0], NumberOfViews=1,
               ImagePixelSpacing=[d, d, d])
    big = ctr.ScanGeometry(make_params(NumberOfImage=[n, n, 1], **det))
    small = ctr.ScanGeometry(make_params(NumberOfImage=[m, m, 1], ReconCenter=[*corner, 0.0], **det))
    block = torch.rand((1, m, m), generator=torch.Generator().manual_seed(0)).cuda()
    vol = torch.zeros((1, n, n), device="cuda")
    vol[:, n - m:, n - m:] = block
    got, ref = ctr.dd_forward(vol, big), ctr.dd_forward(block, small)
    # the block is seen: mean 1/2 over m voxels, the slice filling d of a row's 0.05 mm times 1116 / 1500
    assert ref.max() > 0.5 * (0.5 * m * d) * d / (0.05 * (1000.0 - corner[1]) / 1500.0)
    # index coordinates near 23200 round to 0.002 voxel, footprints are 3.7 voxels wide: below 2 * 0.002 / 3.7 of a
    # voxel's share per slab and edge, 1e-2 with room
    assert (got - ref).abs().max() <= 1e-2 * ref.max()


@pytest.mark.gpu
def test_adjoint_of_very_many_detector_columns():
    _gpu(40)
    views, nu = 65535, 8193
    assert (nu + 31) // 32 * views > (2 ** 32 - 1) // 256
    geom = ctr.ScanGeometry(make_params(NumberOfImage=[16, 16, 1], NumberOfDetectorPixels=[nu, 1], NumberOfViews=views,
                                        DetectorPixelSize=[0.4, 0.4], DetectorOffset=[-(nu / 2 - 30) * 0.4, 0]))
    y = torch.zeros(geom.proj_shape, device="cuda")
    last = list(range(views - 3, views))
    y[last, :, nu - 64:] = torch.rand((3, 1, 64), generator=torch.Generator().manual_seed(1)).cuda()
    ref = P.dd_adjoint(y[last].contiguous(), geom.with_views(last))
    got = P.dd_adjoint(y, geom)
    assert ref.abs().max() > 0.1
    assert (got - ref).abs().max() <= 1e-6 * ref.abs().max()   # the other views add zeros


def test_work_shapes_stay_inside_a_launch():
    """One voxel across: 16-fold padding of the tiles.  The fine detector's 8-voxel work-items would be 2^24
    workgroups; one flag byte per (tile, view) in the workspace tells how many there are."""
    geom = ctr.ScanGeometry(make_params(ImagePixelSpacing=[0.01, 0.01, 0.01], DetectorPixelSize=[0.002, 0.002]))
    g = geom.ctypes_struct()
    g.nx, g.ny, g.nz, g.n_views = 1, 65535, 32767, 1
    assert N.lib().ctr_dd_backproject_workspace_bytes(ctypes.byref(g), 0) < (2 ** 32 - 1) // 256
