"""The row filters over every transform length, with the row counts and detector widths where the
kernels differ: an odd number of rows, fewer rows than a workgroup takes, more rounds than one of the
persistent workgroups, widths that fill half of the transform, one more (the other half's first
sample) and just over a quarter.

Tolerance 1e-4 of the peak against float64, as for every operator (the filter's own error is under
3e-7)."""
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


def _widths(log2n):
    n = 1 << log2n
    return sorted({n // 2 + 1, n // 2, n // 2 - 1, n // 4 + 2})


@pytest.mark.parametrize("log2n", range(4, 14))
@pytest.mark.parametrize("rows", [1, 7, 66])
def test_every_length_matches_the_oracle(log2n, rows):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    for nu in _widths(log2n):
        if nu < 5:
            continue
        p = make_params(NumberOfDetectorPixels=[nu, rows], NumberOfViews=1, FilterType="hann")
        g = O.Geometry(p)
        geom = ctr.ScanGeometry(p)
        x = np.random.default_rng(nu).random((3 if rows == 7 else 1, rows, nu)).astype(np.float32)
        ref = O.filter_projections(g, x)
        xd = torch.from_numpy(x).cuda()
        out = ctr.fdk_filter(xd, geom).cpu().numpy()
        assert np.abs(out - ref).max() <= TOL * np.abs(ref).max(), nu
        same = ctr.fdk_filter(xd, geom, out=xd).cpu().numpy()  # in place
        assert np.array_equal(same, out)
        if rows > 1:
            prm = make_cone_params(DetectorWidth=nu, DetectorHeight=rows, NumberOfViews=2)
            y = np.random.default_rng(nu).random((2, rows, nu)).astype(np.float32)
            q = PF.pixel_filter(torch.from_numpy(y).cuda(), PF.PixelScan(prm)).cpu().numpy()
            qr = PO.filter_projections(PO.PixelGeometry(prm), y)
            assert np.abs(q - qr).max() <= TOL * np.abs(qr).max(), nu


# 1024 (512) resident workgroups at 2048 (4096) points: over four rounds of them, and an odd last pair
@pytest.mark.parametrize("nu,rows", [(1000, 8301), (1025, 8400), (1500, 4203)])
def test_persistent_workgroups_filter_every_row(nu, rows):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    p = make_params(NumberOfDetectorPixels=[nu, rows], NumberOfViews=1, FilterType="shepp-logan")
    geom = ctr.ScanGeometry(p)
    x = torch.rand((1, rows, nu), generator=torch.Generator().manual_seed(1))
    out = ctr.fdk_filter(x.cuda(), geom).cpu().numpy()
    for r0 in range(0, rows, 97):  # the same rows filtered a few at a time by the other kernel
        r1 = min(r0 + 3, rows)
        ref = O.filter_projections(O.Geometry(p), np.where(
            (np.arange(rows) >= r0)[None, :, None] & (np.arange(rows) < r1)[None, :, None], x.numpy(), 0))[:, r0:r1] \
            if r0 in (0, 97 * 40) else None
        if ref is not None:
            assert np.abs(out[:, r0:r1] - ref).max() <= TOL * np.abs(ref).max()
    # every row's sum against the float64 convolution's DC (Shepp-Logan's is zero): rows left out show
    assert np.isfinite(out).all() and (np.abs(out).max(axis=2) > 0).all()
