"""The forward projector where enough column groups are at work that the slabs are not shared out (one wavefront
per group, over 256 groups at fewer than 56 slabs and over 700 above): ragged sizes, row blocks shifted and not,
a coarse and a fine angular step, and a batch whose groups together pass the line that one volume does not.

Tolerance 1e-4 of the peak against the oracle, as for every operator; a batch against single volumes 1e-6 (FP64
partial sums in another order)."""
import numpy as np
import pytest
import torch

import ctreconstruction_amd as ctr
from ctreconstruction_amd import _native as N
from ctreconstruction_amd.autograd import forward_batch
from oracle import dd_oracle as O
from tests.conftest import make_params

pytestmark = pytest.mark.gpu

TOL = 1e-4


def _scan(n, det, views):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    return make_params(NumberOfImage=n, NumberOfDetectorPixels=det, DetectorPixelSize=[0.6, 0.6], NumberOfViews=views,
                       StartAngle=0.05, EndAngle=0.05 + 2 * np.pi)


# 328, 849 (row blocks shifted by 24) and 703 groups
@pytest.mark.parametrize("n,det,views", [([41, 37, 23], [61, 75], 171), ([70, 64, 40], [90, 130], 301),
                                         ([41, 50, 70], [75, 140], 150)])
def test_one_share_matches_the_oracle(n, det, views):
    p = _scan(n, det, views)
    g = O.Geometry(p)
    vol = np.random.default_rng(views).random((g.nz, g.ny, g.nx)).astype(np.float32)
    keep = list(range(0, views, views // 6))
    ref = O.forward_project(g, vol, views=keep)
    out = ctr.dd_forward(torch.from_numpy(vol).cuda(), ctr.ScanGeometry(p)).cpu().numpy()[keep]
    assert np.abs(out - ref).max() <= TOL * np.abs(ref).max()


def test_a_batch_in_one_share_equals_single_volumes_in_four():
    geom = ctr.ScanGeometry(_scan([37, 41, 20], [50, 47], 40))     # 62 groups a volume, 750 together
    vols = torch.rand((12,) + tuple(geom.vol_shape), generator=torch.Generator().manual_seed(0)).cuda()
    got = forward_batch(vols, geom)
    for b in range(12):
        ref = ctr.dd_forward(vols[b], geom)
        assert (got[b] - ref).abs().max() <= 1e-6 * ref.abs().max()
