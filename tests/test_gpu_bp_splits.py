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
