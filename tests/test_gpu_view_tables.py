"""The views that a geometry keeps on the device: their memory is not given to others while another stream
still reads it, and they follow the geometry's arrays."""
import copy
import pickle

import numpy as np
import pytest
import torch

import ctreconstruction_amd as ctr
from ctreconstruction_amd import _native as N
from tests.conftest import make_params

pytestmark = pytest.mark.gpu


def _scan(**kw):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    p = make_params(NumberOfImage=[40, 40, 24], ImagePixelSpacing=[0.8] * 3, NumberOfViews=20,
                    NumberOfDetectorPixels=[64, 48], **kw)
    geom = ctr.ScanGeometry(p)
    return geom, torch.rand(geom.vol_shape, generator=torch.Generator().manual_seed(0)).cuda(), p


def test_tables_outlive_their_geometry_on_another_stream():
    geom, vol, p = _scan()
    ref = ctr.dd_forward(vol, ctr.ScanGeometry(p))
    geom.device_views(vol.device)                   # uploaded, and their memory owned, on the default stream
    load, side = torch.rand((4096, 4096), device="cuda"), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):                         # the projection waits behind this
            load = (load @ load).clamp(0, 1)
        out = ctr.dd_forward(vol, geom)
    del geom
    taken = [torch.zeros(20, dtype=torch.float64, device="cuda") for _ in range(64)]
    torch.cuda.synchronize()
    assert torch.equal(out, ref) and len(taken) == 64


def test_views_follow_the_arrays():
    geom, vol, p = _scan()
    ctr.dd_forward(vol, geom)
    turned = ctr.ScanGeometry({**p, "StartAngle": 0.3, "EndAngle": 0.3 + 2 * np.pi})
    geom.angles[:] = turned.angles                  # in place
    geom.branch[:] = turned.branch
    assert torch.equal(ctr.dd_forward(vol, geom), ctr.dd_forward(vol, turned))


def test_used_geometries_are_copied_and_pickled():
    geom, vol, _ = _scan()
    ref = ctr.dd_forward(vol, geom)
    for other in (copy.copy(geom), copy.deepcopy(geom), pickle.loads(pickle.dumps(geom))):
        assert torch.equal(ctr.dd_forward(vol, other), ref)
