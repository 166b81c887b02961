"""The cached row and column sums of the iterative methods: read from several streams at once, from a graph
captured on another stream, worked out inside a capture, and after the geometry has changed.  The same kernels
on the same inputs, so results are compared bit for bit."""
import pytest
import torch

import ctreconstruction_amd as ctr
from ctreconstruction_amd import _native as N
from ctreconstruction_amd import iterative as IT
from tests.conftest import make_params

pytestmark = pytest.mark.gpu


def _scan(seed=0, **kw):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    N.lib()
    p = make_params(NumberOfImage=[48, 48, 32], ImagePixelSpacing=[0.8] * 3, NumberOfViews=24,
                    NumberOfDetectorPixels=[96, 64], DetectorPixelSize=[0.9, 0.9], **kw)
    geom = ctr.ScanGeometry(p)
    return geom, torch.rand(geom.proj_shape, generator=torch.Generator().manual_seed(seed)).cuda(), p


@pytest.mark.parametrize("backprojector", ["matched", "ref"])
def test_a_second_stream_reads_finished_sums(backprojector):
    geom, proj, p = _scan()
    ref = IT.sart(proj, ctr.ScanGeometry(p), 2, backprojector=backprojector)
    torch.cuda.synchronize()
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    load = torch.rand((4096, 4096), device="cuda")
    with torch.cuda.stream(first):
        for _ in range(20):             # the sums wait behind this
            load = (load @ load).clamp(0, 1)
        a = IT.sart(proj, geom, 2, backprojector=backprojector)
    with torch.cuda.stream(second):
        b = IT.sart(proj, geom, 2, backprojector=backprojector)
    torch.cuda.synchronize()
    assert torch.equal(a, ref) and torch.equal(b, ref)
    assert len(IT._NORM_CACHE[geom]) == 1


def test_changed_geometries_get_their_own_sums():
    geom, proj, p = _scan()
    before = IT.sart(proj, geom, 1)
    assert torch.equal(IT.sart(proj, geom, 1), before)
    geom.det_offset[0] = 4.0            # in place: the array stays the same object
    after = IT.sart(proj, geom, 1)
    fresh = IT.sart(proj, ctr.ScanGeometry({**p, "DetectorOffset": [4.0, 0]}), 1)
    assert torch.equal(after, fresh) and not torch.equal(after, before)
    geom.du *= 1.25
    p["DetectorPixelSize"] = [p["DetectorPixelSize"][0] * 1.25, p["DetectorPixelSize"][1]]
    assert torch.equal(IT.sart(proj, geom, 1), IT.sart(proj, ctr.ScanGeometry({**p, "DetectorOffset": [4.0, 0]}), 1))
    assert len(IT._NORM_CACHE[geom]) == 1   # the old sums are not kept


@pytest.mark.parametrize("warm", [True, False])
def test_capture(warm):
    """Replays equal the eager result; sums captured but not yet run never reach an eager call."""
    geom, proj, p = _scan()
    if warm:
        IT.sart(proj, geom, 1)
    else:
        ctr.dd_forward(torch.zeros(geom.vol_shape, device="cuda"), geom)   # the views are on the device
    data = proj.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = IT.sart(data, geom, 2)
    other = ctr.ScanGeometry(p)
    assert torch.equal(IT.sart(proj, geom, 2), IT.sart(proj, other, 2))    # before the graph has run
    for k in range(3):
        data.copy_(_scan(seed=k + 1)[1])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, IT.sart(data, other, 2))
