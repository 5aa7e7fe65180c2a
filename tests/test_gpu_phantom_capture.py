"""Phantoms beside a captured walk: created after the capture of a graph that uses the
engine's scratch, and destroyed while a stream captures; the graph replays as the eager
walk runs."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _separate, _tile

pytestmark = pytest.mark.gpu


def _walk(engine, t, stream, noalloc):
    engine.walk_device(t["phantom"], t["sequence"], t["params"], t["M0"], t["XYZ0"], t["M1"], t["XYZ1"], t["T"],
                       spatial_order=0, stream=stream, stats=False, noalloc=noalloc)


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("when", ["after", "during"])
def test_phantoms_and_a_captured_walk(engine, when, noalloc):
    import torch
    m, f = cases.blocky_phantom((20, 18, 22), n_labels=2, seed=4)
    case = cases.make_case(cases.gre(2, TE=900, dt=50, P_XY=[[1, 0.5], [0.5, 1]]), m, f, 20.0, n_spins=3000)
    t = _tile(engine, torch, case)
    ref = _separate(engine, torch, t)
    spare = engine.phantom(1 - m, f, case.fov)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        _walk(engine, t, s, noalloc)                                   # the excitation table
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s, capture_error_mode="relaxed"):
        _walk(engine, t, s, noalloc)
        if when == "during":
            spare.close()
    spare.close()
    fresh = engine.phantom(m, f, case.fov)
    for _ in range(3):
        for k in ("M1", "T", "XYZ1"):
            t[k].zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for k in ("M1", "T", "XYZ1"):
            np.testing.assert_array_equal(t[k].cpu().numpy(), ref[k])
        u = dict(t, phantom=fresh)
        np.testing.assert_array_equal(_separate(engine, torch, u)["M1"], ref["M1"])
    fresh.close()
