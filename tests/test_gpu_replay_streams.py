"""Replayed draws come 24 normals and 8 uniforms at a time: streams of every
length and row alignment give the results of long ones, and a stream that ends
within a load is reported, never read beyond."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _separate, _tile
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    eng = E.Engine(0)
    yield eng
    eng.close()


@pytest.fixture(scope="module")
def long(engine):
    import torch
    m, f = cases.blocky_phantom((20, 18, 22), n_labels=2, seed=4)
    case = cases.make_case(cases.gre(2, TE=900, dt=50, P_XY=[[1, 0.5], [0.5, 1]]), m, f, 20.0, n_spins=300)
    t = _tile(engine, torch, case, rng=E.SW_RNG_REPLAY)
    return t, _separate(engine, torch, t)


@pytest.mark.parametrize("cut", [0, 1, 2, 3, 7, 22, 23, 24, 25])
@pytest.mark.parametrize("precision", [E.SW_PREC_F32, E.SW_PREC_F64])
def test_every_length(engine, long, cut, precision):
    import torch
    t, ref = long
    n, u = t["replay"]
    # more than any spin uses of the long streams, by the attempts of the walk
    used = int(3 * ref["stats"]["n_attempts"] / 300 * 3)
    assert used + 32 < n.shape[1]
    s = dict(t, replay=(n[:, :used + cut].contiguous(), u[:, :u.shape[1] - cut].contiguous()), precision=precision)
    if precision == E.SW_PREC_F64:
        s["M1"] = torch.zeros_like(t["M1"], dtype=torch.float64)
    got = _separate(engine, torch, s)
    np.testing.assert_array_equal(got["XYZ1"], ref["XYZ1"])
    np.testing.assert_array_equal(got["T"], ref["T"])
    assert got["stats"]["n_attempts"] == ref["stats"]["n_attempts"]
    if precision == E.SW_PREC_F32:
        np.testing.assert_array_equal(got["M1"], ref["M1"])


@pytest.mark.parametrize("length", [3, 4, 23, 24, 25, 27, 40])
def test_streams_that_end(engine, long, length):
    import torch
    t, _ = long
    n, u = t["replay"]
    # the last row ends where its allocation does
    s = dict(t, replay=(n[:, :length].contiguous(), u))
    with pytest.raises(E.EngineError, match="ran out of recorded draws"):
        _separate(engine, torch, s)
