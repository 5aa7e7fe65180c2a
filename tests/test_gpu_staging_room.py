"""LDS staging where the tables leave no room for it, and beside no tables: a phantom of
9000 voxels along x (36 KB of per-axis tables, so no ring and no staged draws) and one of
16400 (64-bit addresses, staging alone).  Recorded trajectories above the staging line
equal those of their parts below it and of the loop in double precision; replayed walks
equal the oracle's trajectories and labels."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _check as check_tile
from tests.test_gpu_batch import _separate, _tile
from tests.test_gpu_production import run
from tests.test_gpu_replay import _assert_parity, _replay_streams, _run_engine
from oracle import oracle as orc
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu

LONG = [(9000, 3, 3), (16400, 3, 3)]
FOV = {9000: [900.0, 3.0, 3.0], 16400: [1640.0, 3.0, 3.0]}


def _case(dims, n, rec, te=650, **kw):
    m, f = cases.blocky_phantom(dims, n_labels=2, seed=4)
    cfg = cases.gre(2, TE=te, dt=50, RECORD_TRAJECTORY=rec, P_XY=[[1, 0.5], [0.5, 1]], **kw)
    return cases.make_case(cfg, m, f, FOV[dims[0]], n_spins=n)


@pytest.mark.parametrize("dims", LONG)
@pytest.mark.parametrize("dummies", [0, 2])
@pytest.mark.parametrize("n", [73728, 80001])
def test_recorded_rows(engine, dims, dummies, n):
    case = _case(dims, n, 1, DUMMY_SCAN=dummies)
    whole = run(engine, case)
    parts = [run(engine, case, spin_offset=o, n=min(40000, n - o)) for o in range(0, n, 40000)]
    for k in ("XYZ1", "M1", "T"):
        np.testing.assert_array_equal(whole[k], np.concatenate([p[k] for p in parts]))
    np.testing.assert_array_equal(whole["XYZ1"], run(engine, case, precision=E.SW_PREC_F64)["XYZ1"])


@pytest.mark.parametrize("dims", LONG)
def test_recorded_rows_of_a_batch(engine, dims):
    import torch
    case = _case(dims, 73728, 1)
    t = _tile(engine, torch, case)
    ref = _separate(engine, torch, t)
    b = engine.batch([t])
    st = b.run()
    check_tile(t, ref, st["items"][0])
    b.close()


@pytest.mark.parametrize("dims", LONG)
@pytest.mark.parametrize("precision", [E.SW_PREC_F32, E.SW_PREC_F64])
@pytest.mark.parametrize("rec", [0, 1])
def test_replayed_draws(engine, dims, precision, rec):
    case = _case(dims, 300, rec, te=2000)
    rp = _replay_streams(case)
    f64 = precision == E.SW_PREC_F64
    _assert_parity(_run_engine(engine, case, replay=rp, precision=precision), orc.sim(cases.to_oracle(case), f64=f64), f64=f64)
