"""A single walk of 393216 spins or more on records beyond the L2s runs with fewer
waves on a SIMD: on both sides of each line its results equal those of the same
spins walked in two halves, which are below the line; and a batch of such tiles
starts with the cap in its schedule."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _tile
from tests.test_gpu_production import run
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    eng = E.Engine(0)
    yield eng
    eng.close()


@pytest.mark.parametrize("dummies", [0, 2])
@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("side,n", [(96, 393216), (190, 393215), (190, 393216), (190, 400001)])
def test_whole_equals_halves(engine, side, n, order, dummies):
    m, f = cases.blocky_phantom((side,) * 3, n_labels=2, seed=side)
    cfg = cases.gre(2, TE=400, dt=50, P_XY=[[1, 0.5], [0.5, 1]], DUMMY_SCAN=dummies)
    case = cases.make_case(cfg, m, f, 90.0, n_spins=n)
    half = n // 2
    whole = run(engine, case, spatial_order=order)
    parts = [run(engine, case, spin_offset=o, n=k, spatial_order=order) for o, k in ((0, half), (half, n - half))]
    for k in ("M1", "T", "XYZ1"):
        np.testing.assert_array_equal(whole[k], np.concatenate([p[k] for p in parts]))
    for k in ("n_lost", "n_steps", "n_attempts"):
        assert whole["stats"][k] == sum(p["stats"][k] for p in parts)


@pytest.mark.parametrize("side,tiles,waves", [(190, 4, 4), (190, 3, 0), (96, 4, 5), (96, 3, 0)])
def test_default_schedule_of_a_batch(engine, side, tiles, waves):
    import torch
    m, f = cases.blocky_phantom((side,) * 3, n_labels=2, seed=side)
    case = cases.make_case(cases.gre(2, TE=200, dt=50), m, f, 90.0, n_spins=100000)
    ph = engine.phantom(case.mask, case.field_T, case.fov)
    items = [_tile(engine, torch, case, ph=ph) for _ in range(tiles)]
    for k, t in enumerate(items):
        t["params"].seed = 10 + k                          # tiles of one seed would fuse
    b = engine.batch(items)
    assert b.schedule["waves_per_simd"] == waves
    b.close()
