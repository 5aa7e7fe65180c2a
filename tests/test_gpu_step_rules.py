"""Spins of long steps are visited sorted from fewer spins on, with the results of a
walk without order, and batches of scans with dummy TRs start with 5 waves a SIMD
where scans of one TR start with 4."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _tile
from tests.test_gpu_production import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [97000, 100000])            # the line is at 98281 spins for this step (1.26 voxels)
def test_sorted_equals_unsorted(engine, n):
    m, f = cases.blocky_phantom((108,) * 3, n_labels=2, seed=3)
    case = cases.make_case(cases.gre(2, TE=500, dt=50, P_XY=[[1, 0.5], [0.5, 1]]), m, f, 27.1, n_spins=n)
    a, b = (run(engine, case, spatial_order=o) for o in (0, 1))
    for k in ("M1", "T", "XYZ1"):
        np.testing.assert_array_equal(a[k], b[k])
    for k in ("n_lost", "n_steps", "n_attempts"):
        assert a["stats"][k] == b["stats"][k]


@pytest.mark.parametrize("n", [32769, 40001])
@pytest.mark.parametrize("n_sub,fov", [(2, 27.1), (2, 60.0), (20, 100.0)])     # steps of 0.74, 0.34 and 0.2 voxels
def test_general_loop_equals_production_loop(engine, n, n_sub, fov):
    """The whole walk takes the general loop (or, at 0.34, does not), its parts of up to
    32768 spins the production loop."""
    m, f = cases.blocky_phantom((64,) * 3, n_labels=n_sub, seed=3)
    pxy = np.random.default_rng(2).uniform(0.2, 0.8, (n_sub, n_sub)).tolist()
    case = cases.make_case(cases.gre(n_sub, TE=900, dt=50, P_XY=pxy), m, f, fov, n_spins=n)
    whole = run(engine, case)
    parts = [run(engine, case, spin_offset=o, n=min(20000, n - o)) for o in range(0, n, 20000)]
    for k in ("M1", "T", "XYZ1"):
        np.testing.assert_array_equal(whole[k], np.concatenate([p[k] for p in parts]))
    for k in ("n_lost", "n_steps", "n_attempts"):
        assert whole["stats"][k] == sum(p["stats"][k] for p in parts)


@pytest.mark.parametrize("dummies,waves", [(0, 4), (4, 5)])
def test_default_waves_of_a_batch(engine, dummies, waves):
    import torch
    m, f = cases.blocky_phantom((190,) * 3, n_labels=2, seed=3)
    case = cases.make_case(cases.gre(2, TE=200, dt=50, DUMMY_SCAN=dummies), m, f, 90.0, n_spins=100000)
    ph = engine.phantom(case.mask, case.field_T, case.fov)
    items = [_tile(engine, torch, case, ph=ph) for _ in range(4)]
    for k, t in enumerate(items):
        t["params"].seed = 10 + k                          # tiles of one seed would fuse
    b = engine.batch(items)
    assert b.schedule["waves_per_simd"] == waves
    b.close()
