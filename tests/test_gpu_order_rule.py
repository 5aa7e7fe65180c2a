"""A single walk that asks for spatial order visits its spins unsorted up to 212992
spins, and on records that fit an L2: on both sides of those lines its results
equal those of a walk without order, bit for bit."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_production import run
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    eng = E.Engine(0)
    yield eng
    eng.close()


@pytest.mark.parametrize("n", [1, 212991, 212992, 212993])
@pytest.mark.parametrize("side", [24, 108])               # 0.1 MB of records, and more than the 4 MiB of an L2
def test_both_sides_of_the_line(engine, side, n):
    m, f = cases.blocky_phantom((side,) * 3, n_labels=2, seed=side)
    case = cases.make_case(cases.gre(2, TE=500, dt=50, P_XY=[[1, 0.5], [0.5, 1]]), m, f, 40.0, n_spins=n)
    a, b = (run(engine, case, spatial_order=o) for o in (0, 1))
    for k in ("M1", "T", "XYZ1"):
        np.testing.assert_array_equal(a[k], b[k])
    for k in ("n_lost", "n_steps", "n_attempts"):
        assert a["stats"][k] == b["stats"][k]
