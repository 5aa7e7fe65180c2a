"""Spins of long steps are visited sorted from fewer spins on, with the results of a
walk without order."""
import numpy as np
import pytest

from tests import cases
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
