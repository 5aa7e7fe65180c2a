"""A phantom's device memory may be a block an earlier phantom left: every array
in it is written whole, so walks on it equal walks on fresh memory, for every
record format (padding of ragged bricks included)."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_production import run
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu

ALL = (E.SW_FIELD_F32, E.SW_FIELD_F16, E.SW_FIELD_BF16, E.SW_FIELD_Q16)


def _walks(eng, case):
    """Single walks in every format, a replay-layout walk and a batch tile."""
    out = []
    for fmt in ALL:
        out.append(run(eng, case, field_format=fmt, formats=ALL)["M1"])
    return out


@pytest.mark.parametrize("dims", [(13, 7, 9), (24, 24, 24), (25, 31, 18)])
@pytest.mark.parametrize("field", [True, False])
def test_reused_block_equals_fresh_memory(dims, field):
    cfg = cases.gre(2, TE=2000, dt=50, P_XY=[[1, 0.5], [0.5, 1]])
    big_m, big_f = cases.blocky_phantom((26, 31, 24), n_labels=2, seed=7)
    m, f = cases.blocky_phantom(dims, n_labels=2, seed=8)
    case = cases.make_case(cfg, m, f if field else None, 25.0, n_spins=700)
    used = E.Engine(0)
    for _ in range(3):                                   # blocks full of another phantom's records
        used.phantom(np.full_like(big_m, 1), big_f + 1.0, np.full(3, 25e-6, np.float32), formats=ALL).close()
    fresh = E.Engine(0)
    for a, b in zip(_walks(used, case), _walks(fresh, case)):
        np.testing.assert_array_equal(a, b)
    used.close()
    fresh.close()


def test_phantom_outlives_its_engine():
    m, f = cases.two_substrate_phantom(n=12, fov_um=24.0, seed=9)
    eng = E.Engine(0)
    ph = eng.phantom(m, f, np.full(3, 24e-6, np.float32))
    eng.close()
    ph.close()
