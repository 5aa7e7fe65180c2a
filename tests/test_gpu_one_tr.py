"""The step loop of single-TR scans and of recorded trajectories (walk_prod.hpp)
against the two-attempt loop, which shares none of its code: the same draws, so
magnetisation, labels, positions and counts agree bit for bit.  The cases stand
where the two loops differ: walls hit by every lane and steps longer than the
FoV (the reference's int64 subscripts), tissue tables that do not fit LDS,
closed and half-open boundaries, spins stuck on their first attempts, a TR of
one time point, the 64-bit record offsets, and launches of 1 to 65 spins."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_step_loop import both
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu

FORMATS = (E.SW_FIELD_F32, E.SW_FIELD_F16, E.SW_FIELD_BF16, E.SW_FIELD_Q16)
MODES = [(E.SW_PREC_F32, E.SW_FIELD_F32), (E.SW_PREC_F32, E.SW_FIELD_BF16), (E.SW_PREC_F32_KAHAN, E.SW_FIELD_Q16),
         (E.SW_PREC_F64, E.SW_FIELD_F32)]


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("cross", [0, 1])
def test_wild_steps_on_an_uneven_phantom(engine, cross, mode):
    m, f = cases.blocky_phantom((7, 12, 9), n_labels=2, seed=1)
    cfg = cases.se(2, TE=2000, dt=50, DIFFUSIVITY=[4e-7, 1e-7], P_XY=[[1, 0.4], [0.4, 1]], CROSS_FOV=cross)
    case = cases.make_case(cfg, m, f, 12.0, n_spins=2000)
    g = both(engine, case, precision=mode[0], field_format=mode[1], formats=FORMATS)
    assert g["stats"]["n_lost"] > 0


@pytest.mark.parametrize("record", [0, 1])
@pytest.mark.parametrize("n_sub,p", [(2, 0.0), (20, 0.3)])
def test_tissue_tables(engine, n_sub, p, record):
    """Closed boundaries, and more tissues than the LDS tables hold."""
    m, f = cases.blocky_phantom((20, 17, 23), n_labels=n_sub, seed=2, block=4)
    pxy = np.full((n_sub, n_sub), p)
    np.fill_diagonal(pxy, 1.0)
    cfg = cases.gre(n_sub, TE=3000, dt=50, P_XY=pxy.tolist(), RECORD_TRAJECTORY=record,
                    DIFFUSIVITY=np.linspace(0.5e-9, 2e-9, n_sub).tolist(), T1=np.linspace(500, 2000, n_sub).tolist(),
                    T2=np.linspace(20, 60, n_sub).tolist())
    g = both(engine, cases.make_case(cfg, m, f, 20.0, n_spins=3000))
    assert g["stats"]["n_attempts"] > g["stats"]["n_steps"]


@pytest.mark.parametrize("max_iterations", [0, 3])
def test_stuck_spins(engine, max_iterations):
    """Spins enclosed by walls they may not cross are abandoned after
    max_iterations + 2 rejections in a row; rejections apart do not add up."""
    m, f = cases.blocky_phantom((12, 12, 12), n_labels=2, seed=3, block=1)
    cfg = cases.gre(2, TE=1500, dt=50, P_XY=[[1, 0.0], [0.0, 1]], MAX_ITERATIONS=max_iterations,
                    DIFFUSIVITY=[5e-9, 5e-9])
    g = both(engine, cases.make_case(cfg, m, f, 12.0, n_spins=1500))
    assert 0 < g["stats"]["n_lost"] <= 1500


@pytest.mark.parametrize("n_spins", [1, 63, 65])
def test_short_scans_and_few_spins(engine, n_spins):
    m, f = cases.two_substrate_phantom(n=16, fov_um=32.0, seed=4)
    cfg = cases.gre(2, TE=0, dt=50)
    case = cases.make_case(cfg, m, f, 32.0, n_spins=n_spins)
    assert case.params.n_timepoints == 1
    both(engine, case)


def test_64_bit_offsets(engine):
    """Per-axis tables beyond 64 KiB: record offsets in 64-bit arithmetic."""
    m, f = cases.blocky_phantom((16400, 3, 3), n_labels=2, seed=5, block=3)
    cfg = cases.se(2, TE=2000, dt=50, P_XY=[[1, 0.5], [0.5, 1]])
    both(engine, cases.make_case(cfg, m, f, 8200.0, n_spins=2000))
