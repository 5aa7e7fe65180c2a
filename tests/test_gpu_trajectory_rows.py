"""Recorded trajectories written by sectors (73728 spins or more in a walk) equal
those of the same spins walked in parts below that line, word for word: rows of
every alignment, rows shorter than a sector, spins lost on the way, rows of
several TRs, and nothing written outside the rows."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _tile
from tests.test_gpu_production import run
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu

N = 73728


@pytest.fixture(scope="module")
def engine():
    eng = E.Engine(0)
    yield eng
    eng.close()


def _case(n, te, **kw):
    m, f = cases.blocky_phantom((20, 18, 22), n_labels=2, seed=4)
    cfg = cases.gre(2, TE=te, dt=50, RECORD_TRAJECTORY=1, **kw)
    return cases.make_case(cfg, m, f, 20.0, n_spins=n)


@pytest.mark.parametrize("n", [N, N + 1, N + 63, 90001])
@pytest.mark.parametrize("kind", ["1 step", "2 steps", "5 steps", "24 steps", "walls", "lost", "dummies", "wrap"])
def test_rows_equal_those_of_parts(engine, kind, n):
    te = {"1 step": 50, "2 steps": 100, "5 steps": 250, "24 steps": 1200}.get(kind, 650)
    kw = dict(walls={}, lost=dict(MAX_ITERATIONS=0, DIFFUSIVITY=[4e-8, 4e-8]), dummies=dict(DUMMY_SCAN=2),
              wrap=dict(CROSS_FOV=1, P_XY=[[1, 0.5], [0.5, 1]])).get(kind, {})
    case = _case(n, te, **kw)
    whole = run(engine, case)
    parts = [run(engine, case, spin_offset=o, n=min(40000, n - o)) for o in range(0, n, 40000)]
    for k in ("XYZ1", "M1", "T"):
        np.testing.assert_array_equal(whole[k], np.concatenate([p[k] for p in parts]))
    if kind == "lost":
        assert whole["stats"]["n_lost"] > 100


def test_views_and_unaligned_buffers(engine):
    """Tiles that walk the same trajectories write one view each, here at bases a
    word apart, with guard words before and after."""
    import torch
    case = _case(N + 5, 600)
    ph = engine.phantom(case.mask, case.field_T, case.fov)
    tiles, raws = [], []
    for shift in (0, 1, 2, 3):
        t = _tile(engine, torch, case, ph=ph)
        n = t["XYZ1"].numel()
        raw = torch.full((n + 64,), 7.0, device="cuda")
        t["XYZ1"] = raw[16 + shift:16 + shift + n].view(t["XYZ1"].shape)
        tiles.append(t)
        raws.append((raw, 16 + shift, n))
    b = engine.batch(tiles)
    b.run()
    torch.cuda.synchronize()
    ref = np.concatenate([run(engine, case, spin_offset=o, n=min(40000, N + 5 - o))["XYZ1"] for o in range(0, N + 5, 40000)])
    for t, (raw, at, n) in zip(tiles, raws):
        np.testing.assert_array_equal(t["XYZ1"].cpu().numpy(), ref)
        assert (raw[:at] == 7.0).all() and (raw[at + n:] == 7.0).all()
    b.close()
