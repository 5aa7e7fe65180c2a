"""A batch of tiles of every kind: scans of one TR, scans with dummy TRs, recorded
trajectories above and below the staging line, and fused tiles, each equal to its
separate walk; scans with and without dummy TRs share one launch."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _check, _clear, _separate, _tile
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu
PXY = [[1, 0.5], [0.5, 1]]


def _tiles(engine, torch, kinds, **kw):
    m, f = cases.blocky_phantom((20, 18, 22), n_labels=2, seed=4)
    ph = engine.phantom(m, f, np.full(3, 20e-6, np.float32), formats=(E.SW_FIELD_F32, E.SW_FIELD_Q16))
    gre = cases.gre(2, TE=1500, dt=50, P_XY=PXY)
    ssfp = cases.bssfp(2, TE=400, dt=50, dummies=6, lin=90.0, P_XY=PXY, WHAT_TO_SCALE=2, SCALE=[1.0, 0.5])
    out = []
    for k, kind in enumerate(kinds):
        cfg, n = {"gre": (gre, 3000), "cross": (dict(gre, CROSS_FOV=1), 900), "ssfp": (ssfp, 2500),
                  "rows": (dict(gre, TE=[500], TR=550, RECORD_TRAJECTORY=1), 73728),
                  "few rows": (dict(gre, RECORD_TRAJECTORY=1), 700), "fused": (ssfp, 1100)}[kind]
        cfg = dict(cfg, SEED=10 + k)
        case = cases.make_case(cfg, m, f, 20.0, n_spins=n)
        out.append(_tile(engine, torch, case, ph=ph, **kw))
        if kind == "fused":
            out.append(_tile(engine, torch, case, 1, ph=ph, shared={x: out[-1][x] for x in ("M0", "XYZ0")}, **kw))
    return out


@pytest.mark.parametrize("kinds", [("gre", "ssfp"), ("ssfp", "gre", "cross", "few rows"), ("rows", "gre", "ssfp"),
                                   ("fused", "gre", "ssfp", "rows", "few rows")])
@pytest.mark.parametrize("mixed", [False, True])
def test_groups_equal_separate_walks(engine, kinds, mixed):
    import torch
    kw = dict(precision=E.SW_PREC_F32_KAHAN, field_format=E.SW_FIELD_Q16) if mixed else {}
    tiles = _tiles(engine, torch, kinds, **kw)
    refs = [_separate(engine, torch, t) for t in tiles]
    b = engine.batch(tiles)
    for _ in range(3):
        _clear(tiles)
        torch.cuda.synchronize()
        st = b.run()
        for t, r, x in zip(tiles, refs, st["items"]):
            _check(t, r, x)
    b.close()


@pytest.mark.parametrize("kinds,launches", [(("ssfp", "ssfp"), 1), (("gre", "ssfp"), 1), (("gre", "gre", "few rows", "ssfp"), 1),
                                            (("gre", "cross"), 1), (("cross", "gre", "ssfp"), 2), (("rows", "gre"), 2),
                                            (("rows", "ssfp"), 2), (("few rows", "gre"), 1)])
def test_launches(engine, kinds, launches):
    """Graph nodes: counter reset, the walks, and the two passes of the echo sums."""
    import torch
    b = engine.batch(_tiles(engine, torch, kinds))
    assert b.graph_info()["nodes"] == launches + 3
    b.close()
