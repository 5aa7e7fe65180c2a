"""Single walks of up to 32768 spins fill half of each wave's lanes: at the edges of
lanes, blocks and of that line their results equal those of a batch's tile, which
always takes full waves."""
import pytest

from tests import cases
from tests.test_gpu_batch import _check, _separate, _tile
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    eng = E.Engine(0)
    yield eng
    eng.close()


@pytest.mark.parametrize("n", [1, 31, 32, 33, 127, 128, 129, 1024, 1025, 32767, 32768, 32769])
@pytest.mark.parametrize("kind", ["one TR", "dummies", "trajectory", "replay"])
def test_edges(engine, kind, n):
    import torch
    if kind == "replay" and n > 2000:
        n = 2000 + n % 100                                # the draws are made on the host
    m, f = cases.blocky_phantom((20, 18, 22), n_labels=2, seed=4)
    cfg = cases.gre(2, TE=600, dt=50, P_XY=[[1, 0.5], [0.5, 1]], DUMMY_SCAN=2 if kind == "dummies" else 0,
                    RECORD_TRAJECTORY=int(kind == "trajectory"))
    case = cases.make_case(cfg, m, f, 20.0, n_spins=n)
    t = _tile(engine, torch, case, rng=E.SW_RNG_REPLAY if kind == "replay" else E.SW_RNG_PHILOX)
    ref = _separate(engine, torch, t)
    b = engine.batch([t])
    st = b.run()
    torch.cuda.synchronize()
    _check(t, ref, st["items"][0])
    b.close()
