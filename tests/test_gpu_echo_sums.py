"""Echo sums at the edges of the reduction's chunks (1024 spins a block, 256
partials a pass): counts exact, sums within float64 rounding, and those of a
batch's one launch over all its tiles equal to the single call's bit for bit."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _tile
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    eng = E.Engine(0)
    yield eng
    eng.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 2049, 1024 * 256, 1024 * 257 + 3])
def test_edges_of_chunks(engine, n, dtype):
    import torch
    rng = np.random.default_rng(n)
    M1 = rng.normal(size=(n, 2, 3)).astype(dtype)
    T = rng.integers(0, 3, size=(n, 2)).astype(np.uint8)
    out = torch.full((2, 3, 3), 7.0, dtype=torch.float64, device="cuda")
    for _ in range(2):                                    # the second call finds the first one's scratch
        engine.echo_reduce(torch.from_numpy(M1).cuda(), torch.from_numpy(T).cuda(), 3, out)
    got = out.cpu().numpy()
    want = np.array([[[*(M1[:, te, :2].astype(np.float64) * on[:, None]).sum(0), on.sum()]
                      for on in (T[:, te] == lab for lab in range(3))] for te in range(2)])
    np.testing.assert_array_equal(got[..., 2], want[..., 2])
    # n additions of terms of order 1, each rounded to 2^-53 of a sum below 6 sqrt(n)
    np.testing.assert_allclose(got, want, rtol=0, atol=n * 6 * np.sqrt(n) * 2.0 ** -53)


def test_tiles_of_a_batch(engine):
    import torch
    cfg = cases.gre(2, TE=1000, dt=50, P_XY=[[1, 0.5], [0.5, 1]])
    m, f = cases.blocky_phantom((12, 12, 12), n_labels=2, seed=3)
    tiles = [_tile(engine, torch, cases.make_case(cfg, m, f, 12.0, n_spins=n)) for n in (700, 1024, 1, 5000, 1025)]
    b = engine.batch(tiles)
    for _ in range(2):
        b.run()
        for t in tiles:
            one = torch.full_like(t["echo_sums"], 7.0)
            engine.echo_reduce(t["M1"], t["T"], t["params"].n_substrate, one)
            assert torch.equal(t["echo_sums"], one)
            assert one[..., 2].sum().item() == t["T"].numel()
    b.close()
