"""Echo sums over many echoes and labels: chunks of several pieces, one chunk for
everything, and sizes whose blocks of 1024 spins would pass what a grid holds, for
one call and for all the tiles of a batch."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _tile

pytestmark = pytest.mark.gpu


def _sums(M1, T, n_sub):
    """The same sums in float64: by masks where there are few, else by index_add."""
    import torch
    n_te = T.shape[1]
    if n_sub <= 9 and n_te <= 9:
        on = [(T == lab)[..., None] for lab in range(n_sub)]
        return torch.stack([torch.cat([(M1[..., :2].double() * o).sum(0), o.double().sum(0)], -1) for o in on], 1)
    idx = (torch.arange(n_te, device="cuda") * n_sub + T.long()).reshape(-1)
    out = torch.zeros((n_te * n_sub, 3), dtype=torch.float64, device="cuda")
    for i in range(2):
        out[:, i].index_add_(0, idx, M1[..., i].reshape(-1).double())
    out[:, 2].copy_(torch.bincount(idx, minlength=n_te * n_sub))
    return out.view(n_te, n_sub, 3)


@pytest.mark.parametrize("f64", [False, True])
@pytest.mark.parametrize("n,n_te,n_sub", [
    (4095 * 1024, 1, 3), (4096 * 1024, 2, 3), (8192 * 1024 + 1, 1, 5),     # 1, 2 and 2 pieces a chunk
    (100003, 9, 200),                                                      # a ragged last chunk
    (3000, 100, 255), (1024, 4097, 4), (0, 3, 9),                          # one chunk for all spins
])
def test_chunks_of_many_pieces(engine, n, n_te, n_sub, f64):
    _check(engine, n, n_te, n_sub, f64)


def test_more_labels_than_blocks_of_a_grid(engine):
    """1030 pieces x 255 echoes x 64 groups of labels: 1.7e7 blocks of one piece."""
    _check(engine, 1030 * 1024, 255, 256, False)


def _check(engine, n, n_te, n_sub, f64):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n + n_te)
    M1 = torch.randn((n, n_te, 3), generator=g, device="cuda", dtype=torch.float64 if f64 else torch.float32)
    T = torch.randint(0, n_sub, (n, n_te), generator=g, device="cuda", dtype=torch.uint8)
    out = torch.full((n_te, n_sub, 3), 7.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()                             # the engine's stream does not wait for torch's
    engine.echo_reduce(M1, T, n_sub, out)
    engine.sync()
    want = _sums(M1, T, n_sub)
    assert torch.equal(out[..., 2], want[..., 2])
    # n additions of terms of order 1, each rounded to 2^-53 of a sum below 6 sqrt(n)
    assert (out - want).abs().max().item() <= n * 6 * np.sqrt(n) * 2.0 ** -53


def test_tiles_beyond_one_grid(engine):
    """20 tiles of 13200 echoes and 256 labels: 844800 blocks each, 1.7e7 in all."""
    import torch
    n_te = 13200
    cfg = cases.gre(256, TE=50 * n_te, dt=50)
    cfg["TE"] = [50 * (k + 1) for k in range(n_te)]
    m, f = cases.blocky_phantom((12, 12, 12), n_labels=200, seed=3)
    ph, tiles = None, []
    for k in range(20):
        t = _tile(engine, torch, cases.make_case(cfg, m, f, 12.0, n_spins=1 + k % 3), ph=ph)
        ph = t["phantom"]
        t["params"].seed = 10 + k
        tiles.append(t)
    b = engine.batch(tiles)
    for _ in range(2):
        b.run()
        for t in tiles:
            # up to 3 terms of at most 1
            assert (t["echo_sums"] - _sums(t["M1"], t["T"], 256)).abs().max().item() <= 3 * 2.0 ** -52
            one = torch.full_like(t["echo_sums"], 7.0)
            torch.cuda.synchronize()
            engine.echo_reduce(t["M1"], t["T"], 256, one)
            engine.sync()
            assert torch.equal(t["echo_sums"], one)
            assert one[..., 2].sum().item() == t["T"].numel()
    b.close()
