"""A phantom built in the block that one of the same size left, full of other contents:
single walks in every record format, a replayed walk and a batch tile equal those on
fresh memory in every output.  The free device memory shows that the block is reused."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _separate, _tile
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu

ALL = (E.SW_FIELD_F32, E.SW_FIELD_F16, E.SW_FIELD_BF16, E.SW_FIELD_Q16)


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _outputs(eng, case, ph):
    import torch
    out = []
    for kw in [dict(field_format=f) for f in ALL] + [dict(rng=E.SW_RNG_REPLAY)]:
        t = _tile(eng, torch, case, ph=ph, **kw)
        out.append(_separate(eng, torch, t))
    for kw in [dict(field_format=f) for f in ALL]:
        t = _tile(eng, torch, case, ph=ph, **kw)
        b = eng.batch([t])
        b.run()
        out.append({k: t[k].cpu().numpy() for k in ("M1", "T", "XYZ1")})
        b.close()
    return out


@pytest.mark.parametrize("dims", [(128, 128, 128), (131, 127, 129)])
@pytest.mark.parametrize("field", [True, False])
def test_reused_block_equals_fresh_memory(dims, field):
    cfg = cases.gre(2, TE=2000, dt=50, P_XY=[[1, 0.5], [0.5, 1]])
    m, f = cases.blocky_phantom(dims, n_labels=2, seed=8)
    other, _ = cases.blocky_phantom(dims, n_labels=2, seed=9)
    case = cases.make_case(cfg, m, f if field else None, 40.0, n_spins=20000)
    fov = np.full(3, 40e-6, np.float32)
    used, fresh = E.Engine(0), E.Engine(0)
    start = _free()
    used.phantom(other, 1.0 - f if field else None, fov, formats=ALL).close()
    kept = _free()
    assert kept <= start - 4 * m.size                    # the block stays: 5 bytes a voxel or more
    ph = used.phantom(case.mask, case.field_T, fov, formats=ALL)
    assert _free() == kept                               # and serves the next phantom
    a = _outputs(used, case, ph)
    b = _outputs(fresh, case, fresh.phantom(case.mask, case.field_T, fov, formats=ALL))
    for x, y in zip(a, b):
        for k in ("M1", "T", "XYZ1"):
            np.testing.assert_array_equal(x[k], y[k])
    used.close()
    fresh.close()
