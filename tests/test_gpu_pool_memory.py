"""The memory an engine keeps of dropped phantoms goes back when it is needed: for
any allocation of any engine on the device, for the config driver's buffers, and by
Engine.trim; and a phantom holds little more than its own size."""
import os

import numpy as np
import pytest

from tests import cases
from spinwalk_amd import engine as E
from spinwalk_amd import host as H

pytestmark = pytest.mark.gpu

MB = 1 << 20
SIDE = 352                                  # about 1.0 GiB with float32 records


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _drop(eng, side=SIDE):
    """A phantom made and destroyed; the bytes it held."""
    import torch
    before = _free()
    m = torch.zeros((side,) * 3, dtype=torch.uint8, device="cuda")
    f = torch.zeros((side,) * 3, device="cuda")
    torch.cuda.synchronize()
    held = _free()
    ph = eng.phantom_device(m, f, (side,) * 3, np.full(3, 1e-4, np.float32))
    held -= _free()
    ph.close()
    del m, f
    torch.cuda.empty_cache()
    assert _free() <= before - held + 64 * MB                          # kept
    return held


@pytest.fixture()
def full():
    """Leaves `left` bytes of the device free."""
    import torch
    hogs = []

    def fill(left):
        torch.cuda.empty_cache()
        for _ in range(4):                                             # the first leaves more than it is asked to
            if _free() > left + 32 * MB:
                hogs.append(torch.empty(_free() - left, dtype=torch.uint8, device="cuda"))
        assert _free() <= left + 32 * MB
    yield fill
    hogs.clear()
    torch.cuda.empty_cache()


def _sequence(eng, mb):
    """A sequence whose gradient tables take 4 x mb MB of device memory."""
    m, f = cases.blocky_phantom((4, 4, 4), seed=1)
    case = cases.make_case(cases.gre(2, TE=500, dt=50), m, f, 4.0, n_spins=8)
    n = mb * MB // 4
    tab = dict(case.tables, gradient_t=np.arange(n, dtype=np.int32), gx=np.zeros(n, np.float32))
    tab["gy"] = tab["gz"] = tab["gx"]
    return eng.sequence(case.params, tab)


@pytest.mark.parametrize("who", ["own", "other"])
def test_allocations_that_do_not_fit_beside_it(full, who):
    eng = E.Engine(0)
    held = _drop(eng)
    assert held > 900 * MB
    user = eng if who == "own" else E.Engine(0)
    full(300 * MB)
    _sequence(user, 150).close()                                       # 600 MB
    user.close()
    eng.close()


def test_trim_gives_it_back():
    eng = E.Engine(0)
    before = _free()
    held = _drop(eng)
    eng.trim()
    assert _free() >= before - 64 * MB and held > 900 * MB
    eng.trim()
    _drop(eng)                                                          # and the engine goes on
    eng.close()


def test_a_phantom_does_not_hold_twice_its_size():
    import torch
    eng = E.Engine(0)
    held = _drop(eng)
    m = torch.zeros((288,) * 3, dtype=torch.uint8, device="cuda")       # 0.55 of its voxels
    torch.cuda.synchronize()
    before = _free()
    ph = eng.phantom_device(m, m.float(), (288,) * 3, np.full(3, 1e-4, np.float32))
    eng.trim()                                                          # what it does not use goes back
    del m
    torch.cuda.empty_cache()
    assert _free() >= before + held - 0.6 * held - 64 * MB
    ph.close()
    eng.close()


def test_the_drivers_buffers(full, tmp_path):
    eng = E.Engine(0)
    m, f = cases.blocky_phantom((8, 8, 8), seed=1)
    n = 2000000
    cfg = dict(cases.gre(2, TE=100, dt=50), NUMBER_OF_SPINS=n, SCALE=[1.0, 1.1, 1.2, 1.3, 1.4, 1.5])
    H.write_phantom(os.path.join(tmp_path, "p.h5"), m, f, np.full(3, 8e-6, np.float32))
    cases.write_config(os.path.join(tmp_path, "c.ini"), cfg, ["p.h5"])
    _drop(eng)
    full(200 * MB)
    H.run_config(eng, os.path.join(tmp_path, "c.ini"))                  # 24 + 6 * 25 bytes a spin: 332 MB
    assert H.h5_read(os.path.join(tmp_path, "out", "test_p.h5"), "T", np.uint8).size == 6 * n
    eng.close()
