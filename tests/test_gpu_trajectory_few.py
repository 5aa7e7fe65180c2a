"""Recorded trajectories below the staging line: single walks in single precision take
the general loop, in double precision and in batches the production loop with a store
per step.  They share their positions, so the rows agree word for word, and with the
last position of the same walk without trajectories."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_batch import _tile
from tests.test_gpu_production import run
from spinwalk_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 700, 40000])
@pytest.mark.parametrize("kind", ["walls", "lost", "dummies", "wrap", "no field"])
def test_rows_of_every_loop(engine, kind, n):
    import torch
    kw = dict(lost=dict(MAX_ITERATIONS=0, DIFFUSIVITY=[4e-8, 4e-8]), dummies=dict(DUMMY_SCAN=2),
              wrap=dict(CROSS_FOV=1, P_XY=[[1, 0.5], [0.5, 1]])).get(kind, {})
    m, f = cases.blocky_phantom((20, 18, 22), n_labels=2, seed=4)
    field = None if kind == "no field" else f
    make = lambda rec: cases.make_case(cases.gre(2, TE=650, dt=50, RECORD_TRAJECTORY=rec, **kw), m, field, 20.0, n_spins=n)  # noqa: E731
    case = make(1)
    f32, kahan, f64 = (run(engine, case, precision=p) for p in (E.SW_PREC_F32, E.SW_PREC_F32_KAHAN, E.SW_PREC_F64))
    t = _tile(engine, torch, case)
    b = engine.batch([t])
    b.run()
    for other in (kahan["XYZ1"], f64["XYZ1"], t["XYZ1"].cpu().numpy()):
        np.testing.assert_array_equal(f32["XYZ1"], other)
    np.testing.assert_array_equal(f32["M1"], t["M1"].cpu().numpy())
    np.testing.assert_array_equal(f32["T"], t["T"].cpu().numpy())
    b.close()
    if kind != "lost":                                   # every row is whole: it ends where the walk ends
        np.testing.assert_array_equal(f32["XYZ1"][:, -1], run(engine, make(0))["XYZ1"][:, 0])
