"""The work that users of this engine have it do, as cases that can be timed.

One case is one pass through a public entry point with what a program would have
in hand before the call.  The kinds:

  walk      one simulation of one phantom (Engine.walk_device, then the echo
            sums): what a program that holds its phantom on the device calls per
            parameter set.  Covers the sequences of the config files (GRE, SE,
            multi-echo SE, bSSFP with dummy scans, stimulated echo, PGSE), the
            precision modes, the field formats, the boundary rules and recorded
            trajectories.
  replay    the same with recorded draw streams, the mode results are validated
            in against another implementation.
  phantom   a new geometry from device arrays (Engine.phantom_device), walked
            once and dropped: a sweep over geometries.
  sweep     one phantom at many FoV scales, GRE and SE each, as one batch.
  cycles    one phantom, one bSSFP scan at four phase-cycling increments, as one
            batch whose tiles share their trajectories.
  hetero    many phantoms of different sizes and kinds, each with GRE, SE or a
            PGSE scan of four b-values, as one batch.
  config    `spinwalk sim -c config.ini`: INI file and HDF5 phantom in, HDF5
            results out.

Sizes come from spinwalk_amd/workloads.py, the tests and the reference's default
configuration (1000 spins where NUMBER_OF_SPINS is not given).  Schedules of
batches are the ones a batch is created with.
"""
from __future__ import annotations

import math
import os
import tempfile

import numpy as np
import torch

from spinwalk_amd import engine as E
from spinwalk_amd import host as H
from spinwalk_amd import workloads as W

PRECISIONS = {"f32": E.SW_PREC_F32, "kahan": E.SW_PREC_F32_KAHAN, "f64": E.SW_PREC_F64}
FIELDS = {"f32": E.SW_FIELD_F32, "f16": E.SW_FIELD_F16, "bf16": E.SW_FIELD_BF16, "q16": E.SW_FIELD_Q16}

_engine = None


def engine():
    """One engine per process, as a program has it."""
    global _engine
    if _engine is None:
        _engine = E.Engine(0)
    return _engine


# ---------------------------------------------------------------------------
# The cases.
# ---------------------------------------------------------------------------
def listed():
    return [
        # A quick look at a geometry: the default number of spins on a small phantom.
        _walk("walk_gre_64_1e3", (64, 64, 64), 1000, "gre", 20000, 50),
        # The CPU-sized simulation that the reference's documentation starts with.
        _walk("walk_gre_100_1e5", (100, 100, 100), 100000, "gre", 20000, 50),
        # A spin echo with permeable vessels and cells, a million spins on a large phantom.
        _walk("walk_se_500_1e6", (500, 500, 500), 1000000, "se", 40000, 20, shapes="mixed", permeable=True),
        # Steady state on a phantom of uneven sides, mixed precision.
        _walk("walk_bssfp_uneven_q16", (301, 257, 199), 300000, "bssfp", 2500, 50, dummies=50, precision="kahan",
              field="q16"),
        # Multi-echo train in double precision, spins wrap at the walls.
        _walk("walk_multiecho_f64", (181, 210, 163), 200000, "mese", 60000, 50, precision="f64", shapes="mixed",
              permeable=True, cross=True),
        # Recorded trajectories.
        _walk("walk_traj_200_1e5", (200, 200, 200), 100000, "gre", 40000, 50, traj=True),
        # Validation against another implementation's draws.
        dict(name="replay_se_40_2e4", kind="replay", nx=40, ny=40, nz=40, spins=20000, seq="se", te_us=20000, dt_us=50,
             precision="f32", permeable=True),
        # A geometry sweep's step.
        dict(name="phantom_gre_256_2e5", kind="phantom", nx=256, ny=256, nz=256, spins=200000, seq="gre",
             te_us=20000, dt_us=50, precision="f32", field="f32", vessels=60),
        # The FoV-scaling sweep: 32 scales, GRE and SE each.
        dict(name="sweep_256_64x1e5", kind="sweep", nx=256, scales=32, spins=100000, precision="f32", field="f32"),
        # Phase-cycled bSSFP on a billion voxels.
        dict(name="cycles_1000_2e6", kind="cycles", nx=1000, spins=2000000, dummies=100, precision="f32", field="f32"),
        # A dozen phantoms of all kinds, mixed precision.
        dict(name="hetero_12_q16", kind="hetero", phantoms=12, largest=320, precision="kahan", field="q16"),
        # The command line's path, files included.
        dict(name="config_gre_100_5scales", kind="config", nx=100, ny=100, nz=100, spins=20000, scales=5, te_us=20000,
             dt_us=50),
    ]


def _walk(name, dims, spins, seq, te_us, dt_us, dummies=0, precision="f32", field="f32", shapes="cylinders",
          permeable=False, cross=False, traj=False, order=True):
    c = dict(kind="walk", nx=dims[0], ny=dims[1], nz=dims[2], spins=spins, seq=seq, te_us=te_us, dt_us=dt_us,
             dummies=dummies, precision=precision, field=field, shapes=shapes, permeable=permeable, cross=cross,
             traj=traj, order=order)
    return dict(c, name=name) if name else c


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["walk"] * 6 + ["replay", "phantom", "sweep", "cycles", "hetero", "config"])
    prec = rng.choice(["f32", "f32", "kahan", "f64"])
    field = "f32" if prec == "f64" else rng.choice(["f32", "f32", "q16", "f16", "bf16"])
    te = rng.choice([10000, 20000, 30000, 40000])
    if kind == "walk":
        side = _log(rng, 48, 420)
        dims = tuple(max(8, int(side * rng.uniform(0.7, 1.3))) for _ in range(3))
        seq = rng.choice(["gre", "se", "mese", "bssfp", "ste", "pgse"])
        traj = rng.random() < 0.12
        spins = _log(rng, 300, 60000 if traj else 1000000)
        return _walk(None, dims, spins, seq, {"bssfp": 2500, "mese": 60000, "pgse": 50000}.get(seq, te),
                     rng.choice([20, 25, 50]), dummies=rng.choice([10, 37, 80]) if seq == "bssfp" else 0, precision=prec,
                     field=field, shapes=rng.choice(["cylinders", "mixed", "axons"]), permeable=rng.random() < 0.5,
                     cross=rng.random() < 0.3, traj=traj, order=rng.random() < 0.85)
    if kind == "replay":
        side = _log(rng, 16, 96)
        return dict(kind=kind, nx=side, ny=side + rng.randint(0, 9), nz=side + rng.randint(0, 9),
                    spins=_log(rng, 500, 20000), seq=rng.choice(["gre", "se"]), te_us=rng.choice([4000, 10000, 20000]),
                    dt_us=50, precision=rng.choice(["f32", "f64"]), permeable=rng.random() < 0.5)
    if kind == "phantom":
        side = _log(rng, 64, 320)
        return dict(kind=kind, nx=side, ny=side + rng.randint(0, 9), nz=side + rng.randint(0, 9),
                    spins=_log(rng, 1000, 300000), seq=rng.choice(["gre", "se"]), te_us=te, dt_us=50, precision=prec,
                    field=field, vessels=rng.randint(20, 80))
    if kind == "sweep":
        return dict(kind=kind, nx=_log(rng, 96, 300), scales=rng.randint(4, 24), spins=_log(rng, 20000, 100000),
                    precision=prec, field=field)
    if kind == "cycles":
        return dict(kind=kind, nx=_log(rng, 200, 700), spins=_log(rng, 200000, 2000000), dummies=rng.choice([20, 50, 100]),
                    precision=rng.choice(["f32", "kahan"]), field=field)
    if kind == "hetero":
        return dict(kind=kind, phantoms=rng.randint(6, 12), largest=rng.choice([192, 256, 320]),
                    precision=rng.choice(["f32", "kahan"]), field=field)
    side = _log(rng, 40, 128)
    return dict(kind=kind, nx=side, ny=side + rng.randint(0, 9), nz=side + rng.randint(0, 9),
                spins=_log(rng, 1000, 50000), scales=rng.randint(1, 8), te_us=te, dt_us=50)


# ---------------------------------------------------------------------------
# Sequences, as the config generator and the config files write them.
# ---------------------------------------------------------------------------
def _cfg(case, n_sub, seed):
    seq, te, dt = case["seq"], case["te_us"], case["dt_us"]
    pxy = np.full((n_sub, n_sub), 0.5) + 0.5 * np.eye(n_sub) if case.get("permeable") else np.eye(n_sub)
    cfg = dict(B0=9.4, SEED=seed, CROSS_FOV=int(case.get("cross", False)),
               RECORD_TRAJECTORY=int(case.get("traj", False)), MAX_ITERATIONS=1e4, DUMMY_SCAN=case.get("dummies", 0),
               LINEAR_PHASE_CYCLING=0.0, QUADRATIC_PHASE_CYCLING=0.0, WHAT_TO_SCALE=0, SCALE=[1.0],
               DIFFUSIVITY=[1e-9] * n_sub, P_XY=pxy.tolist(), NUMBER_OF_SPINS=case["spins"], TIME_STEP=dt,
               T1=[2200.0] + [1600.0] * (n_sub - 1), T2=[41.0] + [20.0] * (n_sub - 1))
    if seq == "gre":
        cfg.update(TR=te + dt, TE=[te], RF_FA=[90.0], RF_PH=[0.0], RF_T=[0])
    elif seq == "se":
        cfg.update(TR=te + dt, TE=[te], RF_FA=[90.0, 180.0], RF_PH=[0.0, 90.0], RF_T=[0, te // 2])
    elif seq == "mese":                     # eight echoes
        esp = te // 8
        cfg.update(TR=te + dt, TE=[esp * (k + 1) for k in range(8)], RF_FA=[90.0] + [180.0] * 8,
                   RF_PH=[0.0] + [90.0] * 8, RF_T=[0] + [esp * k + esp // 2 // dt * dt for k in range(8)])
    elif seq == "bssfp":
        cfg.update(TR=2 * te, TE=[te], RF_FA=[16.0], RF_PH=[0.0], RF_T=[0], LINEAR_PHASE_CYCLING=180.0)
    elif seq == "ste":                      # config/stimulated_echo.ini
        q = te // 4
        cfg.update(TR=te + dt, TE=[q * 2, te], RF_FA=[90.0, 90.0, 90.0], RF_PH=[0.0, 90.0, 90.0], RF_T=[0, q, q * 3],
                   DEPHASING=[360.0, 360.0, 720.0, 360.0],
                   DEPHASING_T=[q // 2, q + q // 2, q * 2 + q // 2, q * 3 + q // 2])
    else:                                   # pgse along y, b = 1000 s/mm^2
        tab = W.pgse_tables(1000.0, (0, 1, 0), 5, 10, 30, dt)
        cfg.update(TR=50000 + dt, TE=[50000], **tab)
    return cfg


def _specs(shapes, seed, side):
    r = max(2.0, min(8.0, side / 20.0))
    if shapes == "cylinders":
        return [W.cylinders(r, 4.0, seed=seed + 1)]
    if shapes == "mixed":
        return [W.cylinders(r, 4.0, seed=seed + 1), W.spheres(max(2.0, 0.6 * r), 2.0, seed=seed + 2)]
    return [W.axons(3.0, 0.5, 45.0, seed=seed + 1)]


def _formats(case):
    return (FIELDS[case["field"]],)


def _case_on(ph, dims, cfg):
    """A prepared case on a phantom that lives on the device."""
    c = E.prepare_case(cfg, np.zeros((1, 1, 1), np.uint8), None, ph.fov_m)
    for i in range(3):
        c.params.phantom_size[i] = dims[i]
    c.params.matrix_length = int(np.prod(dims))
    c.params.fieldmap_exist = 1
    return c


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _buffers(c, p, precision):
    n, te = c.n_spins, c.n_te
    m = torch.float64 if precision == "f64" else torch.float32
    return dict(M1=torch.zeros((n, te, 3), dtype=m, device="cuda"),
                T=torch.zeros((n, te), dtype=torch.uint8, device="cuda"),
                XYZ1=torch.zeros((n, c.traj_len, 3), dtype=torch.float32, device="cuda"),
                sums=torch.zeros((te, p.n_substrate, 3), dtype=torch.float64, device="cuda"))


def _n_sub(case):
    return 3 if case.get("shapes") == "mixed" else 2


# ---------------------------------------------------------------------------
# prepare / run, by kind.
# ---------------------------------------------------------------------------
def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    return globals()["_run_" + state["kind"]](state)


def _prepare_walk(case, seed):
    dims = (case["nx"], case["ny"], case["nz"])
    eng = engine()
    ph, _ = eng.generate_phantom(dims, [float(d) for d in dims], _specs(case["shapes"], 10 * seed, min(dims)),
                                 formats=_formats(case))
    c = _case_on(ph, dims, _cfg(case, _n_sub(case), 1 + seed % 100000))
    p, xs, gs = c.scale_params(1.0)
    s = dict(kind="walk", ph=ph, params=p, seq=eng.sequence(p, c.tables), M0=_dev(c.M0), XYZ0=_dev(c.XYZ0),
             opts=dict(xyz_scale=xs, gradient_scale=gs, precision=PRECISIONS[case["precision"]],
                       field_format=FIELDS[case["field"]], spatial_order=int(case["order"])))
    s.update(_buffers(c, p, case["precision"]))
    return s


def _run_walk(s):
    eng = engine()
    eng.walk_device(s["ph"], s["seq"], s["params"], s["M0"], s["XYZ0"], s["M1"], s["XYZ1"], s["T"], stats=False,
                    **s["opts"])
    eng.echo_reduce(s["M1"], s["T"], s["params"].n_substrate, s["sums"])
    return dict(M1=s["M1"], T=s["T"], XYZ1=s["XYZ1"], sums=s["sums"])


def _vessels(dims, n, seed, device):
    """Mask and field (tesla per 1 T) of n cylinders of random axes, made on the device."""
    rng = np.random.default_rng(seed)
    mask = torch.zeros(dims, dtype=torch.uint8, device=device)
    field = torch.zeros(dims, dtype=torch.float32, device=device)
    ax = [torch.arange(d, device=device, dtype=torch.float32) + 0.5 for d in dims]
    r, k = max(2.0, min(dims) / 32.0), 2.0 * math.pi * 0.3 * 0.11e-6 * 0.4
    for _ in range(n):
        p0, u = rng.uniform(0, 1, 3) * dims, rng.normal(size=3)
        u /= np.linalg.norm(u)
        d = [(ax[i] - p0[i]).reshape([-1 if j == i else 1 for j in range(3)]) for i in range(3)]
        t = d[0] * u[0] + d[1] * u[1] + d[2] * u[2]
        q2 = d[2] - t * u[2]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] - t * t
        st2 = 1.0 - u[2] * u[2]
        inside = r2 <= r * r
        mask[inside] = 1
        out = k * r * r * (2.0 * q2 * q2 / max(st2, 1e-6) / r2.clamp(min=1e-6) - 1.0) * st2 / r2.clamp(min=r * r)
        field += torch.where(inside, torch.full_like(out, k * (u[2] * u[2] - 1.0 / 3.0)), out)
    return mask, field


def _prepare_phantom(case, seed):
    dims = (case["nx"], case["ny"], case["nz"])
    fov = np.asarray(dims, np.float32) * np.float32(1e-6)
    mask, field = _vessels(dims, case["vessels"], seed, "cuda")
    c = E.prepare_case(_cfg(case, 2, 1 + seed % 100000), np.zeros((1, 1, 1), np.uint8), None, fov)
    for i in range(3):
        c.params.phantom_size[i] = dims[i]
    c.params.matrix_length = int(np.prod(dims))
    c.params.fieldmap_exist = 1
    p, xs, gs = c.scale_params(1.0)
    s = dict(kind="phantom", mask=mask, field=field, dims=dims, fov=fov, params=p, formats=_formats(case),
             seq=engine().sequence(p, c.tables), M0=_dev(c.M0), XYZ0=_dev(c.XYZ0),
             opts=dict(xyz_scale=xs, gradient_scale=gs, precision=PRECISIONS[case["precision"]],
                       field_format=FIELDS[case["field"]], spatial_order=1))
    s.update(_buffers(c, p, case["precision"]))
    return s


def _run_phantom(s):
    s["ph"] = engine().phantom_device(s["mask"], s["field"], s["dims"], s["fov"], formats=s["formats"])
    out = _run_walk(s)
    s["ph"].close()
    return out


def _replay_inputs(case, seed):
    """What a replayed simulation is given: phantom, start, draws (host arrays)."""
    dims = (case["nx"], case["ny"], case["nz"])
    rng = np.random.default_rng(seed)
    block = 5
    coarse = rng.random([-(-d // block) for d in dims]) < 0.2
    mask = np.kron(coarse, np.ones((block,) * 3, bool))[:dims[0], :dims[1], :dims[2]].astype(np.uint8)
    field = (rng.normal(size=dims) * 2e-8 + 1e-8 * mask).astype(np.float32)
    fov = np.asarray(dims, np.float32) * np.float32(1e-6)
    cfg = _cfg(case, 2, 1 + seed % 100000)
    n = case["spins"]
    steps = cfg["TR"] // cfg["TIME_STEP"]
    xyz0 = (fov * rng.uniform(0.01, 0.99, (n, 3))).astype(np.float32)
    normals = rng.standard_normal((n, 3 * (2 * steps + 64)), np.float32)
    uniforms = rng.random((n, steps + 64), np.float32)
    return dims, mask, np.ascontiguousarray(field), fov, cfg, xyz0, normals, uniforms


def _prepare_replay(case, seed):
    dims, mask, field, fov, cfg, xyz0, normals, uniforms = _replay_inputs(case, seed)
    eng = engine()
    c = E.prepare_case(cfg, mask, field, fov, XYZ0=xyz0)
    p, xs, gs = c.scale_params(1.0)
    s = dict(kind="walk", ph=eng.phantom(mask, field, fov), params=p, seq=eng.sequence(p, c.tables), M0=_dev(c.M0),
             XYZ0=_dev(c.XYZ0),
             opts=dict(xyz_scale=xs, gradient_scale=gs, precision=PRECISIONS[case["precision"]], rng=E.SW_RNG_REPLAY,
                       replay=(_dev(normals), _dev(uniforms))))
    s.update(_buffers(c, p, case["precision"]))
    return s


def _tile(ph, dims, cfg, case, shared, eng):
    c = _case_on(ph, dims, cfg)
    p, xs, gs = c.scale_params(cfg["SCALE"][0])
    key = (cfg["NUMBER_OF_SPINS"], cfg["SEED"], id(ph))       # tiles of one start share its arrays
    if key not in shared:
        shared[key] = (_dev(c.M0), _dev(c.XYZ0))
    t = dict(phantom=ph, sequence=eng.sequence(p, c.tables), params=p, xyz_scale=xs, gradient_scale=gs,
             precision=PRECISIONS[case["precision"]], field_format=FIELDS[case["field"]], spatial_order=1,
             M0=shared[key][0], XYZ0=shared[key][1])
    b = _buffers(c, p, case["precision"])
    t.update(M1=b["M1"], T=b["T"], XYZ1=b["XYZ1"], echo_sums=b["sums"])
    return t


def _batch_state(tiles):
    return dict(kind="batch", batch=engine().batch(tiles), tiles=tiles)


def _run_batch(s):
    st = s["batch"].run()
    cat = lambda k: torch.cat([t[k].reshape(-1) for t in s["tiles"]])  # noqa: E731
    return dict(M1=cat("M1"), T=cat("T"), XYZ1=cat("XYZ1"), sums=cat("echo_sums"),
                steps=np.asarray([[i["n_steps"], i["n_attempts"], i["n_lost"]] for i in st["items"]], np.int64))


def _sweep_cfgs(case, seed):
    """W.c4 with another number of scales: (sequence, scale) -> configuration."""
    out = []
    scales = np.logspace(math.log10(1 / 8), math.log10(100 / 8), case["scales"])
    for seq, te in (("gre", 20000), ("se", 40000)):
        for sc in scales:
            ideal = (0.3 * sc * 1e-6) ** 2 / 2e-9 * 1e6
            lo, hi = -(-te // 20000), te // 1000
            dt = W._divisor_at_most(te, int(min(max(ideal, lo), hi)), lo)
            cfg = _cfg(dict(case, seq=seq, te_us=te, dt_us=dt), 2, 1 + seed % 100000)
            cfg.update(SCALE=[float(np.float32(sc))], T1=[2200.0, 2200.0], T2=[41.0, 41.0])
            out.append(cfg)
    return out


def _prepare_sweep(case, seed):
    eng, n = engine(), case["nx"]
    ph, _ = eng.generate_phantom((n,) * 3, (float(n),) * 3, [W.cylinders(max(2.0, n / 32.0), 4.0, seed=10 * seed + 4)],
                                 formats=_formats(case))
    shared = {}
    return _batch_state([_tile(ph, (n,) * 3, cfg, case, shared, eng) for cfg in _sweep_cfgs(case, seed)])


def _prepare_cycles(case, seed):
    eng, n = engine(), case["nx"]
    ph, _ = eng.generate_phantom((n,) * 3, (float(n),) * 3, [W.cylinders(5.0, 4.0, seed=10 * seed + 3)],
                                 formats=_formats(case))
    shared, tiles = {}, []
    for k in range(4):
        cfg = _cfg(dict(case, seq="bssfp", te_us=2500, dt_us=50), 2, 1 + seed % 100000)
        cfg.update(LINEAR_PHASE_CYCLING=90.0, WHAT_TO_SCALE=2, SCALE=[float(k)], T1=[2200.0, 2200.0], T2=[41.0, 41.0])
        tiles.append(_tile(ph, (n,) * 3, cfg, case, shared, eng))
    return _batch_state(tiles)


def _hetero_plan(case, seed):
    """(side, shapes, seq, spins) of each phantom, from the seed; the sizes of one
    case do not depend on it, so that passes of two seeds are alike."""
    rng = np.random.default_rng(case["phantoms"] * 1000 + case["largest"])
    sides = [s for s in (128, 160, 192, 256, 320) if s <= case["largest"]]
    return [(int(rng.choice(sides)), ("cylinders", "spheres", "axons")[i % 3], ("gre", "pgse", "se", "pgse")[i % 4],
             int(round(10 ** rng.uniform(4.0, 5.5)))) for i in range(case["phantoms"])]


def _prepare_hetero(case, seed):
    eng, shared, tiles = engine(), {}, []
    for i, (n, shape, seq, spins) in enumerate(_hetero_plan(case, seed)):
        sd = 1000 * (seed % 100000) + i
        spec = {"cylinders": lambda: W.cylinders(4.0, 4.0, seed=sd), "axons": lambda: W.axons(3.0, 0.5, 45.0, seed=sd),
                "spheres": lambda: W.spheres(3.0, 4.0, seed=sd, label=1)}[shape]()
        ph, _ = eng.generate_phantom((n,) * 3, (float(n),) * 3, [spec], formats=_formats(case))
        for b in (1000.0, 0.0, 2000.0, 3000.0) if seq == "pgse" else (1000.0,):
            cfg = _cfg(dict(seq=seq, te_us=20000 if seq == "gre" else 40000, dt_us=50, spins=spins, permeable=True), 2,
                       1 + sd % 1000000)
            cfg.update(T1=[2200.0, 2200.0], T2=[41.0, 41.0])
            if seq == "pgse":               # b-values as gradient scales of the first
                cfg.update(WHAT_TO_SCALE=1, SCALE=[float(np.float32(math.sqrt(b / 1000.0)))])
            tiles.append(_tile(ph, (n,) * 3, cfg, case, shared, eng))
    return _batch_state(tiles)


def _prepare_config(case, seed):
    dims = (case["nx"], case["ny"], case["nz"])
    tmp = tempfile.TemporaryDirectory(prefix="spinwalk_case_")
    mask, field = _vessels(dims, 12, seed, "cuda")
    H.write_phantom(os.path.join(tmp.name, "ph.h5"), mask.cpu().numpy(), field.cpu().numpy(),
                    np.asarray(dims, np.float32) * np.float32(1e-6))
    cfg = _cfg(dict(case, seq="gre"), 2, 1 + seed % 100000)
    tissue = {}
    for i in range(2):
        tissue[f"DIFFUSIVITY[{i}]"] = cfg["DIFFUSIVITY"][i]
        tissue[f"P_XY[{i}]"] = [float(x) for x in cfg["P_XY"][i]]
        tissue[f"T1[{i}]"], tissue[f"T2[{i}]"] = cfg["T1"][i], cfg["T2"][i]
    scan = {k: cfg[k] for k in ("TR", "TE", "RF_FA", "RF_PH", "RF_T", "TIME_STEP", "DUMMY_SCAN")}
    sim = {k: cfg[k] for k in ("B0", "SEED", "NUMBER_OF_SPINS", "CROSS_FOV", "RECORD_TRAJECTORY", "MAX_ITERATIONS",
                               "WHAT_TO_SCALE")}
    for i in range(case["scales"]):
        sim[f"SCALE[{i}]"] = 1.0 + 0.25 * i
    ini = os.path.join(tmp.name, "gre.ini")
    H.write_ini(ini, {"GENERAL": {"SEQ_NAME": "gre"}, "FILES": {"OUTPUT_DIR": "out", "PHANTOM[0]": "ph.h5"},
                      "TISSUE_PARAMETERS": tissue, "SCAN_PARAMETERS": scan, "SIMULATION_PARAMETERS": sim})
    return dict(kind="config", tmp=tmp, ini=ini, out=os.path.join(tmp.name, "out", "gre_ph.h5"))


def _run_config(s):
    H.run_config(engine(), s["ini"])
    return dict(M=H.h5_read(s["out"], "M"), T=H.h5_read(s["out"], "T", np.uint8), XYZ=H.h5_read(s["out"], "XYZ"))


# ---------------------------------------------------------------------------
# What a pass cannot do without.
# ---------------------------------------------------------------------------
# Operations of one production step: Philox4x32-10 (10 rounds of two 32 x 32 -> 64
# products, as 4 multiplications, and 4 XORs), the Box-Muller transform (18), the
# move (6), the voxel index (8) and the phase (2).  A replayed step has no draw.
STEP_OPS, REPLAY_OPS = 114, 16


def work(case):
    if case["kind"] == "walk" or case["kind"] == "phantom":
        w = _walk_work(case, _cfg(case, _n_sub(case), 1))
        if case["kind"] == "phantom":
            w["bytes"] += 5 * case["nx"] * case["ny"] * case["nz"]
        return w
    if case["kind"] == "replay":
        cfg = _cfg(case, 2, 1)
        w = _walk_work(dict(case, field="f32"), cfg, REPLAY_OPS)
        w["bytes"] += 12 * case["spins"] * (cfg["TR"] // cfg["TIME_STEP"])
        return w
    if case["kind"] == "config":
        w = _walk_work(dict(case, field="f32"), _cfg(dict(case, seq="gre"), 2, 1))
        return dict(bytes=w["bytes"] * case["scales"], flops=w["flops"] * case["scales"])
    cfgs = []
    if case["kind"] == "sweep":
        cfgs = [(case["nx"], cfg, 1.0, 0 if i else 1) for i, cfg in enumerate(_sweep_cfgs(case, 1))]
    elif case["kind"] == "cycles":
        cfg = _cfg(dict(case, seq="bssfp", te_us=2500, dt_us=50), 2, 1)
        cfgs = [(case["nx"], cfg, 0.02 if k else 1.0, 0 if k else 1) for k in range(4)]   # one walk serves four
    else:
        for n, _, seq, spins in _hetero_plan(case, 1):
            c = dict(seq=seq, te_us=20000 if seq == "gre" else 40000, dt_us=50, spins=spins)
            for k in range(4 if seq == "pgse" else 1):
                cfgs.append((n, _cfg(c, 2, 1), 0.02 if k else 1.0, 0 if k else 1))
    tot = dict(bytes=0.0, flops=0.0)
    for n, cfg, share, ph in cfgs:
        w = _walk_work(dict(nx=n if ph else 0, ny=n, nz=n, field=case["field"], precision=case["precision"],
                            spins=cfg["NUMBER_OF_SPINS"]), cfg)
        tot["bytes"] += w["bytes"]
        tot["flops"] += w["flops"] * share
    return tot


def _walk_work(case, cfg, ops=STEP_OPS):
    """One walk: the phantom's voxels and the spins' start read once, the results
    written once; the operations of every step."""
    n, te = case["spins"], len(cfg["TE"])
    steps = (cfg["DUMMY_SCAN"] + 1) * (cfg["TR"] // cfg["TIME_STEP"])
    vox = case["nx"] * case["ny"] * case["nz"] * (1 + (4 if case.get("field", "f32") == "f32" else 2))
    m1 = 24 if case.get("precision") == "f64" else 12
    xyz1 = 12 * steps if cfg["RECORD_TRAJECTORY"] else 12
    gathers = n * steps * 5                 # no more voxels than steps are read
    return dict(bytes=float(min(vox, gathers) + n * (24 + te * (m1 + 1) + xyz1)), flops=float(n * steps * ops))


# ---------------------------------------------------------------------------
# 64-bit values.
# ---------------------------------------------------------------------------
def exact(case, seed):
    """A replayed walk's trajectories are double arithmetic on given draws, so its
    results can be formed here; the other kinds draw in the kernel."""
    if case["kind"] != "replay":
        return None
    dims, mask, field, fov, cfg, xyz0, normals, uniforms = _replay_inputs(case, seed)
    n, dt = case["spins"], cfg["TIME_STEP"]
    nt = cfg["TR"] // dt
    f = [float(x) for x in fov]
    lab, fld = mask.ravel(), field.ravel().astype(np.float64)
    to_deg = np.float64(np.float32(9.4)) * dt * 1e-6 * 267515315.0 * 57.2957795130823
    step = 1e-3 * np.sqrt(2.0 * np.float64(np.float32(1e-9)) * dt)
    pxy = np.asarray(cfg["P_XY"], np.float32)
    T1, T2 = (np.asarray(cfg[k], np.float64) * 1e-3 for k in ("T1", "T2"))
    x = xyz0.astype(np.float64)
    M = np.tile(np.asarray([0.0, 0.0, 1.0]), (n, 1))
    s2g = np.asarray([dims[i] / f[i] for i in range(3)])

    def locate(p):
        j = (p * s2g).astype(np.int64)
        ind = (j[:, 0] * dims[1] + j[:, 1]) * dims[2] + j[:, 2]
        return ind

    def rot(M, fa, ph):
        """Flip by fa about the axis at angle ph in the transverse plane."""
        s, c, sp, cp = (fn(math.radians(a)) for a, fn in ((fa, math.sin), (fa, math.cos), (ph, math.sin), (ph, math.cos)))
        a, b = cp * M[:, 0] + sp * M[:, 1], -sp * M[:, 0] + cp * M[:, 1]
        b, z = c * b - s * M[:, 2], s * b + c * M[:, 2]
        return np.stack([cp * a - sp * b, sp * a + cp * b, z], 1)

    def relax(M, deg, t, lb):
        s, c = np.sin(np.radians(deg)), np.cos(np.radians(deg))
        e1, e2 = np.exp(-t / T1[lb]), np.exp(-t / T2[lb])
        return np.stack([(c * M[:, 0] - s * M[:, 1]) * e2, (s * M[:, 0] + c * M[:, 1]) * e2, 1.0 + e1 * (M[:, 2] - 1.0)], 1)

    label = lab[locate(x)].astype(np.int64)
    M = rot(M, cfg["RF_FA"][0], cfg["RF_PH"][0])
    rf = {t // dt: k for k, t in enumerate(cfg["RF_T"]) if k}
    te = {t // dt: k for k, t in enumerate(cfg["TE"])}
    phase, old = np.zeros(n), 0
    jn, ju = np.zeros(n, np.int64), np.zeros(n, np.int64)
    out_M, out_T = np.zeros((n, len(te), 3)), np.zeros((n, len(te)), np.int64)
    for t in range(nt):
        todo = np.arange(n)
        while todo.size:                     # a rejected spin tries again
            rw = normals[todo[:, None], jn[todo][:, None] + np.arange(3)].astype(np.float64) * step
            jn[todo] += 3
            p = x[todo] + rw
            p = np.where(p < 0, p + 2 * np.abs(rw), np.where(p >= f, p - 2 * np.abs(rw), p))
            ind = locate(p)
            to = lab[ind].astype(np.int64)
            change = to != label[todo]
            ok = np.ones(todo.size, bool)
            c = todo[change]
            ok[change] = uniforms[c, ju[c]] < pxy[label[c], to[change]]
            ju[c] += 1
            good = todo[ok]
            x[good], label[good] = p[ok], to[ok]
            phase[good] += fld[ind[ok]] * to_deg
            todo = todo[~ok]
        if t in rf:
            M = rot(relax(M, phase, (t - old) * dt * 1e-6, label), cfg["RF_FA"][rf[t]], cfg["RF_PH"][rf[t]])
            phase[:], old = 0.0, t
        if t in te:
            M = relax(M, phase, (t - old) * dt * 1e-6, label)
            out_M[:, te[t]], out_T[:, te[t]] = M, label
            phase[:], old = 0.0, t
    sums = np.zeros((len(te), 2, 3))
    for k in range(len(te)):
        for lb in range(2):
            at = out_T[:, k] == lb
            sums[k, lb] = out_M[at, k, 0].sum(), out_M[at, k, 1].sum(), at.sum()
    return dict(M1=out_M, T=None, XYZ1=x[:, None, :], sums=sums)
