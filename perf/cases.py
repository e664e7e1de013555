"""Workloads of the time loop, the adjoint and the set-up, as a user's
program runs them through the Python binding, for timing and for comparing
results.

``listed()`` names the workloads, ``draw(rng)`` gives others of the same
ranges, ``prepare`` makes what a program holds before the call (inputs from
the seed, a loaded context), ``run`` is one pass, ``work`` the bytes and
operations one pass cannot do without, and ``exact`` the same results in 64
bits by plain torch and numpy.

A pass of a time-stepping case runs its steps again on the fields the last
pass left, with the sources firing again, as a program that steps a run block
by block does.
"""
import gc
import math

import numpy as np
import torch

from openswpc_amd import gpu
from openswpc_amd.host import ModelSpec, make_simulation_device

UC = 1e-15          # the seismogram unit factor of moment-tensor runs
FIELD_CELLS = 4_000_000   # runs up to this many cells also return their velocity fields
ARENA_BYTES = 44 << 30    # device memory kept per HBM region for the contexts' per-cell arrays


def listed():
    return [
        # the reference's main loop calling the library routine by routine on the
        # smallest grids users start with (a smoke run, a teaching example): the
        # calls themselves and their launches are what counts
        dict(name="routines_small", kind="routines", nx=48, ny=44, nz=40, na=8, nm=3, steps=20),
        # the plain 128^3 example, stepped in graph blocks, velocity sections and 16 stations
        dict(name="plain_128", kind="run", nx=128, ny=128, nz=128, na=20, nm=3, abc="pml", force=False, stations=16,
             sections=True, steps=400, block=100),
        # a run with the Cerjan sponge and a single force, on a grid no tile divides
        dict(name="cerjan_ragged", kind="run", nx=181, ny=149, nz=117, na=12, nm=1, abc="cerjan", force=True,
             stations=12, sections=False, steps=100, block=20),
        # an elastic run of the size the adjoint workload uses: making synthetic data
        dict(name="elastic_256", kind="run", nx=256, ny=256, nz=192, na=20, nm=0, abc="pml", force=False, stations=64,
             sections=False, steps=100, block=50),
        # a regional viscoelastic run with sections
        dict(name="regional_384", kind="run", nx=384, ny=384, nz=256, na=20, nm=3, abc="pml", force=False,
             stations=128, sections=True, steps=40, block=20),
        # a production run: random medium built on the device, a finite fault, many stations
        dict(name="production", kind="production", nx=768, ny=768, nz=448, na=20, nm=3, stations=256, steps=10,
             block=10),
        # batched Green's functions: uneven members stepped together, autotuned
        dict(name="batch_greens", kind="batch", members=12, low=96, high=256, na=10, nm=2, steps=40),
        # reciprocity Green's functions at many cells
        dict(name="reciprocity", kind="green", nx=168, ny=152, nz=120, na=10, nm=2, points=4096, steps=60, block=20),
        # full-waveform gradient, elastic, single-level checkpoints
        dict(name="adjoint_elastic", kind="adjoint", nx=256, ny=256, nz=192, na=20, nm=0, stations=64, sources=1,
             steps=80, outer=20, inner=20),
        # viscoelastic gradient of two sources summed on the device, two-level checkpoints
        dict(name="adjoint_visco", kind="adjoint", nx=176, ny=160, nz=128, na=20, nm=3, stations=96, sources=2,
             steps=60, outer=30, inner=10),
        # set-up of a heterogeneous run: a random medium and the layered model on the device
        dict(name="medium_setup", kind="medium", nx=256, ny=250, nz=186, na=20, nm=3),
        # one random medium into host memory
        dict(name="random_medium", kind="rmedia", n1=198, n2=262, n3=262, ptype="vonkarman"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["routines", "run", "run", "run", "production", "batch", "green", "adjoint", "adjoint", "medium",
                       "rmedia"])
    if kind == "routines":
        na = rng.randint(5, 10)
        return dict(kind=kind, nx=size(32, 72), ny=size(32, 72), nz=size(28, 60), na=na, nm=rng.choice([0, 1, 2, 3]),
                    steps=rng.randint(10, 24))
    if kind == "run":
        nx, ny, nz = size(64, 400), size(64, 400), size(56, 260)
        abc = rng.choice(["pml", "pml", "pml", "cerjan"])
        steps = max(20, min(300, int(1.0e9 / (nx * ny * nz))))
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, na=rng.randint(8, 20), nm=rng.choice([0, 1, 2, 3, 3]), abc=abc,
                    force=rng.random() < 0.3, stations=rng.randint(4, 160), sections=rng.random() < 0.5, steps=steps,
                    block=rng.choice([10, 20]))
    if kind == "production":
        return dict(kind=kind, nx=size(400, 760), ny=size(400, 760), nz=size(240, 440), na=20, nm=3,
                    stations=rng.randint(32, 256), steps=10, block=rng.choice([5, 10]))
    if kind == "batch":
        low = rng.randint(64, 120)
        return dict(kind=kind, members=rng.randint(4, 14), low=low, high=rng.randint(low + 20, 240),
                    na=rng.randint(8, 14), nm=rng.choice([1, 2, 3]), steps=rng.randint(30, 50))
    if kind == "green":
        return dict(kind=kind, nx=size(96, 220), ny=size(96, 220), nz=size(80, 150), na=rng.randint(8, 16),
                    nm=rng.choice([0, 2, 3]), points=size(64, 8192), steps=rng.randint(30, 80), block=10)
    if kind == "adjoint":
        nm = rng.choice([0, 0, 2, 3])
        steps = rng.randint(40, 64)
        outer = rng.randint(12, 32)
        return dict(kind=kind, nx=size(80, 240), ny=size(80, 240), nz=size(64, 170), na=rng.randint(10, 20), nm=nm,
                    stations=rng.randint(4, 128), sources=rng.randint(1, 2), steps=steps, outer=outer,
                    inner=rng.randint(4, outer))
    if kind == "medium":
        return dict(kind=kind, nx=size(96, 256), ny=size(96, 256), nz=size(64, 200), na=rng.randint(8, 20),
                    nm=rng.choice([0, 2, 3]))
    return dict(kind=kind, n1=size(64, 210), n2=size(64, 270), n3=size(64, 270),
                ptype=rng.choice(["gauss", "exp", "vonkarman"]))


# ---------------------------------------------------------------------------
# inputs (float32, as the reference's modules hold them; arrays in its (k,i,j)
# halo order, k fastest)
# ---------------------------------------------------------------------------
DX = 0.5


def _clamp(n, na, beg):
    """cells -2..n+3 of an axis with the absorber's cells replaced by the nearest interior one"""
    return np.clip(np.arange(-2, n + 4), (na + 1) if beg else 1, n - na)


def _medium(nx, ny, nz, na, nm, rng, abc):
    """Three layers under 3-6 planes of air with gentle topography, velocities
    perturbed by a few per cent, relaxed moduli and tau-method strengths; the
    2nd-order band limits around the free surface."""
    w = na if abc == "pml" else 0
    ci, cj, ck = _clamp(nx, w, True), _clamp(ny, w, True), _clamp(nz, w, False)
    ph = rng.uniform(0, 2 * np.pi, 6).astype(np.float32)
    kx, ky, kz = (2 * np.pi * rng.uniform(1.0, 4.0, 3) / np.array([nx, ny, nz])).astype(np.float32)
    wx, wy = np.sin(kx * ci + ph[0]), np.sin(ky * cj + ph[1])
    ksurf = np.rint(4.0 + 1.2 * wx[None, :] * wy[:, None]).astype(np.int32)      # last plane of air
    tops = np.sort(rng.uniform(0.15, 0.75, 2)) * nz
    layer = (ck[None, :] > tops[:, None]).sum(0)
    vs = (np.array([2.6, 3.2, 3.8]) * rng.uniform(0.95, 1.05))[layer].astype(np.float32)
    rho1 = np.array([2.4, 2.6, 2.9], np.float32)[layer]
    q1 = (50.0 * vs).astype(np.float32)
    shp = (ny + 6, nx + 6, nz + 6)
    pert = (1.0 + 0.03 * np.sin(kx * ci + ph[2])[None, :, None] * np.sin(ky * cj + ph[3])[:, None, None]
            * np.sin(kz * ck + ph[4])[None, None, :]).astype(np.float32)
    solid = (ck[None, None, :] > ksurf[:, :, None])
    rho = np.where(solid, rho1 * pert, np.float32(0.001)).astype(np.float32)
    mu = np.where(solid, rho * np.square(vs * pert), np.float32(0)).astype(np.float32)
    lam = mu.copy()                                       # Vp = sqrt(3) Vs
    taus = np.broadcast_to((nm * 1.6 / np.maximum(q1, 1)).astype(np.float32), shp).copy()
    taup = (taus * np.float32(0.5)).astype(np.float32)
    if nm:
        mu *= np.float32(0.99)
        lam *= np.float32(0.99)
    lo, hi = ksurf.copy(), ksurf.copy()
    for dj in range(-2, 4):
        for di in range(-2, 4):
            s = ksurf[np.clip(np.arange(ny + 6) + dj, 0, ny + 5)][:, np.clip(np.arange(nx + 6) + di, 0, nx + 5)]
            np.minimum(lo, s, out=lo)
            np.maximum(hi, s, out=hi)
    top, bot = np.maximum(lo - 2, 1).astype(np.int32), np.minimum(hi + 2, nz).astype(np.int32)
    return dict(rho=rho, lam=lam, mu=mu, taup=taup, taus=taus, kfs_top=top, kfs_bot=bot, kob_top=top, kob_bot=bot,
                kob=ksurf)


def _visco(nm, dt):
    ts = np.array([1.0 / (2 * np.pi * 0.05 * 100.0 ** (m / max(nm - 1, 1))) for m in range(nm)])
    if nm == 1:
        ts = np.array([1.0 / (2 * np.pi * 0.5)])
    f32 = np.float32
    c1, c2 = (2 * ts - dt) / (2 * ts + dt), 2 / (2 * ts + dt) / max(nm, 1)
    d1, d2 = 2 * ts / (2 * ts - dt), float(f32(np.sum(dt / (2 * ts - dt)) / max(nm, 1)))
    pad = np.zeros(0 if nm else 1)
    return dict(c1=np.append(c1, pad).astype(f32), c2=np.append(c2, pad).astype(f32),
                d1=np.append(d1, pad).astype(f32), d2=d2 if nm else 0.0)


def _pml(n, na, h, dt, edge):
    """(n, 4) ADE-CFS damping profile at cell centres or edges"""
    x = (np.arange(1, n + 1) - 0.5 + (0.5 if edge else 0.0)) * h
    hh = na * h
    r = np.where(x <= hh, hh - x, np.where(x >= n * h - hh, x - (n * h - hh), 0.0))
    r = np.abs(r / hh)
    r0 = 10 ** (-(np.log10(na) - 1) / np.log10(2.0) - 3.0)
    d, a, b = -(6.0 / hh) * np.log(r0) * r, np.pi * (1 - r), 1 + 6 * r ** 2
    den = 1 + dt / 2 * (a + d / b)
    return np.stack([(1 + dt / 2 * a) / b / den, -1 / b / den, (1 - dt / 2 * (a + d / b)) / den, d / b / den],
                    1).astype(np.float32)


def _cerjan(n, na, edge, low):
    i = np.arange(-2, n + 4) + (0.5 if edge else 0.0)
    d = np.minimum(i - 0.5 if low else np.full(n + 6, 1e9), n + 0.5 - i)
    d = np.clip(d / na, 0, 1)
    return np.exp(-0.09 * (1 - d) ** 2).astype(np.float32)


def _wavelet(nt, dt, tr, shift):
    t = (np.arange(1, nt + 1) - shift) * dt
    s = np.where((t >= 0) & (t <= tr), 3 * np.pi / (4 * tr) * np.sin(np.pi * np.clip(t, 0, tr) / tr) ** 3, 0.0)
    return s.astype(np.float32)


def _inputs(case, seed):
    """kernel inputs of one simulation and the absorber's profiles"""
    rng = np.random.default_rng(seed)
    nx, ny, nz, na, nm = (case[k] for k in ("nx", "ny", "nz", "na", "nm"))
    abc, steps = case.get("abc", "pml"), case["steps"]
    vmax = 3.8 * 1.05 * 1.03 * math.sqrt(3)
    dt = float(np.float32(0.75 * 6 / 7 * DX / math.sqrt(3) / vmax))
    inp = dict(nx=nx, ny=ny, nz=nz, na=na, nm=nm, abc=abc, dt=dt, steps=steps,
               medium=_medium(nx, ny, nz, na, nm, rng, abc), visco=_visco(nm, dt))
    if abc == "pml":
        inp["absorb"] = [_pml(n, na, DX, dt, e) for n in (nx, ny, nz) for e in (False, True)]
    else:
        inp["absorb"] = [_cerjan(n, na, e, low) for n, low in ((nx, True), (ny, True), (nz, False))
                         for e in (False, True)]
    # a source per two million cells (a finite fault on the larger grids): every other one a few cells under the
    # surface, all of an inversion's within 20 cells of it
    nsrc = max(1, nx * ny * nz // 2_000_000)
    force, survey = bool(case.get("force", False)), case.get("kind") == "adjoint"
    lo, hi = na + 4, np.array([nx, ny, nz]) - na - 4
    kob = inp["medium"]["kob"]
    inp["shots"] = []
    for _ in range(case.get("sources", 1)):
        shot = dict(i=rng.integers(min(lo, hi[0] - 1), hi[0], nsrc), j=rng.integers(min(lo, hi[1] - 1), hi[1], nsrc),
                    k=rng.integers(min(12, hi[2] - 1), min(24, hi[2]) if survey else hi[2], nsrc),
                    mo=rng.uniform(0.5, 1.5, nsrc).astype(np.float32) * 1e15)
        if not survey:
            shot["k"][::2] = (kob[shot["j"] + 2, shot["i"] + 2] + rng.integers(2, 8, nsrc))[::2]
        shot["comp"] = rng.normal(size=(3 if force else 6, nsrc)).astype(np.float32)
        shot["M0"] = float(np.sum(shot["mo"], dtype=np.float32)) if not force else 1.0
        shot["stf"] = np.stack([_wavelet(steps, dt, float(tr), 0.0 if force else 0.5)
                                for tr in rng.uniform(8 * dt, 16 * dt, nsrc)], 1)
        nst = case.get("stations", 8)
        shot["ist"], shot["jst"] = rng.integers(4, nx - 3, nst), rng.integers(4, ny - 3, nst)
        # stations the waves reach within the steps of a pass: all of an inversion's, half of the others'
        near, some = rng.integers(0, (nsrc + 1) // 2, nst) * (1 if survey else 2), slice(None, None, 1 if survey else 2)
        near, reach = np.minimum(near, nsrc - 1), 14 if survey else 5
        shot["ist"][some] = np.clip(shot["i"][near] + rng.integers(-reach, reach + 1, nst), 4, nx - 4)[some]
        shot["jst"][some] = np.clip(shot["j"][near] + rng.integers(-reach, reach + 1, nst), 4, ny - 4)[some]
        shot["kst"] = kob[shot["jst"] + 2, shot["ist"] + 2] + 1
        # recorded data of an inversion: band-limited traces about as strong as the synthetic ones
        t = np.arange(steps) * dt
        ph, fr = rng.uniform(0, 6.28, (2, nst, 3, 1)), rng.uniform(0.3, 2.0, (nst, 3, 1))
        amp = shot["M0"] * UC * 1e9 * 3e-5
        shot["obs"] = (amp * np.sin(6.28 * fr * t + ph[0]) * (t / t[-1])).astype(np.float32)
        inp["shots"].append(shot)
    inp["force"] = force
    return inp


def _arena():
    """the striped device arena that a program with large runs reserves once"""
    if gpu.stripe_free_bytes(0, 0) == 0:
        gpu.stripe_reserve(ARENA_BYTES)


def _load(inp, what=1, record=True):
    sim = gpu.SwpcGPU(inp["nx"], inp["ny"], inp["nz"], inp["na"], inp["nm"], inp["abc"], DX, DX, DX, inp["dt"])
    m, v = inp["medium"], inp["visco"]
    sim.set_medium(*(m[k] for k in gpu.SwpcGPU.MEDIUM))
    sim.set_visco(v["c1"], v["c2"], v["d1"], v["d2"])
    (sim.set_pml if inp["abc"] == "pml" else sim.set_cerjan)(*inp["absorb"])
    _shot(sim, inp, inp["shots"][0], what, record)
    return sim


def _shot(sim, inp, s, what=1, record=True):
    if record:
        sim.set_sources(s["i"], s["j"], s["k"], s["mo"], s["comp"], s["M0"], s["stf"], bf_mode=inp["force"])
        sim.set_receivers(s["ist"], s["jst"], s["kst"], what, 1, inp["steps"], s["M0"], UC)


SECTIONS = ("xy_v", "yz_v", "xz_v", "fs_v", "fs_u", "xz_ps")


def _every(case):
    return max(1, case["steps"] // 4)


class _Run:
    """what a program keeps between passes"""

    def __init__(self, **kw):
        self.__dict__.update(kw)


def prepare(case, seed):
    gc.collect()
    kind = case["kind"]
    if kind == "rmedia":
        return _Run(kind=kind, seed=seed, case=case)
    _arena()
    if kind == "medium":
        sim = gpu.SwpcGPU(case["nx"], case["ny"], case["nz"], case["na"], case["nm"], "pml", DX, DX, DX, 0.02)
        return _Run(kind=kind, seed=seed, case=case, sim=sim, **_profile(case, seed))
    if kind == "production":
        return _Run(kind=kind, case=case, sim=_production(case, seed))
    if kind == "batch":
        sims = [_load(_inputs(c, s)) for c, s in _members(case, seed)]
        batch = gpu.SwpcBatch(sims)
        batch.tune(1)
        return _Run(kind=kind, case=case, sims=sims, batch=batch)
    inp = _inputs(case, seed)
    if kind == "green":
        sim = _load(inp, record=False)
        p = _green_points(case, seed, inp)
        sim.set_green(p["i"], p["j"], p["k"], *p["src"], "z", True, 1, case["steps"], p["stf"])
        return _Run(kind=kind, case=case, sim=sim)
    sim = _load(inp, what=15 if kind == "routines" else 1)
    if case.get("sections"):
        sim.set_snapshots(SECTIONS, inp["medium"]["kob"], k0_xy=8, i0_yz=inp["nx"] // 2, j0_xz=inp["ny"] // 2,
                          idec=2, jdec=2, kdec=2, ntdec_s=_every(case), nframe=4 + 1, M0=inp["shots"][0]["M0"], UC=UC)
    return _Run(kind=kind, case=case, sim=sim, inp=inp)


def run(state):
    return _PASS[state.kind](state, state.case)


def _pass_routines(state, case):
    sim = state.sim
    for it in range(1, case["steps"] + 1):      # src/swpc_3d/main.f90:119-139
        sim.wav_store(it)
        sim.kernel_update_stress()
        sim.absorb_update_stress()
        sim.source_stressglut(it)
        sim.kernel_update_vel()
        sim.absorb_update_vel()
        sim.source_bodyforce(it)
    return {"vmax": sim.kernel_vmax(), **{k: sim.seismograms(k) for k in ("vel", "disp", "stress", "strain")}}


def _pass_run(state, case):
    sim = state.sim
    sim.step(1, case["steps"], use_graph=True, block=case["block"])
    out = {"vel": sim.seismograms("vel")}
    if case.get("sections"):
        for name in SECTIONS:
            out[name] = sim.snapshot(name, 3)
        out["fs_v_max"] = sim.snap_max("fs_v")
    if case["nx"] * case["ny"] * case["nz"] <= FIELD_CELLS:
        for q in ("Vx", "Vy", "Vz"):
            out[q] = sim.get_field(q)
    return out


def _pass_production(state, case):
    sim = state.sim
    sim.step(1, case["steps"], use_graph=True, block=case["block"])
    return {"vel": sim.seismograms("vel"), **{q: sim.snapshot(q, 1) for q in ("yz_v", "xz_v", "fs_v")}}


def _pass_batch(state, case):
    state.batch.step(1, case["steps"], use_graph=True, block=case["steps"])
    state.batch.synchronize()
    return [s.seismograms("vel") for s in state.sims]


def _pass_green(state, case):
    state.sim.step(1, case["steps"], use_graph=True, block=case["block"])
    return {"gf": state.sim.green()}


def _pass_adjoint(state, case):
    sim, inp = state.sim, state.inp
    if case["sources"] == 1:
        J, gl, gm, gr = sim.adjoint_gradient(case["steps"], inp["shots"][0]["obs"], ckp=case["outer"])
        return {"misfit": J, "lam": gl, "mu": gm, "rho": gr}
    sim.adjoint_reset()
    J = []
    for s in inp["shots"]:
        _shot(sim, inp, s)
        J.append(sim.adjoint_accumulate(case["steps"], s["obs"], case["outer"], case["inner"]))
    gl, gm, gr = sim.adjoint_sums()
    return {"misfit": J, "lam": gl, "mu": gm, "rho": gr}


def _pass_medium(state, case):
    sim = state.sim
    ptr, _ = sim.staging_buffer()
    gpu.rmedia_3d("vonkarman", (case["nz"] + 6, case["nx"] + 6, case["ny"] + 6), (DX,) * 3, (5.0,) * 3, 0.05,
                  kappa=0.5, seed=state.seed, out_ptr=ptr)
    kfs, kob, vr = sim.medium_layered(state.prof, ptr, state.clip, state.tau)
    return {"kfs": kfs, "kob": kob, "vrange": vr, "lam": sim.get_medium("lam"), "mu": sim.get_medium("mu")}


def _pass_rmedia(state, case):
    return {"xi": gpu.rmedia_3d(case["ptype"], (case["n1"], case["n2"], case["n3"]), (DX,) * 3, (4.0, 5.0, 6.0), 0.05,
                                kappa=0.5, seed=state.seed)}


_PASS = dict(routines=_pass_routines, run=_pass_run, production=_pass_production, batch=_pass_batch,
             green=_pass_green, adjoint=_pass_adjoint, medium=_pass_medium, rmedia=_pass_rmedia)


def _production(case, seed):
    rng = np.random.default_rng(seed)
    nx, ny, nz, h = case["nx"], case["ny"], case["nz"], 0.25
    layers = [[0.0, 2.3, 2.0 * math.sqrt(3), 2.0, 200.0, 100.0], [60.0, 3.2, 4.5 * math.sqrt(3), 4.5, 450.0, 225.0]]
    ext = np.array([nx, ny]) * h / 2 - 30 * h
    # a fault of point sources, some at the surface, some in the planes of the sections
    src = [dict(x=float(rng.uniform(-ext[0], ext[0])) * (q % 4 > 0), y=float(rng.uniform(-ext[1], ext[1])) * (q % 4 > 1),
                z=float(rng.uniform(0.5, 3.0 if q % 2 else nz * h - 12.0)), t0=0.0, tr=0.12, mo=1e15,
                strike=float(rng.uniform(0, 360)), dip=float(rng.uniform(0, 90)), rake=float(rng.uniform(-180, 180)))
           for q in range(48)]
    st = [(src[q % 48]["x"] + float(rng.uniform(-2, 2)), src[q % 48]["y"] + float(rng.uniform(-2, 2)), 0.0, "fsb")
          for q in range(case["stations"])]
    spec = ModelSpec(nx=nx, ny=ny, nz=nz, dx=h, dy=h, dz=h, dt=0.0117, nt=case["steps"], na=case["na"], nm=case["nm"],
                     zbeg=-1.0, vmodel="lgm", layers=layers, sources=src, stations=st, fq_min=0.05, fq_max=5.0,
                     rmedia=dict(ptype="vonkarman", a=(5.0, 5.0, 5.0), epsil=0.05, kappa=0.5, seed=seed))
    sim, inp = make_simulation_device(spec)
    sim.set_snapshots(("yz_v", "xz_v", "fs_v"), inp.arrays["kfs"], i0_yz=nx // 2, j0_xz=ny // 2, idec=2, jdec=2, kdec=2,
                      ntdec_s=case["steps"] - 1, nframe=2, M0=inp.scalars["M0"], UC=inp.scalars["UC"])
    return sim


def _members(case, seed):
    """the members' grids (fixed by the case) and seeds"""
    r = np.random.default_rng(case["members"] * 1000 + case["high"])
    top = case["low"] + (case["high"] - case["low"]) * 2 // 3
    return [(dict(nx=int(r.integers(case["low"], case["high"] + 1)), ny=int(r.integers(case["low"], case["high"] + 1)),
                  nz=int(r.integers(case["low"], top + 1)), na=case["na"], nm=case["nm"], steps=case["steps"],
                  force=True, stations=8), seed * 100 + m) for m in range(case["members"])]


def _green_points(case, seed, inp):
    r = np.random.default_rng(seed + 7)
    n = case["points"]
    na = case["na"]
    i, j = r.integers(na, case["nx"] - na, n), r.integers(na, case["ny"] - na, n)
    src = (int(r.integers(na + 10, case["nx"] - na - 10)), int(r.integers(na + 10, case["ny"] - na - 10)), 12)
    return dict(i=i, j=j, k=r.integers(10, case["nz"] - na, n), src=src,
                stf=_wavelet(case["steps"], inp["dt"], 10 * inp["dt"], 0.0))


def _profile(case, seed):
    """per-plane layered model and tau-method scalars of the device medium builder"""
    r = np.random.default_rng(seed)
    nz = case["nz"]
    k = np.arange(-2, nz + 4)
    vs = np.where(k <= 4, 0.0, np.interp(k, [5, nz], np.sort(r.uniform(2.0, 4.2, 2)))).astype(np.float32)
    rho = np.where(k <= 4, 0.001, 2.3 + 0.2 * vs).astype(np.float32)
    mu = rho * vs * vs
    prof = np.stack([rho, mu, mu, np.where(k <= 4, 1e10, 100 * vs + 1), np.where(k <= 4, 1e10, 50 * vs + 1)])
    return dict(prof=prof.astype(np.float32), clip=(0.0, 9.0, 1.0), tau=(1.2, -0.35, 0.28))


# ---------------------------------------------------------------------------
# what one pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "rmedia":
        n = case["n1"] * case["n2"] * case["n3"]
        return {"bytes": 4.0 * n, "flops": 5.0 * n * math.log2(n)}
    if kind == "batch":
        w = [_step_work(c) for c, _ in _members(case, 0)]
        return {k: float(case["steps"] * sum(x[k] for x in w)) for k in ("bytes", "flops")}
    n = case["nx"] * case["ny"] * case["nz"]
    if kind == "medium":        # the perturbation made, five arrays written, two read back
        return {"bytes": 4.0 * n * 10, "flops": n * (60.0 + 5 * math.log2(n))}
    one, steps = _step_work(case), case["steps"]
    if kind == "adjoint":
        # every step forward once with its fields kept, then the adjoint step that reads them: adjoint fields,
        # memory variables and auxiliaries read and written, medium read, three gradients summed
        ni, npm = _cells(case)
        adj = 4.0 * (ni * (18 + 12 * case["nm"] + 9 + 5 + 6) + npm * (18 + 36 + 9 + 18 + 3 + 6))
        shots = case["sources"]
        return {"bytes": shots * steps * (one["bytes"] + 4.0 * 9 * n + adj), "flops": shots * steps * 3.0 * one["flops"]}
    return {"bytes": float(steps * one["bytes"]), "flops": float(steps * one["flops"])}


def _cells(case):
    nx, ny, nz, na = case["nx"], case["ny"], case["nz"], case["na"]
    n = nx * ny * nz
    ni = n if case.get("abc", "pml") != "pml" else (nx - 2 * na) * (ny - 2 * na) * (nz - na)
    return ni, n - ni


def _step_work(case):
    """one time step: fields, memory variables and auxiliaries read and written once, the medium read once"""
    ni, npm = _cells(case)
    nm = case["nm"]
    return {"bytes": 4.0 * (ni * (18 + 12 * nm + (5 if nm else 3)) + npm * (18 + 36 + 3)),
            "flops": ni * (150.0 + 80 * nm) + npm * 180.0}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
class _Fdm64:
    """The staggered-grid scheme in float64, torch operations on whole grids
    (axes j, i, k).  Interior cells take the 4th-order stencils (other weights
    in the band around the free surface) and the memory variables, absorber
    cells the 2nd-order ones and the auxiliaries; both are written as one
    derivative with per-cell weights."""

    def __init__(self, inp):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: torch.as_tensor(np.asarray(a), device=dev, dtype=torch.float64)  # noqa: E731
        self.t, self.dev = t, dev
        self.n = ny, nx, nz = inp["ny"], inp["nx"], inp["nz"]
        self.inp, self.dt, self.nm = inp, inp["dt"], inp["nm"]
        m = inp["medium"]
        self.rho, self.lam, self.mu = t(m["rho"]), t(m["lam"]), t(m["mu"])
        na, pml = inp["na"], inp["abc"] == "pml"
        J, I, K = (torch.arange(1, n + 1, device=dev).reshape(s) for n, s in zip(self.n, ((-1, 1, 1), (1, -1, 1), (1, 1, -1))))
        self.P = (J <= na) | (J > ny - na) | (I <= na) | (I > nx - na) | (K > nz - na) if pml else None
        band = lambda a, b: (K - a) * (b - K)  # noqa: E731
        c = [torch.as_tensor(m[k][3:-3, 3:-3], device=dev)[:, :, None] for k in ("kfs_top", "kfs_bot", "kob_top", "kob_bot")]
        inb = torch.maximum(band(c[0], c[1]), band(c[2], c[3])) >= 0
        near, far = 17.0 / 16 / DX, 1.0 / 48 / DX
        self.A = torch.where(inb, near - 1.0 / 16 / DX, near + 1.0 / 16 / DX)
        self.B = torch.where(inb, far - 1.0 / 48 / DX, far + 1.0 / 48 / DX)
        tp, ts = t(m["taup"])[3:-3, 3:-3, 3:-3].clone(), t(m["taus"])[3:-3, 3:-3, 3:-3].clone()
        if pml:
            self.A[self.P], self.B[self.P] = 1.0 / DX, 0.0
            tp[self.P], ts[self.P] = 0.0, 0.0
            shape = {"y": (-1, 1, 1), "x": (1, -1, 1), "z": (1, 1, -1)}
            self.g = {a + e: [t(p[:, q]).reshape(shape[a]) for q in range(4)]
                      for (a, e), p in zip((("x", "c"), ("x", "e"), ("y", "c"), ("y", "e"), ("z", "c"), ("z", "e")), inp["absorb"])}
        else:
            self.taper = [t(p[3:-3]).reshape(s) for p, s in zip(inp["absorb"], ((1, -1, 1),) * 2 + ((-1, 1, 1),) * 2 + ((1, 1, -1),) * 2)]
        if self.nm == 0:
            tp, ts = torch.zeros_like(tp), torch.zeros_like(ts)
        self.tp, self.ts = tp, ts
        self.vis = [[float(x) for x in inp["visco"][k]] for k in ("c1", "c2", "d1")] + [float(inp["visco"]["d2"])]

    def start(self):
        z = lambda *s: torch.zeros(s, device=self.dev, dtype=torch.float64)  # noqa: E731
        full, cells = tuple(n + 6 for n in self.n), self.n
        aux = 18 if self.P is not None else 0
        return tuple([z(*full) for _ in range(9)] + [z(*cells) for _ in range(6 * self.nm + aux)])

    def at(self, F, ax=0, d=0):
        s = [slice(3, -3)] * 3
        s[ax] = slice(3 + d, F.shape[ax] - 3 + d)
        return F[tuple(s)]

    def fwd(self, F, ax):
        return (self.at(F, ax, 1) - self.at(F)) * self.A - (self.at(F, ax, 2) - self.at(F, ax, -1)) * self.B

    def bwd(self, F, ax):
        return (self.at(F) - self.at(F, ax, -1)) * self.A - (self.at(F, ax, 1) - self.at(F, ax, -2)) * self.B

    def damp(self, d, prof, aux):
        if self.P is None:
            return d, None
        g = self.g[prof]
        return torch.where(self.P, g[0] * d + g[1] * aux, d), torch.where(self.P, g[2] * aux + g[3] * d * self.dt, 0.0)

    def mean(self, mu, a, b):
        c = lambda da, db: mu[tuple(slice(3 + (da if x == a else db if x == b else 0),  # noqa: E731
                                          mu.shape[x] - 3 + (da if x == a else db if x == b else 0)) for x in range(3))]
        p, q, r, s = c(0, 0), c(1, 0), c(0, 1), c(1, 1)
        return 4 * p * q * r * s / (p * q * r + p * q * s + p * r * s + q * r * s + 1.1920928955078125e-07)

    @staticmethod
    def put(F, v):
        return torch.nn.functional.pad(v, (3,) * 6)

    def step(self, state, it, med, shot):
        lam, mu, rho = med
        V, S, nm, dt = list(state[:3]), list(state[3:9]), self.nm, self.dt
        R, aux = state[9:9 + 6 * nm], list(state[9 + 6 * nm:]) or [None] * 18
        c1, c2, d1, d2 = self.vis
        X, Y, Z = 1, 0, 2
        d = [self.damp(*w) for w in (
            (self.bwd(V[0], X), "xc", aux[0]), (self.bwd(V[1], Y), "yc", aux[1]), (self.bwd(V[2], Z), "zc", aux[2]),
            (self.fwd(V[2], Y), "ye", aux[3]), (self.fwd(V[1], Z), "ze", aux[4]), (self.fwd(V[2], X), "xe", aux[5]),
            (self.fwd(V[0], Z), "ze", aux[6]), (self.fwd(V[1], X), "xe", aux[7]), (self.fwd(V[0], Y), "ye", aux[8]))]
        aux_v = [x[1] for x in d]
        ex, ey, ez = d[0][0], d[1][0], d[2][0]
        e4 = [d[3][0] + d[4][0], d[5][0] + d[6][0], d[7][0] + d[8][0]]
        m0 = self.at(mu)
        l2m, d3, tp, ts = self.at(lam) + 2 * m0, ex + ey + ez, self.tp, self.ts
        shear = [self.mean(mu, Y, Z), self.mean(mu, X, Z), self.mean(mu, X, Y)]
        rate, relax = [], []
        for e in (ey + ez, ex + ez, ex + ey):
            rate.append(l2m * (1 + tp * (1 + d2)) * d3 - 2 * m0 * (1 + ts * (1 + d2)) * e)
            relax.append(l2m * tp * d3 - 2 * m0 * ts * e)
        for h, e in zip(shear, e4):
            rate.append(h * (1 + ts * (1 + d2)) * e)
            relax.append(h * ts * e)
        R2 = []
        for c in range(6):
            for q in range(nm):
                R2.append(c1[q] * R[c * nm + q] - c2[q] * relax[c] * dt)
                rate[c] = rate[c] + d1[q] * R2[-1]
        S = [self.at(s) + r * dt for s, r in zip(S, rate)]
        if self.P is None:
            xc, xb, yc, yb, zc, zb = self.taper
            S = [s * w for s, w in zip(S, [xc * yc * zc] * 3 + [xc * yb * zb, xb * yc * zb, xb * yb * zc])]
        S = [self.put(None, s) for s in S]
        if shot is not None and not self.inp["force"]:
            S = self.glut(S, shot, it)
        f = [self.damp(*w) for w in (
            (self.fwd(S[0], X), "xe", aux[9]), (self.bwd(S[5], Y), "yc", aux[10]), (self.bwd(S[4], Z), "zc", aux[11]),
            (self.bwd(S[5], X), "xc", aux[12]), (self.fwd(S[1], Y), "ye", aux[13]), (self.bwd(S[3], Z), "zc", aux[14]),
            (self.bwd(S[4], X), "xc", aux[15]), (self.bwd(S[3], Y), "yc", aux[16]), (self.fwd(S[2], Z), "ze", aux[17]))]
        r0 = self.at(rho)
        V = [self.at(v) + 2 / (r0 + self.at(rho, ax, 1)) * (f[3 * q][0] + f[3 * q + 1][0] + f[3 * q + 2][0]) * dt
             for q, (v, ax) in enumerate(zip(V, (X, Y, Z)))]
        if self.P is None:
            V = [v * w for v, w in zip(V, (xb * yc * zc, xc * yb * zc, xc * yc * zb))]
        V = [self.put(None, v) for v in V]
        if shot is not None and self.inp["force"]:
            V = self.push(V, rho, shot["i"], shot["j"], shot["k"], shot["comp"] / np.float32(shot["M0"]), shot["stf"][it - 1])
        return tuple(V + S + R2 + ((aux_v + [x[1] for x in f]) if self.P is not None else []))

    def glut(self, S, s, it):
        """the moment-rate tensor taken off the stresses around each source cell"""
        rate = (s["mo"] / np.float32(s["M0"])).astype(np.float64) * s["stf"][it - 1] * (self.dt / DX ** 3)
        if not rate.any():
            return S
        S = [x.clone() for x in S]
        for n, r in enumerate(rate):
            j, i, k = int(s["j"][n]) + 2, int(s["i"][n]) + 2, int(s["k"][n]) + 2
            m = [float(v) * float(r) for v in s["comp"][:, n]]
            for c in range(3):
                S[c][j, i, k] -= m[c]
            for a in (0, 1):
                for b in (0, 1):
                    S[3][j - a, i, k - b] -= m[3] / 4
                    S[4][j, i - a, k - b] -= m[4] / 4
                    S[5][j - a, i - b, k] -= m[5] / 4
        return S

    def push(self, V, rho, I, J, K, comp, stf):
        """a force split over the two velocity points around its cell along each axis"""
        V = [v.clone() for v in V]
        for n in range(len(I)):
            at = [int(J[n]) + 2, int(I[n]) + 2, int(K[n]) + 2]
            for q, ax in enumerate((1, 0, 2)):
                f = float(comp[q][n]) * float(stf[n]) * self.dt / DX ** 3
                up, dn = list(at), list(at)
                up[ax] += 1
                dn[ax] -= 1
                V[q][tuple(at)] += f / (rho[tuple(at)] + rho[tuple(up)])
                V[q][tuple(dn)] += f / (rho[tuple(at)] + rho[tuple(dn)])
        return V

    def trace(self, V, s):
        """(nst, 3) velocity samples at the stations"""
        j, i, k = (torch.as_tensor(np.asarray(s[q]) + 2, device=self.dev).long() for q in ("jst", "ist", "kst"))
        u = [(V[0][j, i, k] + V[0][j, i - 1, k]) / 2, (V[1][j, i, k] + V[1][j - 1, i, k]) / 2,
             -(V[2][j, i, k] + V[2][j, i, k - 1]) / 2]
        return torch.stack(u, 1) * (s["M0"] * UC * 1e9)


def exact(case, seed):
    kind = case["kind"]
    if kind == "rmedia":
        return {"xi": _rmedia64((case["n1"], case["n2"], case["n3"]), (4.0, 5.0, 6.0), case["ptype"], seed)}
    if kind == "medium":
        return _medium64(case, seed)
    if kind == "production":
        return None     # hundreds of millions of cells in 64 bits
    if kind == "batch":
        return [_run64(_Fdm64(_inputs(c, s)))[0].cpu().numpy() for c, s in _members(case, seed)]
    inp = _inputs(case, seed)
    if kind == "adjoint":
        return _gradient64(inp)
    if kind == "green":
        return {"gf": _green64(case, inp, _green_points(case, seed, inp))}
    vel, V = _run64(_Fdm64(inp))
    out = {"vel": vel.cpu().numpy()}
    if kind == "routines":
        return {"vmax": None, **out, "disp": None, "stress": None, "strain": None}
    if case.get("sections"):
        out.update({name: None for name in SECTIONS}, fs_v_max=None)
    if case["nx"] * case["ny"] * case["nz"] <= FIELD_CELLS:
        out.update(zip(("Vx", "Vy", "Vz"), (v.cpu().numpy() for v in V)))
    return out


@torch.no_grad()
def _run64(m):
    s, inp = m.inp["shots"][0], m.inp
    med, state, vel = (m.lam, m.mu, m.rho), m.start(), []
    for it in range(1, inp["steps"] + 1):
        vel.append(m.trace(state, s))
        state = m.step(state, it, med, s)
    return torch.stack(vel, 2), state[:3]


@torch.no_grad()
def _green64(case, inp, p):
    """strain and displacement Green's functions at the points of a run forced at the virtual source"""
    m = _Fdm64(inp)
    med, state = (m.lam, m.mu, m.rho), m.start()
    J, I, K = (torch.as_tensor(p[q] + 2, device=m.dev).long() for q in "jik")
    acc, gf = torch.zeros((12, len(p["i"])), device=m.dev, dtype=torch.float64), []
    unit = {0: (0, 1, 0), 1: (1, 0, 0), 2: (0, 0, 1)}       # x, y, z in (j, i, k)
    for it in range(1, case["steps"] + 1):
        V = state[:3]

        def at(q, *offs):
            o = np.sum([np.multiply(unit[a], s) for a, s in offs], axis=0) if offs else (0, 0, 0)
            return V[q][J + int(o[0]), I + int(o[1]), K + int(o[2])]

        def stag(q, a, *offs):
            return ((at(q, *offs) - at(q, (a, -1), *offs)) * 9 / 8 - (at(q, (a, 1), *offs) - at(q, (a, -2), *offs)) / 24) / DX

        for a in range(3):
            for q in range(3):
                d = stag(q, a) if a == q else sum(stag(q, a, (a, s), (q, r)) for s in (0, 1) for r in (0, -1)) / 4
                acc[3 * a + q] += d * m.dt
        for q in range(3):
            acc[9 + q] += 0.5 * (at(q) + at(q, (q, -1))) * m.dt
        u = UC * 1e9
        gf.append(torch.stack([acc[0] * u, acc[4] * u, acc[8] * u, (acc[5] + acc[7]) * u, (acc[2] + acc[6]) * u,
                               (acc[1] + acc[3]) * u] + [acc[9 + q] * u * 1e3 for q in range(3)], 1))
        state = m.step(state, it, med, None)
        i, j, k = p["src"]
        state = tuple(m.push(list(state[:3]), m.rho, [i], [j], [k], [[0.0], [0.0], [1.0]], [p["stf"][it - 1]])) + state[3:]
    return torch.stack(gf, 2).reshape(-1, case["steps"]).cpu().numpy()


def _gradient64(inp):
    """misfits and summed gradients by automatic differentiation of the scheme, recomputed in segments"""
    from torch.utils.checkpoint import checkpoint
    m = _Fdm64(inp)
    med = [x.requires_grad_(True) for x in (m.lam, m.mu, m.rho)]
    nt, many = inp["steps"], len(inp["shots"]) > 1
    seg = max(1, int(round(math.sqrt(nt))))
    J = []
    for s in inp["shots"]:
        obs = m.t(s["obs"])

        def one(it, lam, mu, rho, *state):
            r = m.trace(state, s) - obs[:, :, it - 1]
            return (0.5 * (r * r).sum(),) + m.step(state, it, (lam, mu, rho), s)

        def part(n0, lam, mu, rho, *state):
            total = 0.0
            for it in range(n0 + 1, min(n0 + seg, nt) + 1):
                j, *state = checkpoint(one, it, lam, mu, rho, *state, use_reentrant=False)
                total = total + j
            return (total,) + tuple(state)

        total, state = 0.0, m.start()
        for n0 in range(0, nt, seg):
            j, *state = checkpoint(part, n0, *med, *state, use_reentrant=False)
            total = total + j
        total.backward()
        J.append(float(total))
    g = []
    for x in med:
        v = torch.zeros_like(x)
        v[3:-3, 3:-3, 3:-3] = x.grad[3:-3, 3:-3, 3:-3]
        g.append(v.detach().cpu().numpy())
    return {"misfit": J if many else J[0], "lam": g[0], "mu": g[1], "rho": g[2]}


def _mix(z):
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


def _rmedia64(n, a, ptype, seed):
    """uniform noise, whitened and coloured by the power spectrum, scaled to zero mean and 5 % rms; axis 1 fastest"""
    key = _mix(np.array([seed], np.uint64))
    noise = (_mix(key ^ np.arange(n[0] * n[1] * n[2], dtype=np.uint64)) >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    b = torch.fft.fftn(torch.as_tensor(noise.reshape(n[2], n[1], n[0]), device=dev))
    k = [2 * np.pi * torch.fft.fftfreq(q, DX, device=dev, dtype=torch.float64) * s for q, s in zip(n, a)]
    q2 = (k[2] ** 2)[:, None, None] + (k[1] ** 2)[None, :, None] + (k[0] ** 2)[None, None, :]
    shape = torch.exp(-q2 / 4) if ptype == "gauss" else (1 + q2) ** -2.0
    b = b / b.abs().clamp_min(1e-300) * torch.sqrt(shape)
    b[0, 0, 0] = 0
    x = torch.fft.ifftn(b).real
    x = x - x.mean()
    return (x * (0.05 / torch.sqrt((x * x).mean()))).cpu().numpy()


def _medium64(case, seed):
    """relaxed moduli of the perturbed layered model"""
    nx, ny, nz, na, nm = (case[k] for k in ("nx", "ny", "nz", "na", "nm"))
    p = _profile(case, seed)
    rho, lam, mu, qp, qs = (x[_clamp(nz, na, False) + 2].astype(np.float64)[None, None, :] for x in p["prof"])
    xi = _rmedia64((nz + 6, nx + 6, ny + 6), (5.0,) * 3, "vonkarman", seed)
    xi = xi[_clamp(ny, na, True) + 2][:, _clamp(nx, na, True) + 2][:, :, _clamp(nz, na, False) + 2]
    vp, vs = np.sqrt((lam + 2 * mu) / rho) * (1 + xi), np.sqrt(mu / rho) * (1 + xi)
    solid = mu > 1e-7
    r = np.where(solid, rho * (1 + 0.8 * xi), rho)
    over = solid & (np.maximum(vp, vs) > p["clip"][1])
    ratio = np.divide(p["clip"][1], vp, out=np.ones_like(vp), where=over)
    r = np.where(over, r * (1 + 0.8 * ((1 + xi) * ratio - 1)) / (1 + 0.8 * xi), r)
    r = np.where(solid, np.maximum(r, p["clip"][2]), r)
    m = np.where(solid, r * (vs * ratio) ** 2, mu)
    l2m = np.where(solid, r * (vp * ratio) ** 2, lam + 2 * mu)
    if nm:
        zeta, ccr, cci = (float(np.float32(v)) for v in p["tau"])
        chi = lambda q: 1 / np.real(1 / np.sqrt(1 - (ccr + 1j * cci) * nm * zeta / q))  # noqa: E731
        m, l2m = m / chi(qs) ** 2, l2m / chi(qp) ** 2
    return {"kfs": None, "kob": None, "vrange": None, "lam": l2m - 2 * m, "mu": m}
