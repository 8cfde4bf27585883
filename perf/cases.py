"""The work that users of this library have it do, as timed cases.

Every case goes through the C ABI of include/fteik/fteik_amd.h (the entry
points that C, Fortran and ctypes callers use).  The library keeps one
solver of each kind per process, so what a program sets up once (grid,
velocity model, receivers, travel-time tables, a trained network) is a
session shared by the states of a case; a state holds what changes from call
to call: sources, stations, grids of a batch, picks.

kind        one pass
solve3d     set the source, solve, read the receiver times and the field
batch3d     a batch of independent grids from host models to host fields
stations    station tables by reciprocity, then events located with them
locate      full grid search of a catalogue's events (or of one event)
solve2d     many sources on one 2D model: receiver times, the last field
surrogate   network proposals scored with the exact tables
"""
import ctypes
import math

import numpy as np
import torch

import fteik_amd

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
EPS3D, EPS2D = 5.0, 3.0       # spherical-operator radii of the benchmark
NOISE = 0.05                  # pick noise, s
V0, GRAD = 4000.0, 0.4        # the locator's 1D gradient, m/s and 1/s
BLOCKS = 12                   # event blocks a locator's catalogue holds
_dp = ctypes.POINTER(ctypes.c_double)
_ip = ctypes.POINTER(ctypes.c_int)
_fp = ctypes.POINTER(ctypes.c_float)


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the smallest useful 3D call: a local model, launch latency counts
        dict(name="solve3d_small", kind="solve3d", nz=33, nx=29, ny=31,
             h=10.0, nsweep=2, precision=0, model="gradient", nrec=20),
        # the reference's CPU-sized case: 101^3, gradient, 20 receivers
        dict(name="solve3d_101", kind="solve3d", nz=101, nx=101, ny=101,
             h=10.0, nsweep=2, precision=0, model="gradient", nrec=20),
        # the benchmark's headline: 257^3 layered model, FP64 to convergence
        dict(name="solve3d_257", kind="solve3d", nz=257, nx=257, ny=257,
             h=20.0, nsweep=19, precision=0, model="layered", nrec=20),
        # mixed precision on a ragged grid
        dict(name="solve3d_mixed", kind="solve3d", nz=131, nx=190, ny=157,
             h=20.0, nsweep=12, precision=1, model="layered", nrec=33),
        # grids of uneven size solved together, whole call on host data
        dict(name="batch_uneven", kind="batch3d", ngrids=16, nmin=64,
             nmax=192, h=50.0, nsweep=12, precision=0),
        # a network's travel-time tables, then the day's events
        dict(name="station_tables", kind="stations", nsta=48, nz=81, nx=161,
             ny=161, h=250.0, nsweep=2, nev=256),
        # relocating a catalogue: the benchmark's 10,000 events
        dict(name="locate_10k", kind="locate", nsta=48, nz=81, nx=161,
             ny=161, h=250.0, nev=10000, missing=0.0),
        # a regional network of odd size, picks missing, uneven weights
        dict(name="locate_ragged", kind="locate", nsta=37, nz=41, nx=90,
             ny=77, h=400.0, nev=1500, missing=0.2),
        # one event as it comes in (the reference's own entry point)
        dict(name="locate_one", kind="locate", nsta=48, nz=81, nx=161,
             ny=161, h=250.0, nev=1, missing=0.0),
        # refraction tomography: 256 shots on one 2D model
        dict(name="solve2d_256", kind="solve2d", nz=501, nx=501, h=10.0,
             nsweep=2, nsrc=256, nrec=32),
        # a long profile, a few shots
        dict(name="solve2d_wide", kind="solve2d", nz=301, nx=1201, h=10.0,
             nsweep=2, nsrc=4, nrec=57),
        # the learned locator on the same catalogue
        dict(name="surrogate_10k", kind="surrogate", nsta=48, nz=81, nx=161,
             ny=161, h=250.0, nev=10000, steps=1500),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("solve3d", "solve3d", "batch3d", "stations", "locate",
                       "locate", "solve2d", "solve2d", "surrogate"))
    if kind == "solve3d":
        return dict(kind=kind, nz=_log_int(rng, 24, 200),
                    nx=_log_int(rng, 24, 200), ny=_log_int(rng, 24, 200),
                    h=rng.choice((10.0, 20.0, 50.0)),
                    nsweep=rng.randint(1, 12),
                    precision=rng.choice((0, 0, 1)),
                    model=rng.choice(("gradient", "layered")),
                    nrec=_log_int(rng, 1, 200))
    if kind == "batch3d":
        nmin = rng.randint(32, 80)
        return dict(kind=kind, ngrids=_log_int(rng, 2, 16), nmin=nmin,
                    nmax=rng.randint(nmin + 8, 128), h=50.0,
                    nsweep=rng.randint(2, 8), precision=rng.choice((0, 1)))
    if kind == "stations":
        return dict(kind=kind, nsta=_log_int(rng, 4, 40),
                    nz=rng.randint(28, 81), nx=rng.randint(40, 130),
                    ny=rng.randint(40, 130), h=250.0,
                    nsweep=rng.randint(1, 4), nev=_log_int(rng, 8, 256))
    if kind == "locate":
        nz, nx, ny = (rng.randint(20, 81), rng.randint(24, 161),
                      rng.randint(24, 161))
        nsta = _log_int(rng, 4, 80)
        most = int(2.0e11/(nz*nx*ny*nsta))
        return dict(kind=kind, nsta=nsta, nz=nz, nx=nx, ny=ny,
                    h=rng.choice((250.0, 400.0)),
                    nev=_log_int(rng, 1, max(2, min(5000, most))),
                    missing=rng.choice((0.0, 0.1, 0.3)))
    if kind == "solve2d":
        nz, nx = _log_int(rng, 48, 1200), _log_int(rng, 48, 1600)
        return dict(kind=kind, nz=nz, nx=nx, h=10.0,
                    nsweep=rng.randint(1, 4),
                    nsrc=_log_int(rng, 1, min(200, int(4.0e7/(nz*nx)))),
                    nrec=_log_int(rng, 1, 200))
    return dict(kind=kind, nsta=rng.randint(8, 48), nz=rng.randint(24, 81),
                nx=rng.randint(48, 161), ny=rng.randint(48, 161), h=250.0,
                nev=_log_int(rng, 100, 8000), steps=1000)


# ---------------------------------------------------------------- helpers
def _lib():
    return fteik_amd.load_library()


def _d(a):
    return a.ctypes.data_as(_dp)


def _i(a):
    return a.ctypes.data_as(_ip)


def _call(fn, *args):
    """A call whose last argument is ierr (2: a mixed-precision solve kept
    its field at the correction cap)."""
    ierr = ctypes.c_int(1)
    fn(*args, ctypes.byref(ierr))
    if ierr.value not in (0, 2):
        raise RuntimeError("%s failed (ierr = %d)" % (fn.__name__, ierr.value))


def _smooth_noise(shape, sigma, seed):
    """Gaussian-smoothed noise of the given shape, scaled to max |g| = 1."""
    g = torch.from_numpy(np.random.default_rng(seed).standard_normal(shape))
    f = torch.fft.fftn(g.to(DEVICE))
    for ax, n in enumerate(shape):
        k = torch.fft.fftfreq(n, dtype=torch.float64, device=DEVICE)
        w = torch.exp(-2.0*(math.pi*sigma*k)**2)
        f = f*w.reshape([-1 if a == ax else 1 for a in range(len(shape))])
    g = torch.fft.ifftn(f).real
    return (g/g.abs().max()).cpu().numpy()


def _model3d(nz, nx, ny, h, model, seed):
    """Cell velocities, z fastest: v = 3000 + 0.5 z, or eight layers of
    1500 to 6500 m/s with a smoothed 5 % perturbation."""
    z = (np.arange(nz - 1) + 0.5)*h
    if model == "gradient":
        return np.ascontiguousarray(np.tile(3000.0 + 0.5*z, (nx - 1)*(ny - 1)))
    rng = np.random.default_rng(seed)
    tops = np.sort(rng.uniform(0.0, (nz - 1)*h, 7))
    v = np.linspace(1500.0, 6500.0, 8)[np.searchsorted(tops, z)]
    g = _smooth_noise((ny - 1, nx - 1, nz - 1), 5.0, seed + 1)
    return np.ascontiguousarray((v[None, None, :]*(1.0 + 0.05*g)).ravel())


def _gradient_time(dist, z0, z1):
    """Travel time in v = V0 + GRAD z between depths z0 and z1 (tensors) a
    distance dist apart."""
    a = 1.0 + 0.5*(GRAD*dist)**2/((V0 + GRAD*z0)*(V0 + GRAD*z1))
    return torch.acosh(a)/GRAD


def _stations(c, seed):
    """nsta stations on the surface, (x, y) in metres."""
    r = np.random.default_rng(seed)
    return np.stack([r.uniform(0.0, (c["nx"] - 3)*c["h"], c["nsta"]),
                     r.uniform(0.0, (c["ny"] - 3)*c["h"], c["nsta"])], 1)


def _tables(c):
    """FP32 travel times of every station to every node, z fastest."""
    f = dict(dtype=torch.float64, device=DEVICE)
    h, out = c["h"], []
    z = (torch.arange(c["nz"], **f)*h).reshape(1, 1, -1)
    x = (torch.arange(c["nx"], **f)*h).reshape(1, -1, 1)
    y = (torch.arange(c["ny"], **f)*h).reshape(-1, 1, 1)
    for sx, sy in _stations(c, 9):
        d = torch.sqrt((x - sx)**2 + (y - sy)**2 + z**2)
        out.append(_gradient_time(d, torch.zeros_like(z), z)
                   .to(torch.float32).reshape(-1))
    return torch.stack(out)


def _picks(c, stations, seed):
    """Observations of nev events: for each, its stations (1-based), pick
    times and weights.  Hypocentres uniform, origin times U(0, 100) s."""
    r = np.random.default_rng(seed)
    n, ns = c["nev"], len(stations)
    lim = np.array([c["nz"] - 1, c["nx"] - 1, c["ny"] - 1])*c["h"]
    hyp = r.uniform(0.0, 1.0, (n, 3))*lim
    d = np.sqrt((hyp[:, None, 1] - stations[None, :, 0])**2
                + (hyp[:, None, 2] - stations[None, :, 1])**2
                + hyp[:, None, 0]**2)
    z = torch.from_numpy(hyp[:, :1].copy())
    t = _gradient_time(torch.from_numpy(d), torch.zeros_like(z), z).numpy()
    t = t + r.uniform(0.0, 100.0, (n, 1)) + r.normal(0.0, NOISE, t.shape)
    miss = c.get("missing", 0.0)
    have = r.uniform(0.0, 1.0, t.shape) >= miss
    have[:, :4] = True
    w = r.choice((1.0, 0.5, 0.25), t.shape) if miss > 0 else np.ones(t.shape)
    out = []
    for e in range(n):
        k = np.flatnonzero(have[e])
        out.append(((k + 1).astype(np.int32),
                    np.ascontiguousarray(t[e, k]),
                    np.ascontiguousarray(w[e, k])))
    return out


def _observe(first, obs):
    L = _lib()
    for e, (o2t, t, w) in enumerate(obs):
        _call(L.locate_setObservation64f, first + e, t.size, False, 0.0,
              _i(o2t), _d(t), _d(w))


# --------------------------------------------------------------- sessions
_session = {"key": None}


def _free_all():
    L = _lib()
    L.fteik_surrogate_free()
    L.fteik_batch3d_free()
    L.locate_finalize()
    L.fteik_solver2d_free()
    L.fteik_solver3d_free()


def _open(c):
    """Sets the library up for case c unless it already is."""
    key = tuple(sorted((k, v) for k, v in c.items() if k != "name"))
    if _session["key"] == key:
        return
    _session.clear()
    _session["key"] = None
    _free_all()
    L, kind = _lib(), c["kind"]
    if kind in ("solve3d", "stations"):
        model = c.get("model", "")
        if kind == "stations":
            z = (np.arange(c["nz"] - 1) + 0.5)*c["h"]
            vel = np.ascontiguousarray(
                np.tile(V0 + GRAD*z, (c["nx"] - 1)*(c["ny"] - 1)))
        else:
            vel = _model3d(c["nz"], c["nx"], c["ny"], c["h"], model, 2)
        h = c["h"]
        _call(L.fteik_solver3d_initialize, c["nz"], c["nx"], c["ny"], 0.0,
              0.0, 0.0, h, h, h, c["nsweep"], EPS3D, 0.0, 0)
        _call(L.fteik_solver3d_setVelocityModel64f, vel.size, _d(vel))
        if kind == "solve3d":
            _call(L.fteik_solver3d_setPrecision, c["precision"])
            rec = _receivers3d(c)
            _call(L.fteik_solver3d_setReceivers64f, c["nrec"],
                  *(_d(v) for v in rec))
    if kind in ("stations", "locate", "surrogate"):
        ngrd = c["nz"]*c["nx"]*c["ny"]
        _call(L.locate_initialize, BLOCKS*c["nev"], c["nsta"], ngrd)
        _call(L.locate_setReferenceCompatibility, 0)
        if kind != "stations":
            for k, t in enumerate(_tables(c).cpu().numpy()):
                _call(L.locate_setTravelTimeField32f, ngrd, k + 1,
                      t.ctypes.data_as(_fp))
        _session["owner"] = [None]*BLOCKS
        _session["next"] = 0
    if kind == "surrogate":
        st = _stations(c, 9)
        zs, xs, ys = np.zeros(c["nsta"]), st[:, 0].copy(), st[:, 1].copy()
        h, loss = c["h"], ctypes.c_double()
        _call(L.fteik_surrogate_initialize, c["nsta"], c["nz"], c["nx"],
              c["ny"], h, h, h, _d(zs), _d(xs), _d(ys), 6000.0, 1.0, 13)
        _call(L.fteik_surrogate_train, c["steps"], 8192, 2e-3, 500000,
              ctypes.byref(loss))
    if kind == "solve2d":
        h = c["h"]
        vel = _model2d(c)
        _call(L.fteik_solver2d_initialize, c["nz"], c["nx"], 0.0, 0.0, h, h,
              c["nsweep"], EPS2D, 0.0, 0)
        _call(L.fteik_solver2d_setCellVelocityModel64f, vel.size, 0, _d(vel))
        zr, xr = _receivers2d(c)
        _call(L.fteik_solver2d_setReceivers64f, c["nrec"], _d(zr), _d(xr))
    _session["key"] = key


def _receivers3d(c):
    r = np.random.default_rng(101)
    return (np.zeros(c["nrec"]),
            r.uniform(0.0, (c["nx"] - 1)*c["h"], c["nrec"]),
            r.uniform(0.0, (c["ny"] - 1)*c["h"], c["nrec"]))


def _source3d(c, seed):
    u = np.random.default_rng(seed).uniform(0.02, 0.98, 3)
    return [np.array([v*(n - 3)*c["h"]])
            for v, n in zip(u, (c["nz"], c["nx"], c["ny"]))]


def _model2d(c):
    z = (np.arange(c["nz"] - 1) + 0.5)*c["h"]
    x = (np.arange(c["nx"] - 1) + 0.5)*c["h"]
    p = 1.0 + 0.05*np.sin(x[:, None]/700.0)*np.cos(z[None, :]/450.0)
    return np.ascontiguousarray(((1500.0 + 0.8*z)[None, :]*p).ravel())


def _receivers2d(c):
    return np.zeros(c["nrec"]), np.linspace(0.0, (c["nx"] - 1)*c["h"],
                                            c["nrec"] + 1)[1:].copy()


def _sources2d(c, seed):
    u = np.random.default_rng(seed).uniform(0.01, 0.99, (2, c["nsrc"]))
    return u[0]*(c["nz"] - 3)*c["h"], u[1]*(c["nx"] - 3)*c["h"]


def _batch_models(c, seed):
    """ngrids grids of U{nmin..nmax} nodes an axis (the same sizes for every
    seed), v = 2000 + U(0.3, 0.8) z with a smoothed 3 % perturbation, a
    source in each."""
    dims = np.random.default_rng(5).integers(c["nmin"], c["nmax"] + 1,
                                             (c["ngrids"], 3))
    r, out = np.random.default_rng(seed), []
    for nz, nx, ny in dims.tolist():
        z = (np.arange(nz - 1) + 0.5)*c["h"]
        v = 2000.0 + r.uniform(0.3, 0.8)*z
        g = _smooth_noise((ny - 1, nx - 1, nz - 1), 5.0,
                          int(r.integers(1 << 31)))
        vel = np.ascontiguousarray((v[None, None, :]*(1.0 + 0.03*g)).ravel())
        src = [float(r.uniform(0.02, 0.98)*(n - 3)*c["h"])
               for n in (nz, nx, ny)]
        out.append((nz, nx, ny, vel, src))
    return out


# ------------------------------------------------------------ preparation
def prepare(case, seed):
    c = dict(case)
    s = {"case": c, "kind": c["kind"]}
    kind = c["kind"]
    if kind != "batch3d":
        _open(c)
    if kind == "solve3d":
        s["src"] = _source3d(c, seed)
        s["ttr"] = np.zeros(c["nrec"])
        s["tt"] = np.zeros(c["nz"]*c["nx"]*c["ny"])
    elif kind == "batch3d":
        s["grids"] = _batch_models(c, seed)
        s["tt"] = [np.zeros(nz*nx*ny) for nz, nx, ny, _, _ in s["grids"]]
    elif kind == "solve2d":
        s["src"] = _sources2d(c, seed)
        s["ttr"] = np.zeros(c["nrec"]*c["nsrc"])
        s["tt"] = np.zeros(c["nz"]*c["nx"])
    else:
        st = _stations(c, seed if kind == "stations" else 9)
        s["sta"] = [np.zeros(c["nsta"]), st[:, 0].copy(), st[:, 1].copy()]
        s["obs"] = _picks(c, st, seed + 1)
        s["opt"] = np.zeros(c["nev"], dtype=np.int32)
        s["t0"], s["obj"] = np.zeros(c["nev"]), np.zeros(c["nev"])
        if kind == "stations":
            s["tt"] = np.zeros(c["nz"]*c["nx"]*c["ny"])
        s["block"] = -1
        _enter(s)
    return s


def _enter(s):
    """Enters the state's events in the locator's catalogue."""
    b = _session["next"]
    _session["next"] = (b + 1) % BLOCKS
    _session["owner"][b] = s["obs"]
    s["block"] = b
    n = s["case"]["nev"]
    s["ev"] = np.arange(b*n + 1, b*n + n + 1, dtype=np.int32)
    _observe(b*n + 1, s["obs"])


# ------------------------------------------------------------------- runs
def run(state):
    L, c, kind = _lib(), state["case"], state["kind"]
    if kind == "batch3d":
        return _run_batch(L, c, state)
    _open(c)
    if kind == "solve3d":
        z, x, y = state["src"]
        tt, ttr = state["tt"], state["ttr"]
        _call(L.fteik_solver3d_setSources64f, 1, _d(z), _d(x), _d(y))
        _call(L.fteik_solver3d_solveSourceLSM, 1)
        _call(L.fteik_solver3d_getTravelTimes64f, ttr.size, _d(ttr))
        _call(L.fteik_solver3d_getTravelTimeField64f, tt.size, 0, _d(tt))
        return {"receivers": ttr, "field": tt}
    if kind == "solve2d":
        z, x = state["src"]
        tt, ttr = state["tt"], state["ttr"]
        _call(L.fteik_solver2d_setSources64f, z.size, _d(z), _d(x))
        _call(L.fteik_solver2d_solveLSM)
        _call(L.fteik_solver2d_getTravelTimes64f, c["nrec"], _d(ttr))
        _call(L.fteik_solver2d_getTravelTimeField64f, tt.size, 0, _d(tt))
        return {"receivers": ttr, "field": tt}
    if _session["owner"][state["block"]] is not state["obs"]:
        _enter(state)              # its block went to later events
    ev, opt, t0, obj = (state[k] for k in ("ev", "opt", "t0", "obj"))
    out = {"cell": opt, "origin": t0, "objective": obj}
    if kind == "surrogate":
        nfb = ctypes.c_int()
        _call(L.locate_locateEventsSurrogate, ev.size, _i(ev), 8, 6, _i(opt),
              _d(t0), _d(obj), ctypes.byref(nfb))
        return out
    if kind == "stations":
        sta = state["sta"]
        _call(L.locate_setTravelTimeFieldsFromStations3d, c["nsta"],
              _d(sta[0]), _d(sta[1]), _d(sta[2]), c["nsweep"], EPS3D, 0, 1)
        tt = state["tt"]
        _call(L.fteik_batch3d_getTravelTimeField64f, c["nsta"], tt.size, 0,
              _d(tt))
        out["field"] = tt
    if kind == "locate" and ev.size == 1:
        L.locate_locateEvent(int(ev[0]), _i(opt), _d(t0), _d(obj))
    else:
        _call(L.locate_locateEvents, ev.size, _i(ev), _i(opt), _d(t0),
              _d(obj))
    return out


def _run_batch(L, c, state):
    h = c["h"]
    _session["key"] = None         # the batch solver is set up anew
    _call(L.fteik_batch3d_initialize, c["ngrids"])
    for k, (nz, nx, ny, vel, (zs, xs, ys)) in enumerate(state["grids"]):
        _call(L.fteik_batch3d_setGrid, k + 1, nz, nx, ny, 0.0, 0.0, 0.0, h,
              h, h, _d(vel), zs, xs, ys)
    _call(L.fteik_batch3d_setPrecision, c["precision"])
    _call(L.fteik_batch3d_setMixedParameters, 1.0/64.0, 64)
    _call(L.fteik_batch3d_solve, c["nsweep"], EPS3D)
    for k, tt in enumerate(state["tt"]):
        _call(L.fteik_batch3d_getTravelTimeField64f, k + 1, tt.size, 0,
              _d(tt))
    return state["tt"]


# ------------------------------------------------------------------- work
def work(case):
    """Bytes: inputs read once and outputs written once (FP64 slowness and
    field; FP32 tables).  Operations: a 3D update about 100, a 2D one about
    30, a misfit term 9, a network row 2 per weight and product."""
    c, kind = case, case["kind"]
    if kind == "solve3d":
        n = c["nz"]*c["nx"]*c["ny"]
        return {"bytes": 16.0*n, "flops": 100.0*n*8*(c["nsweep"] + 1)}
    if kind == "batch3d":
        dims = np.random.default_rng(5).integers(c["nmin"], c["nmax"] + 1,
                                                 (c["ngrids"], 3))
        n = float(np.prod(dims, axis=1).sum())
        return {"bytes": 16.0*n, "flops": 100.0*n*8*(c["nsweep"] + 1)}
    if kind == "solve2d":
        n = float(c["nz"]*c["nx"]*c["nsrc"])
        return {"bytes": 8.0*n + 8.0*c["nz"]*c["nx"],
                "flops": 30.0*n*4*(c["nsweep"] + 1)}
    n = float(c["nz"]*c["nx"]*c["ny"])
    if kind == "stations":
        return {"bytes": (8.0 + 12.0*c["nsta"])*n,
                "flops": 100.0*n*c["nsta"]*8*(c["nsweep"] + 1)
                + 9.0*n*c["nsta"]*c["nev"]}
    if kind == "locate":
        return {"bytes": 4.0*n*c["nsta"] + 12.0*c["nev"]*c["nsta"],
                "flops": 9.0*n*c["nsta"]*c["nev"]}
    weights = 3*256 + 3*256*256 + 256*c["nsta"]
    return {"bytes": 4.0*64*c["nsta"]*c["nev"],
            "flops": 7.0*8*c["nev"]*4*2*weights}


# ------------------------------------------------------------------ exact
def exact(case, seed):
    """The same outputs from plain 64-bit torch, for the cases where the
    path has such a value and it is quick to find."""
    c, kind = dict(case), case["kind"]
    if kind == "solve3d" and c["precision"] == 0 and \
            c["nz"]*c["nx"]*c["ny"] <= 1100000 and c["nsweep"] <= 4:
        tt = _plain3d(c, seed)
        rec = _interpolate(tt, _receivers3d(c), c["h"])
        return {"receivers": rec.cpu().numpy(),
                "field": tt.reshape(-1).cpu().numpy()}
    if kind == "solve2d" and c["nz"]*c["nx"]*c["nsrc"] <= 70000000 and \
            (c["nz"] + c["nx"])*(c["nsweep"] + 3) <= 6000:
        tt = _plain2d(c, seed)
        zr, xr = _receivers2d(c)
        h, r = c["h"], []
        for z, x in zip(zr/h, xr/h):
            i, j = min(int(z), c["nz"] - 2), min(int(x), c["nx"] - 2)
            a, b = z - i, x - j
            r.append(tt[:, j, i]*(1 - a)*(1 - b) + tt[:, j, i + 1]*a*(1 - b)
                     + tt[:, j + 1, i]*(1 - a)*b + tt[:, j + 1, i + 1]*a*b)
        return {"receivers": torch.stack(r, 1).reshape(-1).cpu().numpy(),
                "field": tt[-1].reshape(-1).cpu().numpy()}
    if kind == "locate":
        t0, obj = _plain_locate(c, seed)
        return {"cell": None, "origin": t0, "objective": obj}
    return None


def _plain_locate(c, seed):
    """Least objective over the cells and its origin time, per event:
    t0 = sum w r / sum w, objective = sum w^2 (r - t0)^2 / 2, r = o - T."""
    T = _tables(c).to(torch.float64)
    obs = _picks(c, _stations(c, 9), seed + 1)
    n, ns = c["nev"], c["nsta"]
    o, w = np.zeros((n, ns)), np.zeros((n, ns))
    for e, (k, t, wt) in enumerate(obs):
        o[e, k - 1], w[e, k - 1] = t, wt
    base = np.array([t.max() for _, t, _ in obs])
    o = torch.from_numpy((o - base[:, None])*(w > 0)).to(DEVICE)
    w = torch.from_numpy(w).to(DEVICE)
    T2, t0s, objs = T*T, [], []
    step = max(1, int(1.5e8/T.shape[1]))
    for a in range(0, n, step):
        wa, oa = w[a:a + step], o[a:a + step]
        w2 = wa*wa
        t0 = ((wa*oa).sum(1, True) - wa @ T)/wa.sum(1, True)
        wr = (w2*oa).sum(1, True) - w2 @ T
        f = (w2*oa*oa).sum(1, True) - 2.0*((w2*oa) @ T) + w2 @ T2
        f = 0.5*(f - 2.0*t0*wr + t0*t0*w2.sum(1, True))
        m, at = f.min(1)
        objs.append(m)
        t0s.append(t0.gather(1, at[:, None])[:, 0])
    return (torch.cat(t0s).cpu().numpy() + base, torch.cat(objs).cpu().numpy())


def _interpolate(tt, rec, h):
    """Trilinear interpolation of tt[y, x, z] at (z, x, y) positions."""
    ny, nx, nz = tt.shape
    g = [torch.from_numpy(v/h).to(tt.device) for v in rec]
    b = [v.floor().clamp(0, n - 2).long() for v, n in zip(g, (nz, nx, ny))]
    f = [v - i for v, i in zip(g, b)]
    out = torch.zeros_like(g[0])
    for k in range(8):
        d = [k & 1, (k >> 1) & 1, k >> 2]
        w = 1.0
        for q in range(3):
            w = w*(f[q] if d[q] else 1.0 - f[q])
        out = out + w*tt[b[2] + d[2], b[1] + d[1], b[0] + d[0]]
    return out


HUGE = 99999.0
SIGNS3D = [(1, 1, 1), (1, -1, 1), (1, 1, -1), (1, -1, -1),
           (-1, 1, 1), (-1, -1, 1), (-1, 1, -1), (-1, -1, -1)]  # z, x, y


def _sqrt(x):
    return torch.sqrt(x.clamp(min=0.0))


def _plane(ta, tb, s, p):
    """The 2D Cartesian operator on a square cell of slowness s and width h,
    p = 1/h^2 (ta, tb: the neighbour times combined along the two axes)."""
    return ((ta + tb)*p + _sqrt(8.0*s*s*p - p*p*(ta - tb)**2))/(2.0*p)


def _plain3d(c, seed):
    """The factored-eikonal sweeps of the 3D solver, a level at a time, for
    equal spacings: tt[y, x, z]."""
    nz, nx, ny, h = c["nz"], c["nx"], c["ny"], c["h"]
    f = dict(dtype=torch.float64, device=DEVICE)
    vel = _model3d(nz, nx, ny, h, c["model"], 2)
    slow = 1.0/torch.from_numpy(vel).to(DEVICE).reshape(ny - 1, nx - 1, nz - 1)
    src = [float(v[0])/h for v in _source3d(c, seed)]        # z, x, y nodes
    si = [int(v) for v in src]
    s0 = float(slow[si[2], si[1], si[0]])
    eps, p = EPS3D*h*s0, 1.0/h**2
    tt = torch.full((ny, nx, nz), HUGE, **f)
    for k in range(8):
        q = [si[0] + (k & 1), si[1] + ((k >> 1) & 1), si[2] + (k >> 2)]
        tt[q[2], q[1], q[0]] = s0*h*math.dist(q, src)
    # nodes of the flipped frame by level, first row of each axis left out
    dims = (nz, nx, ny)
    a = torch.arange(nz*nx*ny, device=DEVICE)
    fz, fx, fy = a % nz, (a // nz) % nx, a // (nz*nx)
    order = torch.argsort(fz + fx + fy, stable=True)
    fz, fx, fy = fz[order], fx[order], fy[order]
    inside = (fz > 0) & (fx > 0) & (fy > 0)
    for it in range(c["nsweep"] + 1):
        for sg in SIGNS3D:
            keep = inside
            if it == 0:                # initialization: from the source on
                for v, n, s, i in zip((fz, fx, fy), dims, sg, si):
                    keep = keep & (v >= (i if s > 0 else n - 2 - i))
            z, x, y = fz[keep], fx[keep], fy[keep]
            flip = [d for d, s in ((2, sg[0]), (1, sg[1]), (0, sg[2])) if s < 0]
            T = tt.flip(flip).contiguous().reshape(-1)
            S = slow.flip(flip)
            pos = [(v if s > 0 else n - 1 - v).to(torch.float64)
                   for v, n, s in zip((z, x, y), dims, sg)]
            sl = _cells(S, z, x, y)
            g = z + nz*(x + nx*y)
            cut = torch.bincount(z + x + y).cpu().tolist()
            i0 = 0
            for cnt in cut:
                i1 = i0 + cnt
                if cnt:
                    b = g[i0:i1]
                    nb = [T[b - 1], T[b - nz], T[b - nz*nx], T[b - 1 - nz],
                          T[b - nz - nz*nx], T[b - 1 - nz*nx],
                          T[b - 1 - nz - nz*nx]]
                    s7 = [v[i0:i1] for v in sl]
                    if it == 0:
                        w = [v[i0:i1] for v in pos]
                        new = _init3d(nb, s7, w, sg, src, si, s0, eps, h)
                    else:
                        new = _iter3d(nb, s7, h, p)
                    T[b] = torch.minimum(T[b], new)
                i0 = i1
            tt = T.reshape(ny, nx, nz).flip(flip)
    return tt.contiguous()


def _cells(S, z, x, y):
    """The seven least slownesses a node reads (planes, lines, cell)."""
    ncy, ncx, ncz = S.shape
    u = (z - 1, x - 1, y - 1)
    d = (z.clamp(max=ncz - 1), x.clamp(max=ncx - 1), y.clamp(max=ncy - 1))

    def at(a, b, e):
        return S[(u, d)[e][2], (u, d)[b][1], (u, d)[a][0]]
    c = {(a, b, e): at(a, b, e) for a in (0, 1) for b in (0, 1)
         for e in (0, 1)}

    def least(*k):
        v = c[k[0]]
        for q in k[1:]:
            v = torch.minimum(v, c[q])
        return v
    o = (0, 0, 0)
    return [least(o, (0, 1, 0), (0, 0, 1), (0, 1, 1)),
            least(o, (1, 0, 0), (0, 0, 1), (1, 0, 1)),
            least(o, (1, 0, 0), (0, 1, 0), (1, 1, 0)),
            least(o, (0, 0, 1)), least(o, (0, 1, 0)), least(o, (1, 0, 0)),
            c[o]]


def _cube(tv, te, tn, tev, ten, tnv, tnve, s, p):
    ta = te + 0.5*(-tn + ten - tv + tev) - tnv + tnve
    tb = tv + 0.5*(-tn + tnv - te + tev) - ten + tnve
    tc = tn + 0.5*(-te + ten - tv + tnv) - tev + tnve
    d = 27.0*s*s*p - p*p*((ta - tb)**2 + (tb - tc)**2 + (ta - tc)**2)
    t = ((ta + tb + tc)*p + _sqrt(d))/(3.0*p)
    return torch.where(d >= 0, t, HUGE)


def _iter3d(nb, s, h, p):
    tv, te, tn, tev, ten, tnv, tnve = nb
    t = torch.minimum(torch.minimum(tv + h*s[0], te + h*s[1]), tn + h*s[2])
    for a, b, ab, q in ((te, tv, tev, s[3]), (tv, tn, tnv, s[4]),
                        (te, tn, ten, s[5])):
        v = _plane(ab + a - b, ab - a + b, q, p)
        t = torch.where((a - b).abs() < h*q, torch.minimum(t, v), t)
    tmax = torch.maximum(torch.maximum(tv, te), tn)
    v = _cube(tv, te, tn, tev, ten, tnv, tnve, s[6], p)
    return torch.where(t > tmax, torch.minimum(t, v), t)


def _init3d(nb, s, pos, sg, src, si, s0, eps, h):
    tv, te, tn, tev, ten, tnv, tnve = nb
    p = 1.0/h**2
    t = torch.minimum(torch.minimum(tv + h*s[0], te + h*s[1]), tn + h*s[2])
    tmax = torch.maximum(torch.maximum(tv, te), tn)
    cart = torch.minimum(torch.minimum(tv, te), tn) > eps

    def ana(dz, dx, dy):
        q = [(pos[0] - dz*sg[0] - src[0])*h, (pos[1] - dx*sg[1] - src[1])*h,
             (pos[2] - dy*sg[2] - src[2])*h]
        return s0*torch.sqrt(q[0]**2 + q[1]**2 + q[2]**2), q
    t0, q = ana(0, 0, 0)
    r = torch.where(t0 > 0, s0*s0/t0, torch.zeros_like(t0))
    gz, gx, gy = (sg[k]/h*r*q[k] for k in range(3))   # signed slopes / h
    uv, ue, un = tv - ana(1, 0, 0)[0], te - ana(0, 1, 0)[0], tn - ana(0, 0, 1)[0]
    uev, uen = tev - ana(1, 1, 0)[0], ten - ana(0, 1, 1)[0]
    unv, unve = tnv - ana(1, 0, 1)[0], tnve - ana(1, 1, 1)[0]

    def quad(A, B, C, floor):
        D = B*B - 4.0*A*C
        v = torch.where(D >= 0, (_sqrt(D) - B)/(2.0*A) + t0, HUGE)
        for x in floor:
            v = torch.where(v < x, HUGE, v)
        return v
    for a, b, ab, ua, ub, uab, ga, gb, go, ax, sq in (
            (te, tv, tev, ue, uv, uev, gx, gz, gy, 2, s[3]),
            (tv, tn, tnv, uv, un, unv, gz, gy, gx, 1, s[4]),
            (te, tn, ten, ue, un, uen, gx, gy, gz, 0, s[5])):
        gate = (a - b).abs() < h*sq
        flat = cart | (pos[ax] != si[ax])
        ta, tb = uab + ua - ub, uab - ua + ub
        sph = quad(2.0*p, 4.0*(ga + gb) - 2.0*(ta + tb)*p,
                   (ta**2 + tb**2)*p - 4.0*(ga*ta + gb*tb)
                   + 4.0*(s0*s0 - sq*sq + (go*h)**2), (a, b))
        v = torch.where(flat, _plane(ab + a - b, ab - a + b, sq, p), sph)
        t = torch.where(gate, torch.minimum(t, v), t)
    ta = ue + 0.5*(-un + uen - uv + uev) - unv + unve
    tb = uv + 0.5*(-un + unv - ue + uev) - uen + unve
    tc = un + 0.5*(-ue + uen - uv + unv) - uev + unve
    sph = quad(3.0*p, 6.0*(gz + gx + gy) - 2.0*(ta + tb + tc)*p,
               (ta**2 + tb**2 + tc**2)*p - 6.0*(gx*ta + gz*tb + gy*tc)
               + 9.0*(s0*s0 - s[6]*s[6]), (te, tn, tv))
    v = torch.where(cart, _cube(tv, te, tn, tev, ten, tnv, tnve, s[6], p), sph)
    return torch.where(t > tmax, torch.minimum(t, v), t)


def _plain2d(c, seed):
    """The 2D sweeps of every source, a level at a time: tt[source, x, z]."""
    nz, nx, h = c["nz"], c["nx"], c["h"]
    slow = 1.0/torch.from_numpy(_model2d(c)).to(DEVICE).reshape(nx - 1, nz - 1)
    zs, xs = (torch.from_numpy(v/h).to(DEVICE)[:, None]
              for v in _sources2d(c, seed))
    zi, xi = zs.long(), xs.long()
    s0 = slow[xi, zi]
    n = c["nsrc"]
    tt = torch.full((n, nx, nz), HUGE, dtype=torch.float64, device=DEVICE)
    row = torch.arange(n, device=DEVICE)[:, None]
    for a in (0, 1):
        for b in (0, 1):
            d = torch.hypot(xi + b - xs, zi + a - zs)
            tt[row, xi + b, zi + a] = s0*h*d
    for it in range(c["nsweep"] + 1):
        for sz, sx in ((1, 1), (1, -1), (-1, 1), (-1, -1)):
            flip = [d for d, s in ((1, sz), (0, sx)) if s < 0]
            T = tt.flip([d + 1 for d in flip]).contiguous()
            S = slow.flip(flip)
            for lev in range(2, nz + nx - 1):
                x = torch.arange(max(1, lev - nz + 1), min(nx, lev),
                                 device=DEVICE)
                z = lev - x
                b = z + nz*x
                V = T.reshape(n, -1)
                tv, te, tev, old = V[:, b - 1], V[:, b - nz], \
                    V[:, b - nz - 1], V[:, b]
                s3 = S[x - 1, z - 1]
                s1 = torch.minimum(s3, S[x.clamp(max=nx - 2), z - 1])
                s2 = torch.minimum(s3, S[x - 1, z.clamp(max=nz - 2)])
                new = torch.minimum(tv + h*s1, te + h*s2)
                iz, ix = (z if sz > 0 else nz - 1 - z), (x if sx > 0
                                                         else nx - 1 - x)
                if it == 0:
                    v = _init2d(tv, te, tev, s3, iz, ix, sz, sx, zs, xs, zi,
                                xi, s0, h)
                    box = (z >= (zi if sz > 0 else nz - 2 - zi)) & \
                          (x >= (xi if sx > 0 else nx - 2 - xi))
                    new = torch.where(box, torch.minimum(new, v), HUGE)
                else:
                    v = _plane(tev + te - tv, tev - te + tv, s3, 1.0/h**2)
                    new = torch.where((te - tv).abs() < h*s3,
                                      torch.minimum(new, v), new)
                V[:, b] = torch.minimum(old, new)
            tt = T.flip([d + 1 for d in flip])
    return tt


def _init2d(tv, te, tev, s, iz, ix, sz, sx, zs, xs, zi, xi, s0, h):
    p = 1.0/h**2
    far = ((iz - zi).abs() > EPS2D) | ((ix - xi).abs() > EPS2D)
    out = torch.full_like(tv, HUGE)
    up = (te >= tev) & (tv >= tev)
    g1 = up & ((te - tv).abs() <= h*s)
    g2 = ~g1 & (te - tev <= h*s/math.sqrt(2.0)) & (te > tev)
    g3 = ~g1 & ~g2 & (tv - tev <= h*s/math.sqrt(2.0)) & (tv > tev)
    far_t = torch.where(g1, _plane(tev + te - tv, tev - te + tv, s, p), out)
    far_t = torch.where(g2, te + h*_sqrt(s*s - ((te - tev)/h)**2), far_t)
    far_t = torch.where(g3, tv + h*_sqrt(s*s - ((tv - tev)/h)**2), far_t)

    def ana(a, b):
        return s0*h*torch.hypot(ix - b*sx - xs, iz - a*sz - zs)
    t0 = ana(0, 0)
    r = torch.where(t0 > 0, s0*s0*h/t0, torch.zeros_like(t0))
    gz, gx = sz/h*r*(iz - zs), sx/h*r*(ix - xs)
    uv, ue, uev = tv - ana(1, 0), te - ana(0, 1), tev - ana(1, 1)
    ta, tb = uev + ue - uv, uev - ue + uv
    B = 4.0*(gx + gz) - 2.0*(ta + tb)*p
    C = (ta*ta + tb*tb)*p - 4.0*(gx*ta + gz*tb) + 4.0*(s0*s0 - s*s)
    D = B*B - 8.0*p*C
    near = torch.where(D >= 0, 0.5*(_sqrt(D) - B)/(2.0*p) + t0, HUGE)
    ok = up & ((te - tv).abs() < h*s) & (near >= tv) & (near >= te)
    return torch.where(far, far_t, torch.where(ok, near, out))
