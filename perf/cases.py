"""The work that a user of this framework has it do, as cases to time.

Each case is one pass of a program through the public entry points
(lare3d_amd.device.Device, lare3d_amd.surrogate.Surrogate, and the C-ABI of
include/lare3d_dev.h where that is the interface):

  steps      a run between two dumps: the host fields go to the device, the
             loop body of the driver runs a number of times, and the dump
             comes back (every state array, ghost layers included)
  conduct    conduction super-steps on their own (conduct_heat in a loop)
  sur_heat   the same with the learned surrogate and its residual check
  sur_train  a training job of the surrogate: rows collected from a state,
             standardised, Adam steps; the trained parameters come back
  potential  the potential-field initial condition (red-black SOR)
  energy     energy_account on device arrays that the caller owns

The library holds one device state per process, so a program keeps one open
Device for its grid and parameters, and new inputs are uploaded into it:
that is what prepare() opens and run() uses.  Sizes, parameters and initial
states are those of lare3d_amd.configs, the tests and bench.py.
"""
import ctypes as C
import json
import math

import numpy as np
import torch

from lare3d_amd import BC_OPEN, BC_PERIODIC, BC_USER, configs
from lare3d_amd.abi import EOS_PI, LareFields, PREC_FP32, PREC_FP64, check, load_library
from lare3d_amd.device import Device
from lare3d_amd.fields import KIND, Fields, shape_of
from lare3d_amd.grid import Grid, grid_struct
from lare3d_amd.initial import potential_inputs
from lare3d_amd.surrogate import NCH, Surrogate, initial_params

STATE = ("rho", "energy", "vx", "vy", "vz", "bx", "by", "bz")
DUMP = STATE + ("eta", "visc_dep", "ohmic_dep")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _steps(name, problem, n, steps, precision="fp64", physics="plain", stretch=False, energies=True):
    return {"name": name, "kind": "steps", "problem": problem, "nx": n[0], "ny": n[1], "nz": n[2], "steps": steps,
            "precision": precision, "physics": physics, "stretch": stretch, "energies": energies}


def listed():
    return [
        # the smallest call: the energy diagnostics of a caller's own arrays
        {"name": "energy_64", "kind": "energy", "nx": 64, "ny": 64, "nz": 64},
        # a smoke-sized run, as a user tries a set-up out: every launch counts
        _steps("vortex_16", "orszag_tang", (16, 16, 16), 50, energies=False),
        # the ideal 3-D vortex at a common test resolution
        _steps("vortex_64", "orszag_tang", (64, 64, 64), 100, energies=False),
        # the headline workload: resistive Harris sheet at 256^3 in FP64, with
        # the energies that the driver's output routine makes every step
        _steps("harris_256", "harris", (256, 256, 256), 100),
        # the same sheet in the FP32 mode, as a parameter scan runs it
        _steps("harris_192_fp32", "harris", (192, 192, 192), 100, precision="fp32"),
        # a production-like box: odd, unequal sizes, stretched axes, viscous
        # damping
        _steps("harris_ragged", "harris", (97, 61, 130), 50, physics="damped", stretch=True),
        # the kink-unstable flux tube: resistive with Braginskii conduction,
        # FP32 mode
        _steps("kink_fp32", "kink", (64, 64, 128), 50, precision="fp32"),
        # partially ionised plasma with Cowling resistivity on an odd box
        _steps("harris_ionised", "harris", (45, 37, 41), 30, physics="ionised"),
        # conduction alone: 20 super-steps of about 21 stages on the arcade
        {"name": "arcade_heat", "kind": "conduct", "nx": 64, "ny": 64, "nz": 128, "stages": 21, "steps": 20,
         "precision": "fp64"},
        # surrogate inference with its check, on a held-out sheet
        {"name": "surrogate_heat", "kind": "sur_heat", "nx": 96, "ny": 96, "nz": 96, "stages": 9, "steps": 10,
         "precision": "fp64"},
        # surrogate training: forward, backward and Adam
        {"name": "surrogate_train", "kind": "sur_train", "nx": 32, "ny": 32, "nz": 32, "stages": 5, "rows": 4096,
         "batch": 512, "steps": 200},
        # the initial potential field of an active region above a flux patch
        {"name": "potential_48", "kind": "potential", "nx": 48, "ny": 48, "nz": 40, "periodic": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps"] * 8 + ["conduct", "sur_heat", "sur_train", "potential", "energy"])
    if kind == "energy":
        return {"kind": kind, "nx": _log_int(rng, 8, 200), "ny": _log_int(rng, 8, 200), "nz": _log_int(rng, 8, 200)}
    if kind == "conduct":
        return {"kind": kind, "nx": _log_int(rng, 12, 100), "ny": _log_int(rng, 12, 100), "nz": _log_int(rng, 16, 160),
                "stages": rng.choice([5, 7, 9, 15, 21, 25]), "steps": rng.randint(5, 20),
                "precision": rng.choice(["fp64", "fp64", "fp32"])}
    if kind == "sur_heat":
        n = _log_int(rng, 20, 110)  # the conduction states of the surrogate are cubes
        return {"kind": kind, "nx": n, "ny": n, "nz": n, "stages": rng.choice([5, 7, 9]), "steps": rng.randint(3, 12),
                "precision": rng.choice(["fp64", "fp32"])}
    if kind == "sur_train":
        n = _log_int(rng, 16, 48)
        return {"kind": kind, "nx": n, "ny": n, "nz": n, "stages": rng.choice([3, 5, 7]),
                "rows": _log_int(rng, 500, 8000), "batch": 16 * rng.randint(2, 64), "steps": rng.randint(50, 250)}
    if kind == "potential":
        ny = _log_int(rng, 12, 56)
        return {"kind": kind, "nx": 2 * _log_int(rng, 6, 28), "ny": ny, "nz": min(ny + 2, _log_int(rng, 8, 56)),
                "periodic": rng.random() < 0.3}
    problem = rng.choice(["orszag_tang", "harris", "harris", "harris", "kink"])
    precision = rng.choice(["fp64", "fp64", "fp32"])
    if problem == "orszag_tang":
        n = (_log_int(rng, 10, 180),) * 3
        physics = rng.choice(["plain", "plain", "compression", "rke", "cauchy"])
    elif problem == "kink":
        n = _log_int(rng, 10, 80)
        n = (n, n, 2 * n)
        physics = rng.choice(["plain", "plain", "rk4"] + (["open"] if precision == "fp64" else []))
    else:
        n = tuple(_log_int(rng, 10, 180) for _ in range(3))
        physics = rng.choice(["plain"] * 4 + ["damped", "damped", "rke", "cauchy", "rk4", "limiter"] +
                             (["open", "ionised"] if precision == "fp64" else []))
    cells = n[0] * n[1] * n[2]
    steps = max(8, min(100, int(rng.uniform(0.3, 1.0) * 3.0e8 / cells)))
    if physics == "ionised":
        steps = min(steps, 30)
    c = _steps("", problem, n, steps, precision, physics, problem == "harris" and rng.random() < 0.4,
               rng.random() < 0.6)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# states
# ---------------------------------------------------------------------------
class _Held:
    """The one open Device of this process, and the case it was opened for."""
    key = None
    dev = None


def _close():
    if Device._open is not None:
        Device._open.close()
    _Held.key = _Held.dev = None


def _device(case, grid, params, fields):
    key = json.dumps({k: v for k, v in case.items() if k not in ("name", "steps", "energies", "stages")},
                     sort_keys=True)
    if _Held.key != key or _Held.dev is None or _Held.dev.lib is None:
        _close()
        _Held.dev = Device(grid, params, fields)
        _Held.key = key
    return _Held.dev


def _initial(case, seed):
    """(grid, params, fields, dt) of a case; dt is None where the step sets it."""
    n = (case["nx"], case["ny"], case["nz"])
    kind, problem = case["kind"], case.get("problem")
    rng = np.random.default_rng(seed)
    dt = None
    if kind in ("sur_heat", "sur_train"):
        grid, params, f, dt = configs.harris_conduction(n[0], seed=seed % 100003, s_target=case["stages"])
    elif kind == "conduct":
        grid, params, f, dt = configs.arcade_conduction(*n, s_target=case["stages"])
        # hot plasma is not smooth: a seeded unevenness of the temperature
        f.energy *= 1.0 + 0.1 * rng.random(f.energy.shape)
        dt *= 0.9
    elif problem == "orszag_tang":
        grid, params, f = configs.orszag_tang(n[0])
    elif problem == "kink":
        grid, params, f = configs.kink_tube(*n)
    else:
        damping = 0.05 if case["physics"] == "damped" else None
        stretch = (24.0, 10.0, 24.0) if case["stretch"] else (None, None, None)
        grid, params, f = configs.harris(n[0], seed=seed, ny=n[1], nz=n[2], stretch=stretch, damping=damping)
    if problem in ("orszag_tang", "kink"):
        for v in (f.vx, f.vy, f.vz):
            v += 0.01 * (2.0 * rng.random(v.shape) - 1.0)
    physics = case.get("physics", "plain")
    if physics == "open":
        bcs = (BC_OPEN,) * 4 if problem == "kink" else (BC_PERIODIC, BC_PERIODIC, BC_OPEN, BC_OPEN)
        grid = Grid(*grid.n, grid.extent, bcs + (BC_PERIODIC, BC_PERIODIC), grid.stretch, grid.widths)
    elif physics == "ionised":
        configs.partially_ionised((grid, params, f), EOS_PI, 1)
    elif physics != "plain" and physics != "damped":
        setattr(params, {"rke": "rke", "cauchy": "cauchy", "rk4": "fourth_order", "limiter": "shock_limiter",
                         "compression": "shock_compression"}[physics], 1)
    params.precision = PREC_FP32 if case.get("precision") == "fp32" else PREC_FP64
    return grid, params, f, dt


def _norm(f, params, grid, dt):
    """Channel means and spreads of a state, as a trained network would carry
    them, and an output scale of a thousandth of the temperature's spread."""
    s = slice(2, -2)
    T = (params.gamma - 1.0) / (2.0 - params.xi_n) * f.energy
    b = [0.5 * (f.interior(q) + f.view(q, *lo)) for q, lo in (
        ("bx", (0, grid.nx - 1, 1, grid.ny, 1, grid.nz)), ("by", (1, grid.nx, 0, grid.ny - 1, 1, grid.nz)),
        ("bz", (1, grid.nx, 1, grid.ny, 0, grid.nz - 1)))]
    bm = np.sqrt(b[0] ** 2 + b[1] ** 2 + b[2] ** 2)
    grads = [g[s, s, s] for g in np.gradient(T, *(float(grid.dxb[a][2]) for a in range(3)))]
    chan = [T[s, s, s]] + [c / np.maximum(bm, 1e-30) for c in b] + [f.interior("rho"), np.array([math.log(dt)]), bm]
    chan += grads
    assert len(chan) == NCH
    sd = [float(c.std()) for c in chan]
    return ([float(c.mean()) for c in chan], [v if v > 1e-6 else 1.0 for v in sd], 1e-3 * sd[0])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "energy":
        return _prepare_energy(case, seed)
    if kind == "potential":
        s = _potential(case, seed)
        _device(case, s["grid"], s["params"], s["fields"])
        return s
    grid, params, f, dt = _initial(case, seed)
    s = {"case": case, "grid": grid, "params": params, "fields": f, "dt": dt, "seed": seed}
    if kind in ("sur_heat", "sur_train"):
        s["weights"] = initial_params(seed)
    if kind == "sur_heat":
        s["norm"] = _norm(f, params, grid, dt)
    if kind != "sur_train":
        _device(case, grid, params, f)
    return s


def _potential(case, seed):
    rng = np.random.default_rng(seed)
    n = (case["nx"], case["ny"], case["nz"])
    xbc = BC_PERIODIC if case["periodic"] else BC_USER
    grid = Grid(*n, ((-5.0, 15.0), (-10.0, 10.0), (0.0, 20.0)), (xbc, xbc) + (BC_USER,) * 4)
    f = Fields(*n)
    f.rho[...] = 1.0
    f.energy[...] = 1.0
    pf = potential_inputs(grid, centre=rng.uniform(3.0, 7.0), radius=rng.uniform(1.5, 3.0))
    return {"case": case, "grid": grid, "params": configs.default_params(), "fields": f, "pf": pf}


def _prepare_energy(case, seed):
    """The caller's own device arrays in the Fortran layout, x fastest."""
    n = (case["nx"], case["ny"], case["nz"])
    grid = Grid(*n, ((0.0, 2.0 * math.pi),) * 3, (BC_PERIODIC,) * 6)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    bufs = {}
    for q in STATE:
        shape = shape_of(KIND[q], n)
        u = torch.rand(shape[::-1], generator=gen, device="cuda", dtype=torch.float64)
        bufs[q] = 0.5 + u if q in ("rho", "energy") else 2.0 * u - 1.0
    st = LareFields()
    for q, t in bufs.items():
        setattr(st, q, _pointer(t))
    # the entry point works on the null stream of its own: the arrays are
    # complete before they are handed over
    torch.cuda.synchronize()
    return {"case": case, "grid": grid, "gs": grid_struct(grid), "bufs": bufs, "st": st, "lib": load_library()}


def _pointer(t):
    return C.cast(C.c_void_p(t.data_ptr()), C.POINTER(C.c_double))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
FRESH = dict(dt=0.0, dtr=0.0, time=0.0, total_visc_heating=0.0, total_ohmic_heating=0.0, n_s_stages=0,
             peak_substeps=0, last_substeps=0, first_set_dt=1, step=0)


def _load(s):
    dev = _device(s["case"], s["grid"], s["params"], s["fields"])
    dev.upload(s["fields"])
    dev.set_scalars(**dict(FRESH, dt=s.get("dt") or 0.0))
    dev.boundary_conditions()
    return dev


def _dump(dev, names):
    f = dev.fields()
    return {q: getattr(f, q) for q in names}


def _run_steps(s):
    c, p = s["case"], s["params"]
    dev = _load(s)
    dev.eta_calc()
    if c["physics"] == "ionised":
        dev.neutral_fraction()
        dev.perpendicular_resistivity()
    log = []
    for q in range(1, c["steps"] + 1):
        if c["energies"]:
            i = dev.step_info(q, with_energy=True)
            log.append((i.dt, i.time, i.en_b, i.en_ke, i.en_int, i.total_visc_heating, i.total_ohmic_heating))
        else:
            log.append(dev.step(q))
    sc = dev.scalars()
    out = _dump(dev, DUMP)
    out["log"] = np.array(log)
    out["counts"] = [sc.n_s_stages if p.conduction else 0, sc.last_substeps, sc.peak_substeps]
    return out


def _run_conduct(s):
    dev = _load(s)
    for _ in range(s["case"]["steps"]):
        dev.conduct_heat()
    out = _dump(dev, ("energy",))
    out["stages"] = dev.scalars().n_s_stages
    return out


def _run_sur_heat(s):
    dev = _load(s)
    sur = Surrogate(dev)
    sur.set_params(s["weights"])
    sur.set_norm(*s["norm"])
    # every other super-step is held to a tolerance that this network misses,
    # so that the fallback to the plain solver is in the pass too
    log = []
    for q in range(s["case"]["steps"]):
        sur.enable(False, 1.0e30 if q % 2 == 0 else 1.0e-9)
        log.append(sur.conduct())
    out = _dump(dev, ("energy",))
    out["residual"] = np.array([r for r, _ in log])
    out["accepted"] = [int(a) for _, a in log]
    return out


def _run_sur_train(s):
    c = s["case"]
    _close()
    dev = Device(s["grid"], s["params"], s["fields"])
    try:
        dev.boundary_conditions()
        dev.set_scalars(dt=s["dt"])
        sur = Surrogate(dev)
        sur.set_params(s["weights"])
        sur.collect(c["rows"], 500 + s["seed"] % 1000)
        sur.fit_norm()
        loss = sur.train(c["steps"], batch=c["batch"], lr=1e-3, seed=9 + s["seed"] % 1000)
        return {"params": sur.params(), "loss": loss}
    finally:
        dev.close()


def _run_potential(s):
    dev = _load(s)
    it, res, bm = dev.potential_field(s["pf"])
    out = _dump(dev, ("bx", "by", "bz"))
    out["iterations"], out["residual"], out["bz_max"] = it, res, bm
    return out


def _run_energy(s):
    en, divb = (C.c_double * 3)(), C.c_double()
    check(s["lib"], s["lib"].lare_dev_energy_account_noalloc(C.byref(s["gs"]), C.byref(s["st"]), en, C.byref(divb)),
          "energy_account_noalloc")
    return {"energies": np.array(en), "divb": divb.value}


RUN = {"steps": _run_steps, "conduct": _run_conduct, "sur_heat": _run_sur_heat, "sur_train": _run_sur_train,
       "potential": _run_potential, "energy": _run_energy}


def run(state):
    return RUN[state["case"]["kind"]](state)


# ---------------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------------
def work(case):
    """Each step (super-step, iteration) reads its state and writes it once;
    the host arrays of the upload and the dump count once each.  Operations
    per cell are counted from the reference's loops, a division or root as
    one."""
    cells = float(case["nx"] * case["ny"] * case["nz"])
    word = 4.0 if case.get("precision") == "fp32" else 8.0
    kind = case["kind"]
    if kind == "energy":
        return {"bytes": 8 * 8.0 * cells, "flops": 90 * cells}
    if kind == "potential":
        its = 4.0 * max(case["nx"], case["ny"], case["nz"])  # about the iterations SOR takes at its fixed w
        return {"bytes": (8 + 3) * 8.0 * cells + its * 2 * 8.0 * cells, "flops": its * 16 * cells}
    if kind == "sur_train":
        par = 336 * 64 + 64 * 64 + 64
        return {"bytes": 8 * 8.0 * cells + case["steps"] * 4.0 * (336 * case["batch"] + 7 * par),
                "flops": case["steps"] * 6.0 * par * case["batch"]}
    if kind in ("conduct", "sur_heat"):
        net = 2.0 * (324 * 64 + 64 * 64 + 64) if kind == "sur_heat" else 0.0
        # per super-step: energy in and out, density and B in
        return {"bytes": (11 + 1) * 8.0 * cells + case["steps"] * (3 * word + 3 * 8.0) * cells,
                "flops": case["steps"] * (case["stages"] * 190.0 + net) * cells}
    ops = 1900.0
    if case["problem"] != "orszag_tang":
        ops += 2 * 110.0
    if case["problem"] == "kink":
        ops += 5 * 190.0
    return {"bytes": 2 * 11 * 8.0 * cells + case["steps"] * 2 * (5 * word + 3 * 8.0) * cells,
            "flops": case["steps"] * ops * cells}


# ---------------------------------------------------------------------------
# 64-bit values from plain numpy
# ---------------------------------------------------------------------------
def exact(case, seed):
    """The diagnostics and the potential field in plain 64-bit numpy.  The
    other kinds are evolutions over tens to hundreds of steps: in numpy they
    take longer than a check may, so their outputs have no value here."""
    if case["kind"] == "energy":
        return _exact_energy(case, seed)
    if case["kind"] == "potential":
        return _exact_potential(case, seed)
    return None


def _exact_energy(case, seed):
    s = _prepare_energy(case, seed)
    a = {q: t.cpu().numpy().transpose(2, 1, 0) for q, t in s["bufs"].items()}
    grid = s["grid"]
    nx, ny, nz = grid.n
    w = [np.asarray(grid.dxb[q]) for q in range(3)]  # [i + 1]
    cv = w[0][:, None, None] * w[1][None, :, None] * w[2][None, None, :]
    inner = (slice(2, nx + 2), slice(2, ny + 2), slice(2, nz + 2))  # cells 1..n of arrays from -1

    def faces(q, ax):
        hi = [slice(2, m + 2) for m in grid.n]
        lo = list(hi)
        hi[ax], lo[ax] = slice(3, grid.n[ax] + 3), slice(2, grid.n[ax] + 2)
        return a[q][tuple(hi)], a[q][tuple(lo)]

    en_b, div = 0.0, 0.0
    for ax, q in enumerate(("bx", "by", "bz")):
        hi, lo = faces(q, ax)
        en_b = en_b + 0.5 * (hi * hi + lo * lo)
        shape = [1, 1, 1]
        shape[ax] = -1
        div = div + (hi - lo) / w[ax][2:grid.n[ax] + 2].reshape(shape)
    en_b = float((0.5 * en_b * cv[inner]).sum())
    en_int = float((a["energy"][inner] * a["rho"][inner] * cv[inner]).sum())
    dmin = np.minimum(np.minimum(w[0][2:nx + 2][:, None, None], w[1][2:ny + 2][None, :, None]),
                      w[2][2:nz + 2][None, None, :])
    m, v = 0.0, 0.0
    for o in np.ndindex(2, 2, 2):  # the eight cells of the nodes 0..n
        sl = tuple(slice(1 + o[q], grid.n[q] + 2 + o[q]) for q in range(3))
        m = m + (a["rho"] * cv)[sl]
        v = v + cv[sl]
    N = tuple(slice(2, q + 3) for q in grid.n)
    ke = 0.5 * (m / v) * (v / 8.0) * (a["vx"][N] ** 2 + a["vy"][N] ** 2 + a["vz"][N] ** 2)
    for ax in range(3):  # nodes on a boundary plane belong to it by half
        for edge in (0, -1):
            sl = [slice(None)] * 3
            sl[ax] = edge
            ke[tuple(sl)] *= 0.5
    return {"energies": np.array([en_b, float(ke.sum()), en_int]), "divb": float((np.abs(div) * dmin).max())}


def _exact_potential(case, seed):
    s = _potential(case, seed)
    grid, pf, per = s["grid"], s["pf"], case["periodic"]
    nx, ny, nz = grid.n
    flux = pf._keep.reshape((nx, ny), order="F")
    d = (pf.dx1, pf.dy1, pf.dz1)
    phi = np.zeros((nz + 4, ny + 4, nx + 4))  # phi(i, j, k) at [k + 1, j + 1, i + 1]
    X, Y = slice(2, nx + 2), slice(2, ny + 2)
    colour = (np.arange(1, ny + 1)[:, None] + np.arange(1, nx + 1)[None, :]) % 2

    def fill():
        if per:
            phi[:, :, nx + 2:], phi[:, :, :2] = phi[:, :, 2:4].copy(), phi[:, :, nx:nx + 2].copy()
        phi[1, Y, X] = phi[2, Y, X] + flux.T
        phi[0, Y, X] = phi[1, Y, X]
        phi[nz + 2:] = 0.0
        if not per:
            phi[:, :, :2], phi[:, :, nx + 2:] = phi[:, :, 2:3], phi[:, :, nx + 1:nx + 2]
        phi[:, :2], phi[:, ny + 2:] = phi[:, 2:3], phi[:, ny + 1:ny + 2]

    its, res = 0, 0.0
    while True:
        res = 0.0
        for par in (0, 1):
            at = colour == par
            for k in range(2, nz + 2):
                p = phi[k]
                cur = p[Y, X]
                r = ((p[Y, 3:nx + 3] - 2.0 * cur + p[Y, 1:nx + 1]) * d[0] +
                     (p[3:ny + 3, X] - 2.0 * cur + p[1:ny + 1, X]) * d[1] +
                     (phi[k + 1, Y, X] - 2.0 * cur + phi[k - 1, Y, X]) * d[2]) / 2.0 / sum(d)
                r = np.where(at, r, 0.0)
                res = max(res, float(np.abs(r).max()))
                p[Y, X] = cur + pf.omega * r
            fill()
        its += 1
        if res < pf.fractional_error or its >= pf.max_iterations:
            break
    B = {}
    for ax, q in enumerate(("bx", "by", "bz")):
        b = np.zeros(shape_of(KIND[q], grid.n))
        hi = [slice(2, m + 2) for m in grid.n]
        lo = list(hi)
        lo[ax] = slice(1, grid.n[ax] + 2)
        hi[ax] = slice(2, grid.n[ax] + 3)
        dst = [slice(2, m + 2) for m in grid.n]
        dst[ax] = slice(2, grid.n[ax] + 3)
        t = phi.transpose(2, 1, 0)
        shape = [1, 1, 1]
        shape[ax] = -1
        b[tuple(dst)] = -(t[tuple(hi)] - t[tuple(lo)]) / np.asarray(grid.dxc[ax])[1:grid.n[ax] + 2].reshape(shape)
        B[q] = b

    def ghosts():
        for axis in sorted(range(3), key=lambda x: 0 if (per and x == 0) else 1):
            m = grid.n[axis]
            for q, b in B.items():
                v = np.moveaxis(b, axis, 0)
                face = "xyz"[axis] == q[1]
                z = 2 if face else 1  # index of layer 0
                if per and axis == 0:
                    src = {m + 1: 1, m + 2: 2, -1: m - 1, 0: m}
                    if face:
                        src[-2] = m - 2
                elif face:
                    src = {-1: 1, -2: 2, m + 1: m - 1, m + 2: m - 2}
                else:
                    src = {0: 1, -1: 2, m + 1: m, m + 2: m - 1}
                new = {dst: v[z + sc].copy() for dst, sc in src.items()}
                for dst, val in new.items():
                    v[z + dst] = val

    ghosts()
    bm = float(B["bz"][2:nx + 2, 2:nz + 2, 2].max())
    for b in B.values():
        b /= bm
    ghosts()
    return {"bx": B["bx"], "by": B["by"], "bz": B["bz"], "iterations": its, "residual": res, "bz_max": bm}
