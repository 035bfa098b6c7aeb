"""Performance cases of the framework: what a program that uses it has it do.

Every case advances (or diagnoses) device-resident members through the public
entry points of the C ABI as epic_amd binds it, and hands the result fields
back.  The listed cases are the configurations this repository benchmarks,
tests and serves; draw() gives others of the same ranges.

Members are taken past the Adams-Bashforth start-up (two steps) in prepare():
a long run spends its time in the third-order steps that follow.  An engine
case steps and then reads its fields into pinned host arrays, as a program
that writes output every few steps does; the diagnostics case works on the
caller's own device arrays.

Comparisons with 64-bit values: exact() restates the hydrostatic diagnostics
(pressure, temperature, density, geopotential) in numpy.  A whole step has no
such short form; its FP64 results are held to the start's by their type.
"""
import ctypes
import math

import numpy as np
import torch

import epic_amd as ea

# prognostic state, and two diagnostics whose formation spans the whole step
STATE = ("U", "V", "HDRY", "THETA", "P3")
STATE_DIAG = STATE + ("GZ3", "PV3", "W3")
LARGE = 16_000_000  # points from which a program writes out the state alone


def listed():
    return [
        # The smallest calls: a teaching- or tuning-size run looked at every
        # few steps.  Launches and latency decide, not bandwidth.
        dict(name="venus_32x19x7_fp64", planet=ea.VENUS_LIKE, ni=32, nj=19, nk=7, dt=300, members=1, mixed=False,
             steps=5),
        # The dry-Earth benchmark of Held & Suarez at its usual coarse grid.
        dict(name="held_suarez_64x32x10_fp64", planet=ea.HELD_SUAREZ, ni=64, nj=32, nk=10, dt=600, members=1,
             mixed=False, steps=10),
        # One gas-giant integration, the configuration of the benchmark, in
        # both precision modes.
        dict(name="jupiter_256x128x20_fp64", planet=ea.JUPITER_LIKE, ni=256, nj=128, nk=20, dt=60, members=1,
             mixed=False, steps=20),
        dict(name="jupiter_256x128x20_mixed", planet=ea.JUPITER_LIKE, ni=256, nj=128, nk=20, dt=60, members=1,
             mixed=True, steps=20),
        # An ensemble: 64 members of one grid in every launch.
        dict(name="jupiter_ensemble_64x128x64x16_mixed", planet=ea.JUPITER_LIKE, ni=128, nj=64, nk=16, dt=60,
             members=64, mixed=True, steps=8),
        # A ragged ensemble in FP64: odd rows and levels, a member count that
        # fills no tile.
        dict(name="saturn_ensemble_23x128x51x13_fp64", planet=ea.SATURN_LIKE, ni=128, nj=51, nk=13, dt=60, members=23,
             mixed=False, steps=10),
        # The options a study turns on together: monotonized fourth-order
        # advection of both fields, Arakawa-Lamb PV averaging, del^8 (the
        # reference's default order), divergence damping, Rayleigh drag and
        # the relaxation to a sounding.
        dict(name="saturn_128x64x20_options_fp64", planet=ea.SATURN_LIKE, ni=128, nj=64, nk=20, dt=60, members=1,
             mixed=False, steps=10, nu4=0.0, nu8=0.5, nudiv=0.1, adv_mass=1, adv_nonmass=1, pv_scheme=1, newt_cool=1,
             tau_drag=2.0e4, drag_v=1),
        # What the request loop holds at one moment: members of three grids,
        # several launch buckets in one step.
        dict(name="serving_mix_mixed", mix=True, mixed=True, steps=10),
        # The largest request of the serving mix.
        dict(name="jupiter_512x256x32_mixed", planet=ea.JUPITER_LIKE, ni=512, nj=256, nk=32, dt=30, members=1,
             mixed=True, steps=10),
        # The largest domain one GPU is given, in both precision modes.
        dict(name="hot_jupiter_1024x512x64_fp64", planet=ea.HOT_JUPITER, ni=1024, nj=512, nk=64, dt=30, members=1,
             mixed=False, steps=10),
        dict(name="hot_jupiter_1024x512x64_mixed", planet=ea.HOT_JUPITER, ni=1024, nj=512, nk=64, dt=30, members=1,
             mixed=True, steps=10),
        # The priming call of a caller that owns the device arrays: every
        # diagnostic of one state, no step.
        dict(name="diagnostics_venus_256x128x20", planet=ea.VENUS_LIKE, ni=256, nj=128, nk=20, dt=75, diagnose=True),
    ]


# a stable timestep per planet and row length (dt scales with the spacing)
_DT = {
    ea.HELD_SUAREZ: {16: 900, 32: 600, 64: 400, 128: 200},
    ea.VENUS_LIKE: {16: 300, 32: 300, 64: 200, 128: 100, 256: 30, 512: 15},
    ea.JUPITER_LIKE: {16: 60, 32: 60, 64: 60, 128: 60, 256: 40, 512: 30, 1024: 15},
    ea.SATURN_LIKE: {16: 60, 32: 60, 64: 60, 128: 60, 256: 40, 512: 25},
    ea.HOT_JUPITER: {64: 30, 128: 30, 256: 30, 512: 30, 1024: 30},
}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    planet = rng.choice(sorted(_DT))
    ni = rng.choice(sorted(_DT[planet]))
    nj = max(8, rng.randint(int(0.42 * ni), int(0.53 * ni)))
    nk = _log_int(rng, 5, 12 if planet == ea.HELD_SUAREZ else 40)
    if ni <= 256 and rng.random() < 0.15:  # bounded by the static working memory of the call
        nk = max(4, min(nk, 700_000 // ((ni + 2) * (nj + 3)) - 2))
        return dict(planet=planet, ni=ni, nj=nj, nk=nk, dt=_DT[planet][ni], diagnose=True)
    points = ni * (nj + 1) * nk
    members = max(1, min(64, _log_int(rng, 1, max(1, 6_000_000 // points)))) if points < 6_000_000 else 1
    case = dict(planet=planet, ni=ni, nj=nj, nk=nk, dt=_DT[planet][ni], members=members, mixed=rng.random() < 0.5,
                steps=_log_int(rng, 3, 20))
    # options, each as a study would add it to the defaults
    if rng.random() < 0.2:
        case["adv_mass"] = 1
    if rng.random() < 0.2:
        case["adv_nonmass"] = 1
    if rng.random() < 0.15:
        case["pv_scheme"] = 1
    if planet in (ea.JUPITER_LIKE, ea.SATURN_LIKE) and rng.random() < 0.2:
        case["pgrad_traditional"] = 1
    if rng.random() < 0.2:
        case["nudiv"] = 0.1
    if rng.random() < 0.15:
        case.update(nu4=0.25, nu6=0.2)
    if rng.random() < 0.15:
        case.update(tau_drag=2.0e4, drag_v=1)
    if planet in (ea.JUPITER_LIKE, ea.SATURN_LIKE, ea.VENUS_LIKE) and rng.random() < 0.2:
        case["newt_cool"] = 1
    return case


def _spec(planet, ni, nj, nk, dt, seed, **opt):
    """The seeded initial state of a planet: jets and 0.5 m/s of noise on the
    gas giants, 1 K of theta noise on the hot Jupiter at rest (levels without
    a sponge), 0.1 K on the terrestrial planets."""
    opt.setdefault("nu4", 0.5)
    if planet == ea.HOT_JUPITER:
        opt.setdefault("k_sponge", 0)
        return ea.spec(planet, ni, nj, nk, dt, seed=seed, noise_theta=1.0, noise_uv=0.0, **opt)
    gas = planet in (ea.JUPITER_LIKE, ea.SATURN_LIKE)
    return ea.spec(planet, ni, nj, nk, dt, seed=seed, noise_theta=0.0 if gas else 0.1, noise_uv=0.5 if gas else 0.1,
                   **opt)


_OPTIONS = ("nu4", "nu6", "nu8", "nudiv", "adv_mass", "adv_nonmass", "pv_scheme", "pgrad_traditional", "newt_cool",
            "tau_drag", "drag_v")


def _specs(case, seed):
    base = 1 + seed * 1009
    if case.get("mix"):
        kinds = [(ea.HELD_SUAREZ, 64, 32, 10, 600)] * 3 + [(ea.JUPITER_LIKE, 128, 64, 16, 60)] * 3 + \
                [(ea.VENUS_LIKE, 128, 64, 16, 150), (ea.SATURN_LIKE, 256, 128, 20, 60)]
        return [_spec(*k, base + m) for m, k in enumerate(kinds)]
    opt = {k: case[k] for k in _OPTIONS if k in case}
    return [_spec(case["planet"], case["ni"], case["nj"], case["nk"], case["dt"], base + m, **opt)
            for m in range(case.get("members", 1))]


def _shape(sp):
    return tuple(reversed(ea.dims(sp)))


def _fields(case, specs):
    return STATE if sum(s.ni * (s.nj + 1) * s.nk for s in specs) >= LARGE else STATE_DIAG


class _Run:
    """An engine with its members past the start-up steps, and the pinned
    arrays its fields are read into (members of one grid stacked)."""

    def __init__(self, case, seed):
        specs = _specs(case, seed)
        self.steps = case["steps"]
        self.engine = ea.Engine(ea.MIXED if case["mixed"] else ea.FP64, len(specs))
        slots = [self.engine.add(sp) for sp in specs]
        self.engine.step(2)
        self.engine.wait()
        names = _fields(case, specs)
        self.out, self.reads = [], []
        for shape in sorted({_shape(sp) for sp in specs}):
            mine = [s for s, sp in zip(slots, specs) if _shape(sp) == shape]
            group = {f: torch.empty((len(mine),) + shape, dtype=torch.float64, pin_memory=True) for f in names}
            self.out.append(group)
            for m, s in enumerate(mine):
                for f, t in group.items():
                    self.reads.append((s, ea.FIELD[f], t[m].data_ptr()))


class _Diag:
    """One member's fields in the caller's own device arrays."""

    def __init__(self, case, seed):
        sp = _specs(case, seed)[0]
        self.case = ea.build_case(sp)
        host = _initial(self.case, sp)
        n3 = int(np.prod(_shape(sp)))
        zero = lambda n: torch.zeros(n, dtype=torch.float64, device="cuda")  # noqa: E731
        self.t = {f: zero(n3) for f in ea.FIELDS if f[:4] not in ("DUDT", "DVDT")}
        self.t["GZ_SURFACE"] = zero(n3 // _shape(sp)[0])
        self.t["DUDT"], self.t["DVDT"] = zero(3 * n3), zero(3 * n3)
        for f in ("U", "V", "THETA", "P3", "HDRY", "GZ_SURFACE"):
            self.t[f].copy_(torch.from_numpy(np.ascontiguousarray(host[f]).reshape(-1)))
        self.ptrs = (ctypes.c_void_p * len(ea.FIELDS))()
        for q, f in enumerate(ea.FIELDS):
            if f[:4] in ("DUDT", "DVDT"):
                self.ptrs[q] = self.t[f[:4]].data_ptr() + 8 * n3 * int(f[4])
            else:
                self.ptrs[q] = self.t[f].data_ptr()
        self.err = ctypes.create_string_buffer(256)
        self.fn = ea.lib().epic_step_noalloc
        self.fn.restype = ctypes.c_int
        self.fn.argtypes = [ctypes.POINTER(ea.Case), ctypes.POINTER(ctypes.c_void_p), ctypes.POINTER(ctypes.c_int),
                            ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_char_p, ctypes.c_size_t]
        self.shape = _shape(sp)
        self.out = {f: self.t[f].view(self.shape) for f in DIAGNOSED}

    def __del__(self):
        ea.free_case(self.case)


# what the diagnosing call forms
DIAGNOSED = ("P3", "HDRY", "THETA", "P2", "H3", "THETA2", "T2", "T3", "RHO2", "RHO3", "EXNER3", "GZ3", "MONT3", "PV3",
             "DIV_UV3", "W3", "RI2")


def _initial(c, sp):
    """The prognostic fields of a built case; h from the layers' pressure
    thickness over g dsgth, periodic in longitude."""
    K, J, I = _shape(sp)
    a = {f: c.array(f.lower(), K * J * I).reshape(K, J, I) for f in ("U", "V", "THETA", "P3")}
    a["GZ_SURFACE"] = c.array("gz_surface", J * I)
    g, dsg = c.array("g", 2 * sp.nj + 3)[1::2], c.array("dsgth", 2 * sp.nk + 3)
    h = np.zeros((K, J, I))
    rows, cols = slice(1, sp.nj + 2), slice(1, sp.ni + 1)
    h[1:sp.nk + 1, rows, cols] = np.diff(a["P3"][:sp.nk + 1, rows, cols], axis=0) / (
        g[None, :sp.nj + 1, None] * dsg[2:2 * sp.nk + 1:2, None, None])
    h[:, :, 0], h[:, :, sp.ni + 1] = h[:, :, sp.ni], h[:, :, 1]
    a["HDRY"] = h
    return a


def prepare(case, seed):
    return _Diag(case, seed) if case.get("diagnose") else _Run(case, seed)


def run(state):
    if isinstance(state, _Diag):
        it = (ctypes.c_int * 4)(0, 1, 2, 0)
        rc = state.fn(ctypes.byref(state.case), state.ptrs, it, ea.SYNC_DIAGS_ONLY, 0,
                      torch.cuda.current_stream().cuda_stream, state.err, len(state.err))
        if rc:
            raise ea.EpicError(state.err.value.decode())
        return state.out
    state.engine.step(state.steps)
    read, handle = ea.lib().epic_engine_read, state.engine._e
    for slot, field, ptr in state.reads:
        if read(handle, slot, field, ptr):
            raise ea.EpicError("read failed")
    return state.out


def work(case):
    """A step must read and write u, v, h, theta and the Adams-Bashforth
    history once (two planes of each wind in, one out: 112 B a point with an
    FP64 history, 88 B with FP32); every field handed back is written once.
    The operations are those of the step's expressions per point, a division,
    square root or transcendental counted as one."""
    specs = _specs(case, 0)
    points = sum(s.ni * (s.nj + 1) * s.nk for s in specs)
    if case.get("diagnose"):
        return {"bytes": points * 8 * (5 + len(DIAGNOSED)), "flops": points * 250}
    steps = case["steps"]
    per = 88 if case["mixed"] else 112
    return {"bytes": points * (per * steps + 8 * len(_fields(case, specs))), "flops": points * 1500 * steps}


def exact(case, seed):
    """The hydrostatic diagnostics of a terrestrial planet's state (its
    surface geopotential is given; a gas giant's follows from its winds)."""
    if not case.get("diagnose"):
        return None
    sp = _specs(case, seed)[0]
    c = ea.build_case(sp)
    try:
        return _hydrostatics(c, sp, _initial(c, sp))
    finally:
        ea.free_case(c)


def _hydrostatics(c, sp, a):
    ni, nj, nk, ks = sp.ni, sp.nj, sp.nk, c.k_sigma
    R = 8.314472e3
    sg, dsg = c.array("sigmatheta", 2 * nk + 3), c.array("dsgth", 2 * nk + 3)
    g = c.array("g", 2 * nj + 3)[1::2][:nj + 1][:, None]
    hmin = c.array("h_min", nk + 2)
    kap, p0 = c.kappa, c.press0
    out = {f: np.zeros(_shape(sp)) for f in DIAGNOSED}
    for f in ("P3", "HDRY", "THETA"):
        out[f] = a[f].copy()
    rows = slice(1, nj + 2)
    # pressure from the top down; sigma levels follow the column's bottom
    P = np.empty((nk + 1,) + a["P3"].shape[1:])[:, rows]
    P[0] = a["P3"][0, rows]
    for K in range(1, nk + 1):
        P[K] = P[K - 1] + dsg[2 * K] * g * a["HDRY"][K, rows]
    lr = np.log(P[0] / P[nk])
    for K in range(ks - 1, nk):
        P[K] = P[nk] * np.exp((sg[2 * K + 1] - c.zeta0) / (c.zeta1 - c.zeta0) * lr)

    def theta_at(level, p):
        s = np.log(p / P[nk]) / lr
        gs = (1. - np.exp(-c.hybrid_alpha * (s - c.sigma_sigma))) / (
            1. - math.exp(-c.hybrid_alpha * (1. - c.sigma_sigma)))
        return (sg[level] - (1. - gs) * (c.zeta0 + s * (c.zeta1 - c.zeta0))) / gs

    TH, TH2, P2, H, H3 = (np.zeros_like(P) for _ in range(5))
    TH[:] = a["THETA"][:nk + 1, rows]
    for K in range(0, ks - 1):
        TH[K] = theta_at(2 * K + 1, P[K])
    for K in range(1, nk + 1):
        H[K] = (P[K] - P[K - 1]) / (g * dsg[2 * K])
        P2[K] = ((P[K] ** (kap + 1.) - P[K - 1] ** (kap + 1.)) / ((kap + 1.) * (P[K] - P[K - 1]))) ** (1. / kap)
    for K in range(1, nk):
        H3[K] = (dsg[2 * K] * H[K] + dsg[2 * K + 2] * H[K + 1]) / (dsg[2 * K] + dsg[2 * K + 2])
    H3[nk], H3[0] = H[nk], H3[1]
    P2[0] = P[0] * P[0] / P2[1]
    for K in range(1, nk + 1):
        if K < ks - 1:
            TH2[K] = theta_at(2 * K, P2[K])
        elif K == ks - 1:
            TH2[K] = .5 * (TH[K] + TH[K - 1])
        else:
            w = (sg[2 * K] - sg[2 * K + 1]) / (sg[2 * K - 1] - sg[2 * K + 1])
            TH2[K] = TH[K] + w * (TH[K - 1] - TH[K])
    TH2[0] = sg[0]
    mu = R / c.rgas
    T3 = TH * (P / p0) ** kap
    T2 = TH2 * (P2 / p0) ** kap
    RHO3, RHO2 = P * mu / (R * T3), P2 * mu / (R * T2)
    T2[0], RHO2[0] = T3[0], RHO3[0] ** 2 / RHO2[1]
    G = np.zeros_like(P)
    G[nk] = c.topo_scale * a["GZ_SURFACE"].reshape(nj + 3, ni + 2)[rows]
    # the four-point integral of p/rho in ln p, one-sided at the ends
    lg = np.zeros_like(P)
    lg[1:] = np.log(P[1:] / P[:-1])
    q = P / RHO3
    for K in range(nk, 0, -1):
        if K in (1, nk):
            v = (P[K] + P[K - 1]) / (RHO3[K] + RHO3[K - 1]) * lg[K]
        else:
            x10, x21, x32 = lg[K + 1], lg[K], lg[K - 1]
            x20, x30, x31 = x21 + x10, x32 + x21 + x10, x32 + x21
            v = -(q[K + 1] * x21 ** 3 * (x31 + x32) / (x10 * x20 * x30) +
                  q[K] * x21 * (x21 * (x21 + 2. * (x10 - x31)) - 6. * x10 * x31) / (x10 * x31) +
                  q[K - 1] * x21 * (x21 * (x21 + 2. * (x32 - x20)) - 6. * x20 * x32) / (x20 * x32) +
                  q[K - 2] * x21 ** 3 * (x10 + x20) / (x30 * x31 * x32)) / 12.
        G[K - 1] = G[K] + v
    for f, v in (("P3", P), ("THETA", TH), ("P2", P2), ("H3", H3), ("THETA2", TH2), ("T2", T2), ("T3", T3),
                 ("RHO2", RHO2), ("RHO3", RHO3), ("EXNER3", c.cp * T3 / np.where(TH == 0., 1., TH)), ("GZ3", G),
                 ("MONT3", G + c.cpr * T3 * c.rgas)):
        out[f][:nk + 1, rows] = v
    out["HDRY"][1:nk + 1, rows] = np.maximum(hmin[1:nk + 1, None, None], H[1:])
    for f in ("PV3", "DIV_UV3", "W3", "RI2"):
        out[f] = None
    if c.planet_type == b"gas-giant":
        out["GZ3"] = out["MONT3"] = None
    return out
