"""Performance cases of the MHD framework: the work its users run, through the public entry points.

Grids follow the sizes of this repository's tests and benchmark (16^3 to 512^3, cubes and boxes,
multiples of the launch tiles and not). Every case starts from a smooth random state of all eight
fields (a few Fourier modes each, as in decaying-turbulence runs) with the benchmark's physics.

Paths:
  cfl        acDeviceIntegrateStepsCFL: time stepping with the CFL timestep kept on the device
  substeps   the reference API's own loop: periodic fill, substep, swap, at a fixed timestep
  monitor    diagnostics and reductions of a state, as a run's time-series output takes them
  gradient   MHDSolve forward and backward: dL/df0, dL/dnu, dL/deta of the final kinetic energy
"""
import ctypes
import math

import numpy as np
import torch

from astaroth_amd import adjoint as AD
from astaroth_amd import astaroth as ac

NF = ac.NUM_VTXBUF_HANDLES
R = 3
COURANT = 0.2
PARAMS = dict(AC_cs_sound=1.0, AC_gamma=5.0 / 3.0, AC_nu_visc=5e-3, AC_eta=5e-3, AC_chi=5e-3,
              AC_K_heatcond=5e-3)
# amplitude of the modes of lnrho, u, A and ss
AMPLITUDE = (0.02, 0.05, 0.05, 0.05, 0.05, 0.05, 0.05, 0.02)
MODES = 4


def _case(name, path, precision, n, steps=1, kahan=0, upwind=True, entropy=True, forcing=False,
          timestep="courant"):
    c = {"path": path, "precision": precision, "nx": n[0], "ny": n[1], "nz": n[2], "steps": steps,
         "kahan": kahan, "upwind": upwind, "entropy": entropy, "forcing": forcing,
         "timestep": timestep}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one step of a small run between host decisions: launch latency dominates
        _case("cfl_32_fp32", "cfl", "fp32", (32, 32, 32)),
        # an interactive run in the reference's own call pattern
        _case("substeps_64_fp32", "substeps", "fp32", (64, 64, 64), steps=2),
        # a small double-precision run on a box no tile divides (verification runs)
        _case("substeps_100x90x75_fp64", "substeps", "fp64", (100, 90, 75)),
        # the headline: many steps at 256^3
        _case("cfl_256_fp32", "cfl", "fp32", (256, 256, 256), steps=4),
        # the same in the precise (32-bit compensated) mode
        _case("cfl_256_fp32_precise", "cfl", "fp32", (256, 256, 256), steps=2, kahan=32),
        # the reference's default precision
        _case("cfl_256_fp64", "cfl", "fp64", (256, 256, 256)),
        # a production box whose sides are round numbers but not multiples of a tile
        _case("cfl_200x150x100_fp32", "cfl", "fp32", (200, 150, 100), steps=2),
        # driven turbulence with the reference's timestep (Alfven speed included), isothermal
        _case("forced_128_fp32", "cfl", "fp32", (128, 128, 128), steps=2, entropy=False,
              forcing=True, timestep="reference"),
        # what the time series of a 256^3 run costs at each output
        _case("monitor_256_fp32", "monitor", "fp32", (256, 256, 256)),
        # gradients for initial conditions and diffusivities (optimisation, data assimilation)
        _case("gradient_128_fp32", "gradient", "fp32", (128, 128, 128), steps=3),
        # gradient checking in double precision on a small odd box
        _case("gradient_72x60x50_fp64", "gradient", "fp64", (72, 60, 50), steps=2),
        # the largest: a long-run production grid with 16-bit compensation
        _case("cfl_512_fp32_k16", "cfl", "fp32", (512, 512, 512), kahan=16),
    ]


def draw(rng):
    path = rng.choices(("cfl", "substeps", "monitor", "gradient"), (4, 3, 1, 2))[0]
    precision = rng.choices(("fp32", "fp64"), (2, 1))[0]
    top = {"cfl": 288, "substeps": 288, "monitor": 320, "gradient": 144}[path]
    if precision == "fp64":
        top = top * 3 // 4

    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    n = [side(16, top)] * 3
    if rng.random() < 0.5:  # a box
        n = [min(top, max(16, int(round(n[0] * rng.uniform(0.6, 1.5))))) for _ in range(3)]
    if rng.random() < 0.5:  # sides in round numbers, as configurations have them
        n = [max(16, v // 16 * 16) for v in n]
    kahan = 0
    if precision == "fp32" and path in ("cfl", "substeps"):
        kahan = rng.choices((0, 8, 16, 32), (5, 1, 1, 1))[0]
    steps = 1 if path == "monitor" else rng.choice((1, 2, 3))
    timestep = rng.choice(("courant", "courant", "reference", "additive")) if path == "cfl" else "courant"
    return _case("", path, precision, tuple(n), steps=steps, kahan=kahan,
                 upwind=rng.random() < 0.8, entropy=rng.random() < 0.8,
                 forcing=path == "cfl" and rng.random() < 0.25, timestep=timestep)


# ------------------------------------------------------------------ inputs
def _fields(case, seed):
    """The initial state (NF, mz, my, mx) in the case's precision, halos periodic."""
    rng = np.random.RandomState(seed % (1 << 31))
    dt = torch.float32 if case["precision"] == "fp32" else torch.float64
    n = (case["nx"], case["ny"], case["nz"])
    ax = [torch.remainder(torch.arange(-R, m + R, device="cuda"), m).double() * (2 * math.pi / m)
          for m in n]
    f = torch.empty((NF, n[2] + 2 * R, n[1] + 2 * R, n[0] + 2 * R), dtype=dt, device="cuda")
    for q in range(NF):
        acc = 0.0
        for _ in range(MODES):
            k = rng.randint(-3, 4, 3)
            a, ph = rng.uniform(0.4, 1.0) * AMPLITUDE[q], rng.uniform(0, 2 * math.pi)
            xy = torch.polar(torch.ones_like(ax[0]), ax[0] * int(k[0]) + ph)[None, :] * \
                torch.polar(torch.ones_like(ax[1]), ax[1] * int(k[1]))[:, None]
            z = torch.polar(torch.full_like(ax[2], a), ax[2] * int(k[2]))[:, None, None]
            acc = acc + (z.real * xy.real - z.imag * xy.imag)
        f[q] = acc
        del acc
    return f


def _real(case, v):
    return float(np.float32(v)) if case["precision"] == "fp32" else float(v)


def _forcing(case, seed):
    """One helical forcing mode, as the driver loads before a step."""
    rng = np.random.RandomState((seed + 77) % (1 << 31))
    k = [float(v) for v in rng.randint(1, 4, 3)]
    vec = lambda: [_real(case, v) for v in rng.uniform(-0.6, 0.6, 3)]  # noqa: E731
    return {"k": k, "re": vec(), "im": vec(), "phase": _real(case, rng.uniform(-3, 3)),
            "magnitude": _real(case, 0.05), "kaver": _real(case, 2.5)}


def _fixed_dt(case):
    return _real(case, COURANT * 2 * math.pi / max(case["nx"], case["ny"], case["nz"]) / 1.3)


class _Field:
    """One slab of device memory as torch sees it; it holds its device."""

    def __init__(self, dev, ptr, shape, typestr):
        self.dev = dev
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False),
                                         "version": 3, "strides": None}


def _state(s):
    """The device's current state, interior cells, without a copy."""
    ptr = s["dev"].field_ptrs(0)[0]
    if ptr not in s["views"]:
        t = torch.as_tensor(_Field(s["dev"], ptr, s["shape"], s["typestr"]), device="cuda")
        s["views"][ptr] = t[:, R:-R, R:-R, R:-R]
    return s["views"][ptr]


def _load(s):
    ac.check(s["lib"].acDeviceLoadMeshFromDevicePtr(s["dev"].handle, ac.STREAM_DEFAULT,
                                                    s["f0"].data_ptr()), "load")


def _cfl(s):
    ac.check(s["lib"].acDeviceIntegrateStepsCFL(s["dev"].handle, ac.STREAM_DEFAULT,
                                                s["case"]["steps"], COURANT, None), "steps")


def prepare(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    lib = ac.load(case["precision"])
    info = lib.config(n, AC_len=(2 * math.pi,) * 3, AC_lupwd=case["upwind"],
                      AC_lentropy=case["entropy"], AC_lforcing=case["forcing"],
                      AC_switch_forcing=-1.0, AC_additive_timestep=case["timestep"] == "additive",
                      AC_kahan_bits=case["kahan"], **PARAMS)
    f0 = _fields(case, seed)
    s = {"case": case, "lib": lib, "f0": f0, "views": {}, "shape": tuple(f0.shape),
         "typestr": "<f4" if case["precision"] == "fp32" else "<f8"}
    torch.cuda.synchronize()
    if case["path"] == "gradient":
        s["runner"] = AD.MHDAdjoint(lib, info, case["steps"], _fixed_dt(case), snaps=2)
        s["dev"] = s["runner"].dev
        s["f0"] = f0.requires_grad_(True)
        s["nu"] = torch.tensor(PARAMS["AC_nu_visc"], dtype=torch.float64, requires_grad=True)
        s["eta"] = torch.tensor(PARAMS["AC_eta"], dtype=torch.float64, requires_grad=True)
        s["runner"].advance(1)  # the launch autotuner's trials
        s["runner"]._sync()
        return s
    dev = s["dev"] = ac.Device(lib, info)
    if case["path"] == "monitor":
        _load(s)
        dev.periodic()
        dev.sync()
        return s
    s["dt"] = lib.np_real(_fixed_dt(case))
    if case["forcing"]:
        p = _forcing(case, seed)
        fp = lib.ForcingParams(p["magnitude"], lib.Real3(*p["k"]), lib.Real3(*p["re"]),
                               lib.Real3(*p["im"]), p["phase"], p["kaver"])
        ac.check(lib.acDeviceLoadForcingParams(dev.handle, ac.STREAM_DEFAULT, fp), "forcing")
    if case["timestep"] != "courant":
        ac.check(lib.acDeviceSetTimestepMode(dev.handle, 1), "mode")
    _load(s)
    dev.step(s["dt"])  # the launch autotuner's trials
    _load(s)
    dev.periodic()
    ac.check(lib.acDeviceUpdateTimestepCFL(dev.handle, ac.STREAM_DEFAULT, COURANT), "cfl")
    dev.sync()
    return s


def run(s):
    case, dev = s["case"], s["dev"]
    if case["path"] == "cfl":
        _cfl(s)
        return _state(s)
    if case["path"] == "substeps":
        for _ in range(case["steps"]):
            dev.step(s["dt"])
        return _state(s)
    if case["path"] == "monitor":
        d = dev.diagnostics()
        out = {k: np.array(getattr(d, k)) for k in ("min", "max", "rms")}
        out.update({k: getattr(d, k) for k in ("uu_rms", "uu_max", "bb_rms", "bb_max", "va_rms", "va_max")})
        out["lnrho_min"] = dev.reduce_scal("RTYPE_MIN", 0)
        out["ss_rms"] = dev.reduce_scal("RTYPE_RMS", 7)
        out["u_max"] = dev.reduce_vec("RTYPE_MAX", 1, 2, 3)
        out["u_rms"] = dev.reduce_vec("RTYPE_RMS", 1, 2, 3)
        return out
    out = AD.MHDSolve.apply(s["f0"], s["nu"], s["eta"], s["runner"])
    u = out[1:4, R:-R, R:-R, R:-R]
    loss = 0.5 * (u * u).sum()
    g, gnu, geta = torch.autograd.grad(loss, (s["f0"], s["nu"], s["eta"]))
    return {"state": out.detach(), "f0": g, "nu_eta": torch.stack((gnu, geta))}


def work(case):
    cells = case["nx"] * case["ny"] * case["nz"]
    size = 4 if case["precision"] == "fp32" else 8
    if case["path"] == "monitor":  # the fields once for the diagnostics, then 1 + 1 + 3 + 3 of them
        return {"bytes": float(cells * size * (NF + 8)), "flops": float(cells * 150)}
    # one step: ten touches of each field (f, w read and written; w unread at the first substep
    # and unwritten at the last), compensation read and written per substep
    step = cells * NF * (10 * size + 6 * case["kahan"] // 8)
    flops = cells * 3 * (760 + (100 if case["upwind"] else 0) + (120 if case["entropy"] else 0))
    if case["path"] == "gradient":
        # forward, recomputation of each step once, and per adjoint substep the state read and
        # lambda_f, lambda_w read and written; the adjoint does about twice the forward's work
        return {"bytes": float(case["steps"] * (2 * step + 3 * cells * NF * 5 * size)),
                "flops": float(case["steps"] * 4 * flops)}
    return {"bytes": float(case["steps"] * step), "flops": float(case["steps"] * flops)}


# ------------------------------------------------------------------ exact values (64 bits)
_D1 = (3.0 / 4.0, -3.0 / 20.0, 1.0 / 60.0)
_D2 = (-49.0 / 18.0, 3.0 / 2.0, -3.0 / 20.0, 1.0 / 90.0)
_UP = (-20.0 / 60.0, 15.0 / 60.0, -6.0 / 60.0, 1.0 / 60.0)
_MX = (270.0 / 720.0, -27.0 / 720.0, 2.0 / 720.0)
_ALPHA = (0.0, -5.0 / 9.0, -153.0 / 128.0)
_BETA = (1.0 / 3.0, 15.0 / 16.0, 8.0 / 15.0)


def _sh(f, ax, o):
    """f at offset o along axis ax (0 = x) of a periodic (z, y, x) array."""
    return torch.roll(f, -o, 2 - ax)


def _d1(f, ax, h):
    return sum(c * (_sh(f, ax, o) - _sh(f, ax, -o)) for o, c in enumerate(_D1, 1)) / h


def _sym(f, ax, c):
    return sum(c[o] * ((_sh(f, ax, o) - f) + (_sh(f, ax, -o) - f)) for o in (1, 2, 3))


def _mixed(f, a, b, ds):
    r = 0.0
    for o, c in enumerate(_MX, 1):
        p, m = _sh(f, a, o), _sh(f, a, -o)
        r = r + c * ((_sh(p, b, o) - _sh(p, b, -o)) - (_sh(m, b, o) - _sh(m, b, -o)))
    return r / (ds[a] * ds[b])


def _curl(A, ds):
    return [_d1(A[2], 1, ds[1]) - _d1(A[1], 2, ds[2]), _d1(A[0], 2, ds[2]) - _d1(A[2], 0, ds[0]),
            _d1(A[1], 0, ds[0]) - _d1(A[0], 1, ds[1])]


def _rhs(case, f, P, nu, eta, ds):
    """The right-hand side of the eight fields (lnrho, u, A, ss) of a periodic state."""
    lr, u, A, ss = f[0], f[1:4], f[4:7], f[7]
    g = lambda q: [_d1(q, a, ds[a]) for a in range(3)]  # noqa: E731
    d2 = lambda q, a: _sym(q, a, _D2) / ds[a] ** 2  # noqa: E731
    lap = lambda q: sum(d2(q, a) for a in range(3))  # noqa: E731

    def grad_div(v):
        return [sum(d2(v[b], b) if a == b else _mixed(v[b], a, b, ds) for b in range(3))
                for a in range(3)]

    def upwind(q):
        return sum(u[a].abs() * _sym(q, a, _UP) / ds[a] for a in range(3))

    glr, gu = g(lr), [g(v) for v in u]
    divu = gu[0][0] + gu[1][1] + gu[2][2]
    S = [[0.5 * (gu[i][j] + gu[j][i]) - (divu / 3.0 if i == j else 0.0) for j in range(3)]
         for i in range(3)]
    cont = -sum(u[a] * glr[a] for a in range(3)) - divu
    if case["upwind"]:
        cont = cont + upwind(lr)
    B = _curl(A, ds)
    lapA = [lap(v) for v in A]
    j = [(gd - la) / P["mu0"] for gd, la in zip(grad_div(A), lapA)]
    inv_rho = torch.exp(-lr)
    gs = g(ss) if case["entropy"] else None
    cs2 = P["cs2"]
    if case["entropy"]:
        lnT = P["gamma"] * ss / P["cp"] + (P["gamma"] - 1.0) * (lr - P["lnrho0"])
        cs2 = cs2 * torch.exp(lnT)
    jxB = [j[1] * B[2] - j[2] * B[1], j[2] * B[0] - j[0] * B[2], j[0] * B[1] - j[1] * B[0]]
    gdu = grad_div(u)
    out = [cont]
    for i in range(3):
        m = -sum(gu[i][a] * u[a] for a in range(3)) + inv_rho * jxB[i]
        m = m - cs2 * (glr[i] + (gs[i] / P["cp"] if case["entropy"] else 0.0))
        m = m + nu * (lap(u[i]) + gdu[i] / 3.0 + 2.0 * sum(S[i][a] * glr[a] for a in range(3)))
        m = m + P["zeta"] * gdu[i]
        out.append(m + upwind(u[i]) if case["upwind"] else m)
    del gdu, jxB
    uxB = [u[1] * B[2] - u[2] * B[1], u[2] * B[0] - u[0] * B[2], u[0] * B[1] - u[1] * B[0]]
    out += [x + eta * la for x, la in zip(uxB, lapA)]
    if not case["entropy"]:
        return out
    rho = torch.exp(lr)
    heat = eta * P["mu0"] * sum(x * x for x in j) + P["zeta"] * rho * divu * divu + \
        2.0 * rho * nu * sum(S[a][b] * S[a][b] for a in range(3) for b in range(3))
    first = P["gamma"] / P["cp"] * lap(ss) + (P["gamma"] - 1.0) * lap(lr)
    for a in range(3):
        lt = P["gamma"] / P["cp"] * gs[a] + (P["gamma"] - 1.0) * glr[a]
        first = first + lt * (P["gamma"] * (gs[a] / P["cp"] + glr[a]) - glr[a])
    st = -sum(u[a] * gs[a] for a in range(3)) + torch.exp(-(lr + lnT + P["lnT0"])) * heat
    return out + [st + P["K"] * inv_rho * first]


def _substep(case, f, w, s, dt, P, nu, eta, ds):
    r = _rhs(case, f, P, nu, eta, ds)
    nw = [dt * x if s == 0 else _ALPHA[s] * y + dt * x for x, y in zip(r, w)]
    del r
    nf = [x + _BETA[s] * y for x, y in zip(f, nw)]
    return (nf if case["entropy"] else nf + [f[7]]), nw


def _timestep(case, f, P, ds):
    h = min(ds)
    u2 = f[1] * f[1] + f[2] * f[2] + f[3] * f[3]
    if case["timestep"] == "courant":
        return COURANT * h / (1.0 + float(u2.max()) ** 0.5)
    va2 = sum(b * b for b in _curl(f[4:7], ds)) / torch.exp(f[0])
    visc = max(PARAMS["AC_nu_visc"], PARAMS["AC_eta"])
    if case["timestep"] == "additive":
        adv = 0.4 * h / float((u2.sqrt() + (P["cs2"] + va2).sqrt()).max())
        visc = max(visc, PARAMS["AC_gamma"] * PARAMS["AC_chi"])
    else:
        adv = 0.4 * h / (float(u2.max()) ** 0.5 + (P["cs2"] + float(va2.max())) ** 0.5)
    return min(adv, 0.3 * h * h / visc)


def _force(case, seed, f, dt):
    p = _forcing(case, seed)
    ax = [torch.arange(m, device="cuda").double() * (2 * math.pi * k / m)
          for m, k in zip((case["nx"], case["ny"], case["nz"]), p["k"])]
    ky = ax[0][None, None, :] + ax[1][None, :, None] + ax[2][:, None, None] + p["phase"]
    amp = math.sqrt(dt) * p["magnitude"] * math.sqrt(p["kaver"])
    for d in range(3):
        f[1 + d] = f[1 + d] + amp * (p["re"][d] * torch.cos(ky) - p["im"][d] * torch.sin(ky))


def _exact_gradient(case, f, P, ds, dt):
    """State after the steps and the gradients of its kinetic energy, substep by substep."""
    nu, eta = PARAMS["AC_nu_visc"], PARAMS["AC_eta"]
    states, ws, w = [], [], [torch.zeros_like(x) for x in f[:8]]
    for s in range(3 * case["steps"]):
        states.append(f)
        ws.append(w)
        with torch.no_grad():
            f, w = _substep(case, f, w, s % 3, dt, P, nu, eta, ds)
    lf = [x if q in (1, 2, 3) else torch.zeros_like(x) for q, x in enumerate(f)]
    lw, gp = [torch.zeros_like(x) for x in w], [0.0, 0.0]
    for s in reversed(range(3 * case["steps"])):
        x = [t.detach().requires_grad_(True) for t in states.pop()]
        y = [t.detach().requires_grad_(True) for t in ws.pop()[:len(lw)]]
        p = [torch.tensor(v, dtype=torch.float64, device="cuda", requires_grad=True) for v in (nu, eta)]
        nf, nw = _substep(case, x, y, s % 3, dt, P, p[0], p[1], ds)
        g = torch.autograd.grad(nf + nw, x + y + p, lf + lw, allow_unused=True)
        g = [torch.zeros_like(v) if t is None else t for t, v in zip(g, x + y + p)]
        lf, lw = list(g[:NF]), list(g[NF:-2])
        gp = [gp[0] + float(g[-2]), gp[1] + float(g[-1])]
        del nf, nw, g
    grad = torch.zeros((NF,) + tuple(n + 2 * R for n in f[0].shape), dtype=torch.float64, device="cuda")
    grad[:, R:-R, R:-R, R:-R] = torch.stack(lf)
    state = torch.stack(f)
    for d in (1, 2, 3):
        n = state.shape[d]
        state = state.index_select(d, torch.remainder(torch.arange(-R, n + R, device="cuda"), n))
    return {"state": state, "f0": grad, "nu_eta": torch.tensor(gp, dtype=torch.float64)}


def exact(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    ds = [2 * math.pi / m for m in n]
    P = {"cs2": 1.0, "gamma": _real(case, PARAMS["AC_gamma"]), "cp": 1.0, "mu0": _real(case, 1.4),
         "zeta": _real(case, 0.01), "lnT0": _real(case, 1.2), "lnrho0": _real(case, 1.3),
         "K": PARAMS["AC_K_heatcond"]}
    f = [x[R:-R, R:-R, R:-R].double() for x in _fields(case, seed)]
    if case["path"] == "monitor":
        B2 = sum(b * b for b in _curl(f[4:7], ds))
        u2 = f[1] * f[1] + f[2] * f[2] + f[3] * f[3]
        va2 = B2 / torch.exp(f[0])
        rms = lambda sq: float(sq.mean()) ** 0.5  # noqa: E731
        out = {"min": np.array([float(x.min()) for x in f]), "max": np.array([float(x.max()) for x in f]),
               "rms": np.array([rms(x * x) for x in f])}
        for k, v in (("uu", u2), ("bb", B2), ("va", va2)):
            out[k + "_rms"], out[k + "_max"] = rms(v), float(v.max()) ** 0.5
        out.update(lnrho_min=float(f[0].min()), ss_rms=rms(f[7] * f[7]), u_max=float(u2.max()) ** 0.5,
                   u_rms=rms(u2))
        return out
    if case["path"] == "gradient":
        return _exact_gradient(case, f, P, ds, _fixed_dt(case))
    nu, eta = PARAMS["AC_nu_visc"], PARAMS["AC_eta"]
    dt = _fixed_dt(case) if case["path"] == "substeps" else _timestep(case, f, P, ds)
    w = [None] * NF
    for _ in range(case["steps"]):
        nxt = dt
        for s in range(3):
            if s == 2 and case["path"] == "cfl" and case["timestep"] != "courant":
                nxt = _timestep(case, f, P, ds)
            f, w = _substep(case, f, w, s, dt, P, nu, eta, ds)
        if case["forcing"]:
            _force(case, seed, f, dt)
        if case["path"] == "cfl":
            dt = _timestep(case, f, P, ds) if case["timestep"] == "courant" else nxt
    return torch.stack(f)
