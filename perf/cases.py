"""Timed cases of the split-step dipolar GPE solver.

Each case is one thing a user of the framework has it do, through the public
Python binding of the C ABI (dbecpy, dbecserve): runs of split steps with the
wave function fetched at the end, the observables of a check, the density
files of an output, the operators one by one, and a served set of requests.
`exact` restates each of them in plain torch FP64 (dense Crank-Nicolson
propagators and library FFTs) on the same inputs.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "dbec-gp-mpi-cuda_amd", "python"))

import dbecpy  # noqa: E402
import dbecserve  # noqa: E402

TRAP = (0.5, 1.0, 1.5)  # gamma, nu, lambda of the example inputs and the benchmark
PAR = 2.0               # OPTION = 2
LENGTHS = (16, 32, 48, 64, 80, 96, 128, 160, 192, 256, 320, 384, 512)
LARGEST = 256 * 256 * 384
DENSITIES = (dbecpy.DEN_XYZ, dbecpy.DEN_X, dbecpy.DEN_Y, dbecpy.DEN_Z, dbecpy.DEN_XY, dbecpy.DEN_XZ, dbecpy.DEN_YZ,
             dbecpy.CUT_XY0, dbecpy.CUT_X0Z, dbecpy.CUT_0YZ)


def _case(kind, n, h, dt, cutoff, mode, prec, **more):
    return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "hx": h[0], "hy": h[1], "hz": h[2], "dt": dt,
            "cutoff": cutoff, "mode": mode, "prec": prec, **more}


def listed():
    example = ((128, 96, 80), (0.2, 0.2, 0.2), 0.005, 10.0)  # the reference's example inputs
    bench = ((256, 256, 256), (0.1, 0.1, 0.1), 0.0005, 12.8)  # the benchmark's grid
    h192 = (16 / 192,) * 3                                    # the serving stream's largest grid
    cases = {
        # a small ground state (the 64^3 CPU configuration): launches and latency count
        "steps_imag_64_fp64": _case("steps", (64, 64, 64), (0.25,) * 3, 0.004, 8.0, "imag", "fp64", steps=100),
        # the example's NSTP phase: the couplings grow with every step; nz = 80
        "ramp_imag_128x96x80_fp64": _case("ramp", *example, "imag", "fp64", steps=100),
        # the example's real-time run: rms sizes printed after every step (OUTSTPT = 1)
        "dynamics_real_128x96x80_fp64": _case("dynamics", *example, "real", "fp64", steps=50),
        # the largest real-time grid of the serving stream, mixed precision
        "steps_real_192_mixed": _case("steps", (192, 192, 192), h192, 0.001, 8.0, "real", "mixed", steps=100),
        # the benchmark's ground state, FP64 and mixed, between two outputs
        "steps_imag_256_fp64": _case("steps", *bench, "imag", "fp64", steps=100),
        "steps_imag_256_mixed": _case("steps", *bench, "imag", "mixed", steps=200),
        # the real-time quench grid, between two outputs: the largest case
        "steps_real_256x256x384_fp64": _case("steps", (256, 256, 384), (0.1,) * 3, 0.0002, 12.8, "real", "fp64",
                                             steps=100),
        # one convergence check (OBSSTP) of the benchmark's ground state
        "observe_imag_256_fp64": _case("observe", *bench, "imag", "fp64"),
        # one line of the real-time observables, with the phase-gradient energy
        "observe_real_192_mixed": _case("observe", (192, 192, 192), h192, 0.001, 8.0, "real", "mixed"),
        # the ten density files of one output (NPASOUT, NRUNOUT)
        "density_imag_192_fp64": _case("density", (192, 192, 192), h192, 0.01, 8.0, "imag", "fp64", outstp=1),
        # the operators called one by one, as a program with its own step does
        "operators_real_80x96x160_mixed": _case("operators", (80, 96, 160), (0.2, 0.17, 0.1), 0.002, 8.0, "real",
                                                "mixed"),
        # a few requests of the serving stream's kinds and sizes at once
        "serve_48_to_96": {"kind": "serve", "requests": 16, "smallest": 48, "largest": 96, "steps": 300},
    }
    return [{"name": k, **v} for k, v in cases.items()]


def draw(rng):
    kind = rng.choice(["steps"] * 5 + ["ramp", "dynamics", "observe", "observe", "density", "operators", "operators"] +
                      ["serve"])
    if kind == "serve":
        small = rng.choice((32, 48, 64))
        return {"kind": kind, "requests": rng.randint(4, 20), "smallest": small,
                "largest": rng.choice([m for m in LENGTHS if small <= m <= 96]), "steps": 10 * rng.randint(6, 30)}
    goal = math.exp(rng.uniform(math.log(16 ** 3), math.log(LARGEST)))
    while True:
        n = tuple(rng.choice(LENGTHS) for _ in range(3))
        if goal / 1.5 <= n[0] * n[1] * n[2] <= min(1.5 * goal, LARGEST):
            break
    points = n[0] * n[1] * n[2]
    box = rng.uniform(12.0, 20.0)
    h = tuple(box / m for m in n)
    mode, prec = rng.choice(("imag", "real")), rng.choice(("fp64", "fp64", "mixed"))
    more = {}
    if kind in ("steps", "ramp"):
        more["steps"] = max(10, min(rng.randint(40, 100), int(1.5e9 / points)))
    elif kind == "dynamics":
        more["steps"] = max(5, min(rng.randint(10, 50), int(3e8 / points)))
        mode = "real"
    elif kind == "density":
        more["outstp"] = rng.randint(1, 4)
    return _case(kind, n, h, rng.uniform(0.0002, 0.004), 0.5 * box, mode, prec, **more)


# ---- inputs ------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _couplings(seed):
    """g, gd of a stable condensate (eps_dd < 0.85), par * G0 and par * GDD0."""
    r = np.random.RandomState(seed % (1 << 31))
    g0 = r.uniform(100.0, 340.0)
    return PAR * g0, PAR * g0 * r.uniform(0.05, 0.2)


def _axes(case):
    return [(torch.arange(n, dtype=torch.float64, device=_dev()) - n // 2) * h
            for n, h in ((case["nx"], case["hx"]), (case["ny"], case["hy"]), (case["nz"], case["hz"]))]


def _psi0(case, seed):
    """A Gaussian near the trap's, off centre and with a smooth ripple (real
    time: and a smooth phase), on the device in FP64."""
    r = np.random.RandomState((seed + 77) % (1 << 31))
    x, y, z = _axes(case)
    cut = [0.1 * case["n" + a] * case["h" + a] for a in "xyz"]
    w = [t * r.uniform(0.7, 1.2) for t in TRAP]
    s = [r.uniform(-0.1, 0.1) * c for c in cut]
    k = r.uniform(0.3, 1.0, 3) / np.asarray(cut)
    f = [torch.exp(-0.5 * wi * (a - si) ** 2) for wi, a, si in zip(w, (x, y, z), s)]
    psi = f[0][:, None, None] * f[1][None, :, None] * f[2][None, None, :]
    arg = (k[0] * x)[:, None, None] + (k[1] * y)[None, :, None] + (k[2] * z)[None, None, :]
    psi *= 1.0 + 0.2 * torch.sin(arg + r.uniform(0, 6))
    psi *= math.sqrt(1.0 / float((psi * psi).sum() * case["hx"] * case["hy"] * case["hz"]))
    if case["mode"] == "real":
        q = r.uniform(-0.5, 0.5, 3)
        arg = (q[0] * x)[:, None, None] + (q[1] * y)[None, :, None] + (q[2] * z)[None, None, :]
        psi = torch.polar(psi, arg + 0.1 * torch.sin(arg * 2.0))
    return psi


def _params(case):
    return dbecpy.make_params(case["nx"], case["ny"], case["nz"], case["hx"], case["hy"], case["hz"], case["dt"],
                              *TRAP, case["cutoff"], PAR)


def _requests(case, seed):
    """Ground states and real-time runs of cubic grids in both precisions, as
    the serving stream mixes them, with stable couplings."""
    r = np.random.RandomState((seed + 5) % (1 << 31))
    sizes = [m for m in LENGTHS if case["smallest"] <= m <= case["largest"] and m != 80]
    out = []
    for i in range(case["requests"]):
        n = sizes[i % len(sizes)]
        mode = dbecpy.REAL if i % 5 == 4 else dbecpy.IMAG
        prec = dbecpy.MIXED if i % 2 else dbecpy.FP64
        g0 = r.uniform(20.0, 60.0)
        out.append(dbecserve.make_request(i, n, mode, prec, g0, g0 * r.uniform(0.02, 0.2), tuple(r.uniform(0.5, 2.0, 3)),
                                          0.001 if mode == dbecpy.REAL else 0.004, case["steps"]))
    return out


_lib = None


def _library():
    global _lib
    if _lib is None:
        _lib = dbecpy.load(dbecpy.HIP_LIB)
    return _lib


def prepare(case, seed):
    if case["kind"] == "serve":
        return {"case": case, "server": dbecserve.Server(_library(), device=0, max_batch=16, check_every=50),
                "requests": _requests(case, seed)}
    mode = dbecpy.IMAG if case["mode"] == "imag" else dbecpy.REAL
    s = dbecpy.Solver(_library(), _params(case), mode, dbecpy.FP64 if case["prec"] == "fp64" else dbecpy.MIXED)
    psi = _psi0(case, seed).cpu().numpy()
    s.set_psi(psi)
    if mode == dbecpy.IMAG:
        s.calcnorm(rescale=True)
    g, gd = _couplings(seed)
    s.set_coupling(g, gd)
    return {"case": case, "solver": s, "psi": psi if case["kind"] == "operators" else None, "g": g, "gd": gd}


# ---- one pass ----------------------------------------------------------------
def _field(case, a):
    """A field the solver hands out, in the precision the solver holds it in."""
    t = torch.from_numpy(a)
    if case["prec"] == "mixed":
        t = t.to(torch.complex64 if t.is_complex() else torch.float32)
    return t


def _number(case, v):
    """The norm that a step or an operator chain ends with, in the solver's precision."""
    return np.array([v], dtype=np.float32 if case["prec"] == "mixed" else np.float64)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "serve":
        return _run_serve(state)
    s = state["solver"]
    if kind == "steps" or kind == "ramp":
        k = case["steps"]
        if kind == "ramp":
            s.set_coupling(0.0, 0.0)
            norm = s.step(k, state["g"] / k, state["gd"] / k)
        else:
            norm = s.step(k)
        psi = _field(case, s.get_psi())
        return {"psi": psi, "norm": _number(case, norm)} if case["mode"] == "imag" else {"psi": psi}
    if kind == "dynamics":
        rms = np.empty((case["steps"], 4))
        for i in range(case["steps"]):
            s.step(1, want_norm=False)
            rms[i] = s.calcrms()
        return {"rms": _field(case, rms), "psi": _field(case, s.get_psi())}
    if kind == "observe":
        norm = s.calcnorm()
        mu, en = s.calcmuen()
        out = {"norm": np.array([norm]), "muen": np.array([mu, en]), "rms": s.calcrms(),
               "centre": np.array([s.psi_center()])}
        if case["mode"] == "real":
            out["muen_phase"] = np.array(s.calcmuen_phase())
        return out
    if kind == "density":
        o = case["outstp"]
        return [s.density(d, o, o, o) for d in DENSITIES]
    s.set_psi(state["psi"])
    s.calcpsidd2()
    phi = s.get_psidd2()
    s.calcnu()
    s.calclux()
    s.calcluy()
    s.calcluz()
    norm = s.calcnorm(rescale=case["mode"] == "imag")
    return {"phi": _field(case, phi), "norm": _number(case, norm), "psi": _field(case, s.get_psi())}


def _run_serve(state):
    got = state["server"].run_all(state["requests"])
    out = {"steps": np.array([got[r.id]["steps"] for r in state["requests"]], dtype=np.int64)}
    for name, prec, dtype in (("fp64", dbecpy.FP64, np.float64), ("mixed", dbecpy.MIXED, np.float32)):
        out[name] = np.array([[got[r.id]["mu"], got[r.id]["en"], got[r.id]["norm"], *got[r.id]["rms"]]
                              for r in state["requests"] if r.prec == prec], dtype=dtype)
    return out


# ---- what a pass cannot do without -------------------------------------------
def work(case):
    if case["kind"] == "serve":
        bytes_, flops = 0.0, 0.0
        for r in _requests(case, 0):
            c = _served_case(r)
            w = work({**c, "kind": "steps", "steps": r.max_steps})
            bytes_, flops = bytes_ + w["bytes"], flops + w["flops"]
        return {"bytes": bytes_, "flops": flops}
    n = float(case["nx"] * case["ny"] * case["nz"])
    real = 8 if case["prec"] == "fp64" else 4
    psi = real * (2 if case["mode"] == "real" else 1)
    host = 16 if case["mode"] == "real" else 8
    fft = 2.5 * n * math.log2(n)  # one real transform
    sweeps = 3 * n * (36 if case["mode"] == "real" else 12)
    step = 2 * fft + n + sweeps + n * (60 if case["mode"] == "real" else 40)
    if case["kind"] in ("steps", "ramp"):
        return {"bytes": case["steps"] * 2 * n * psi + n * host, "flops": case["steps"] * step}
    if case["kind"] == "dynamics":
        return {"bytes": case["steps"] * 2 * n * psi + n * host, "flops": case["steps"] * (step + 8 * n)}
    if case["kind"] == "observe":
        return {"bytes": n * psi, "flops": 2 * fft + n * (60 if case["mode"] == "imag" else 120)}
    if case["kind"] == "density":
        return {"bytes": n * psi + 8 * n / case["outstp"] ** 3, "flops": 8 * n}
    return {"bytes": 2 * n * host + 8 * n + 5 * 2 * n * psi, "flops": step}


# ---- the same in plain FP64 ----------------------------------------------------
def _simpson(n, h):
    """Weights of the reference's Simpson rule with its even-n end correction."""
    w = np.zeros(n)
    for i in range(1, n - 1, 2):
        w[i - 1:i + 2] += (1.0, 4.0, 1.0)
    if n % 2 == 0:
        w[n - 3:] += (-0.25, 2.0, 1.25)
    return torch.from_numpy(w * h / 3.0).to(_dev())


def _propagator(n, h, dt, complex_):
    """The Crank-Nicolson sweep of one axis as a dense matrix: the reference's
    recurrences (zero ends) on the identity."""
    r = dt / (h * h) / (3.0 - PAR)
    a0, a0r, a = (1 + 1j * r, 1 - 1j * r, -0.5j * r) if complex_ else (1 + r, 1 - r, -0.5 * r)
    t = np.complex128 if complex_ else np.float64
    alpha, gamma = np.zeros(n - 1, t), np.zeros(n - 1, t)
    gamma[n - 2] = -1.0 / a0
    for i in range(n - 2, 0, -1):
        alpha[i - 1] = a * gamma[i]
        gamma[i - 1] = -1.0 / (a0 + a * alpha[i - 1])
    psi, beta, out = np.eye(n, dtype=t), np.zeros((n - 1, n), t), np.zeros((n, n), t)
    beta[n - 2] = psi[n - 1]
    for i in range(n - 2, 0, -1):
        c = -a * psi[i + 1] + a0r * psi[i] - a * psi[i - 1]
        beta[i - 1] = gamma[i] * (a * beta[i] - c)
    for i in range(1, n - 1):
        out[i] = alpha[i - 1] * out[i - 1] + beta[i - 1]
    return torch.from_numpy(out).to(_dev())


class _Plain:
    """The solver's operators on a dense FP64 psi."""

    def __init__(self, case, trap=TRAP):
        self.n = (case["nx"], case["ny"], case["nz"])
        self.h = (case["hx"], case["hy"], case["hz"])
        self.dt, self.complex = case["dt"], case["mode"] == "real"
        x, y, z = _axes(case)
        self.x2 = (x * x, y * y, z * z)
        self.w = [_simpson(n, h) for n, h in zip(self.n, self.h)]
        self.u = [_propagator(n, h, case["dt"], self.complex) for n, h in zip(self.n, self.h)]
        self.pot = 0.5 * PAR * (self._outer(*[t * t * q for t, q in zip(trap, self.x2)], add=True))
        k2 = []
        for n, h in zip(self.n, self.h):
            i = torch.arange(n, dtype=torch.float64, device=_dev())
            k2.append((torch.where(i <= n // 2, i, i - n) * (2.0 * dbecpy.PI_REF / (n * h))) ** 2)
        k2[2] = k2[2][: self.n[2] // 2 + 1]
        kk = self._outer(*k2, add=True)
        kr = torch.sqrt(kk) * case["cutoff"]
        dd = (4.0 * dbecpy.PI_REF * (3.0 * k2[2][None, None, :] / kk - 1.0) / 3.0) * (
            1.0 + 3.0 * torch.cos(kr) / kr ** 2 - 3.0 * torch.sin(kr) / kr ** 3)
        dd[0, 0, 0] = 0.0
        self.potdd = dd

    @staticmethod
    def _outer(a, b, c, add=False):
        a, b, c = a[:, None, None], b[None, :, None], c[None, None, :]
        return a + b + c if add else a * b * c

    @staticmethod
    def mod2(psi):
        return psi.real ** 2 + psi.imag ** 2 if psi.is_complex() else psi * psi

    def integral(self, f, *axes):
        """Simpson sums of f over the axes."""
        for a in sorted(axes, reverse=True):
            f = torch.tensordot(f, self.w[a], dims=([a], [0]))
        return f

    def norm(self, psi):
        return float(torch.sqrt(self.integral(self.mod2(psi), 0, 1, 2)))

    def phi(self, psi):
        """The dipolar potential over N, after the periodic face copies."""
        f = torch.fft.irfftn(self.potdd * torch.fft.rfftn(self.mod2(psi)), s=self.n)
        f[-1, :-1, :-1] = f[0, :-1, :-1]
        f[:-1, -1, :-1] = f[:-1, 0, :-1]
        f[:-1, :-1, -1] = f[:-1, :-1, 0]
        return f

    def nu(self, psi, phi, g, gd):
        v = self.dt * (self.pot + g * self.mod2(psi) + gd * phi)
        return psi * (torch.polar(torch.ones_like(v), -v) if self.complex else torch.exp(-v))

    def sweeps(self, psi):
        nx, ny, nz = self.n
        psi = (self.u[0] @ psi.reshape(nx, ny * nz)).reshape(nx, ny, nz)
        psi = torch.stack([self.u[1] @ psi[i] for i in range(nx)])
        return (psi.reshape(nx * ny, nz) @ self.u[2].T.contiguous()).reshape(nx, ny, nz)

    def step(self, psi, g, gd):
        """One split step: psi and, in imaginary time, its norm before rescaling."""
        psi = self.sweeps(self.nu(psi, self.phi(psi), g, gd))
        if self.complex:
            return psi, None
        norm = self.norm(psi)
        return psi / norm, norm

    def rms(self, psi):
        m = self.mod2(psi)
        r2 = []
        for a in range(3):
            q = [torch.ones_like(v) for v in self.x2]
            q[a] = self.x2[a]
            r2.append(float(self.integral(m * self._outer(*q), 0, 1, 2)))
        return np.sqrt([sum(r2), *r2])

    def _slope2(self, f):
        """Sum over the axes of the squared five-point derivatives, over 3 - par."""
        total = torch.zeros_like(f)
        for a in range(3):
            h, v = self.h[a], f.movedim(a, 0)
            d = torch.zeros_like(v)
            d[2:-2] = (v[:-4] - 8.0 * v[1:-3] + 8.0 * v[3:-1] - v[4:]) / (12.0 * h)
            d[1] = (v[2] - v[0]) / (2.0 * h)
            d[-2] = (v[-1] - v[-3]) / (2.0 * h)
            total += (d * d).movedim(0, a) / (3.0 - PAR)
        return total

    def muen(self, psi, g, gd, phase=False):
        m, phi = self.mod2(psi), self.phi(psi)
        if phase:
            d = self._slope2(psi.real.contiguous()) + self._slope2(psi.imag.contiguous())
        else:
            d = self._slope2(psi.abs() if self.complex else psi)
        mu = (self.pot + g * m + gd * phi) * m + d
        en = (self.pot + 0.5 * g * m + 0.5 * gd * phi) * m + d
        return float(self.integral(mu, 0, 1, 2)), float(self.integral(en, 0, 1, 2))


def _served_case(r):
    return _case("steps", (r.nx, r.ny, r.nz), (r.dx, r.dy, r.dz), r.dt, r.cutoff,
                 "imag" if r.mode == dbecpy.IMAG else "real", "fp64" if r.prec == dbecpy.FP64 else "mixed")


def _held(case, psi):
    """psi as the solver stores it, in FP64."""
    if case["prec"] == "mixed":
        return psi.to(torch.complex64 if psi.is_complex() else torch.float32).to(psi.dtype)
    return psi


def exact(case, seed):
    if case["kind"] == "serve":
        return _exact_serve(case, seed)
    p, kind = _Plain(case), case["kind"]
    psi = _held(case, _psi0(case, seed))
    if case["mode"] == "imag":
        psi = _held(case, psi / p.norm(psi))
    g, gd = _couplings(seed)
    if kind in ("steps", "ramp"):
        norm = None
        for i in range(case["steps"]):
            f = (i + 1) / case["steps"] if kind == "ramp" else 1.0
            psi, norm = p.step(psi, g * f, gd * f)
        return {"psi": psi, "norm": np.array([norm])} if case["mode"] == "imag" else {"psi": psi}
    if kind == "dynamics":
        rms = []
        for _ in range(case["steps"]):
            psi, _n = p.step(psi, g, gd)
            rms.append(p.rms(psi))
        return {"rms": np.array(rms), "psi": psi}
    if kind == "observe":
        c = complex(psi[case["nx"] // 2, case["ny"] // 2, case["nz"] // 2])
        out = {"norm": np.array([p.norm(psi)]), "muen": np.array(p.muen(psi, g, gd)), "rms": p.rms(psi),
               "centre": np.array([c])}
        if case["mode"] == "real":
            out["muen_phase"] = np.array(p.muen(psi, g, gd, phase=True))
        return out
    m = p.mod2(psi)
    if kind == "density":
        o = case["outstp"]
        cut = [n // 2 for n in p.n]
        full = [m, p.integral(m, 1, 2), p.integral(m, 0, 2), p.integral(m, 0, 1), p.integral(m, 2), p.integral(m, 1),
                p.integral(m, 0), m[:, :, cut[2]], m[:, cut[1], :], m[cut[0]]]
        return [f[(slice(None, None, o),) * f.dim()].reshape(-1).contiguous() for f in full]
    psi = _held(case, _psi0(case, seed))
    phi = p.phi(psi)
    psi = p.sweeps(p.nu(psi, phi, g, gd))
    norm = p.norm(psi)
    if case["mode"] == "imag":
        psi = psi / norm
    return {"phi": phi * float(p.n[0] * p.n[1] * p.n[2]), "norm": np.array([norm]), "psi": psi}


def _exact_serve(case, seed):
    rows = {dbecpy.FP64: [], dbecpy.MIXED: []}
    for r in _requests(case, seed):
        c = _served_case(r)
        trap = (r.vgamma, r.vnu, r.vlambda)
        p = _Plain(c, trap)
        psi = p._outer(*[torch.exp(-0.5 * t * q) for t, q in zip(trap, p.x2)])
        psi = psi / math.sqrt(dbecpy.PI_REF * math.sqrt(dbecpy.PI_REF / (trap[0] * trap[1] * trap[2])))
        if r.mode == dbecpy.IMAG:
            psi = psi / p.norm(psi)
        else:
            psi = psi.to(torch.complex128)
        for _ in range(r.max_steps):
            psi, norm = p.step(psi, r.g, r.gd)
        mu, en = p.muen(psi, r.g, r.gd)
        rows[r.prec].append([mu, en, norm if norm is not None else p.norm(psi), *p.rms(psi)])
    return {"steps": None, "fp64": np.array(rows[dbecpy.FP64]), "mixed": np.array(rows[dbecpy.MIXED])}
