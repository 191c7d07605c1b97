"""What a user of this framework has it do, as timed cases.

Solves of the driven-dissipative NLS equation through the public entry
points, over their real range: host models (Problem().model(...).solve(), the
reference's own API), device solves (native.advance) of lines and grids in
both precisions and every order, parameter sweeps (Batch, sweep.solve_models)
and the split-step Fourier scheme.  A pass starts from the initial fields, as
a program with a new initial state does, and returns the whole final state.

kind of a case:
  advance  one line or grid on device buffers (native.advance)
  model    one host solve, the reference's mode: single precision, 1-D radial
           or 2-D zero-outside boundaries, algebraic reservoir
  batch    many grids of mixed sizes on the device (Batch.advance)
  sweep    the reference worker's job list, one model per pumping power
           (sweep.solve_models), host arrays in and out
"""
import math

import numpy as np
import torch

from nls_amd import native
from nls_amd.batch import Batch
from nls_amd.model import Problem
from nls_amd.sweep import solve_models

REAL = {"f32": np.float32, "f64": np.float64}
COMPLEX = {"f32": np.complex64, "f64": np.complex128}


def listed():
    return [
        # the smallest standard workload: a periodic line of 256 points, in
        # full (2000 steps); latency of one workgroup's step
        {"name": "line256_f32", "kind": "advance", "dim": 1, "n": 256, "order": 5, "bc": "periodic", "dtype": "f32",
         "dynamic": True, "scheme": "rk4", "steps": 2000, "dx": 20.0 / 256, "dt": 1e-3},
        # the reference's default 1-D model (1000 nodes, order 5, radial
        # grid), a host solve of 2000 iterations
        {"name": "radial1000_model", "kind": "model", "dim": 1, "n": 1000, "order": 5, "steps": 2000, "dx": 0.1,
         "dt": 1e-3},
        # the longest line the request loop serves, double precision
        {"name": "line4096_f64", "kind": "advance", "dim": 1, "n": 4096, "order": 5, "bc": "periodic", "dtype": "f64",
         "dynamic": True, "scheme": "rk4", "steps": 1000, "dx": 20.0 / 1024, "dt": 5e-5},
        # the reference's default 2-D model (40 x 40 nodes, order 3, 1000
        # iterations): the smallest host solve
        {"name": "model2d_40", "kind": "model", "dim": 2, "n": 40, "order": 3, "steps": 1000, "dx": 0.1, "dt": 1e-3},
        # the reference worker's job (200 x 200 nodes, order 5) for sixteen
        # pumping powers, host arrays in and out
        {"name": "worker200_x16", "kind": "sweep", "n": 200, "order": 5, "count": 16, "steps": 1000, "dx": 0.2,
         "dt": 2e-3},
        # one 256 x 256 grid: a device that is mostly idle, latency of a step
        {"name": "square256_f32", "kind": "advance", "dim": 2, "n": 256, "order": 5, "bc": "periodic", "dtype": "f32",
         "dynamic": True, "scheme": "rk4", "steps": 1000, "dx": 32.0 / 256, "dt": 5e-4},
        # an odd size, the widest stencil, double precision, zero outside,
        # algebraic reservoir; too few steps for a replayed block
        {"name": "grid777_f64_o7_ref", "kind": "advance", "dim": 2, "n": 777, "order": 7, "bc": "ref", "dtype": "f64",
         "dynamic": False, "scheme": "rk4", "steps": 100, "dx": 0.125, "dt": 8e-4},
        # the large grid in double precision
        {"name": "square2048_f64", "kind": "advance", "dim": 2, "n": 2048, "order": 5, "bc": "periodic",
         "dtype": "f64", "dynamic": True, "scheme": "rk4", "steps": 200, "dx": 0.0625, "dt": 2.5e-4},
        # and in single precision
        {"name": "square2048_f32", "kind": "advance", "dim": 2, "n": 2048, "order": 5, "bc": "periodic",
         "dtype": "f32", "dynamic": True, "scheme": "rk4", "steps": 300, "dx": 0.0625, "dt": 2.5e-4},
        # the benchmark's parameter sweep: 512 grids of 64, 128 and 256 points
        # a side in one batch (a tenth of its 5000 steps)
        {"name": "sweep512_f32", "kind": "batch", "order": 5, "bc": "periodic", "dtype": "f32", "dynamic": True,
         "sides": "64*256 128*154 256*102", "length": 32.0, "steps": 500, "dt": 5e-4},
        # split-step Fourier on the large grid, double precision
        {"name": "ssf2048_f64", "kind": "advance", "dim": 2, "n": 2048, "order": 5, "bc": "periodic", "dtype": "f64",
         "dynamic": True, "scheme": "ssf", "steps": 60, "dx": 0.0625, "dt": 2.5e-4},
        # and on a middle-sized one in single precision
        {"name": "ssf512_f32", "kind": "advance", "dim": 2, "n": 512, "order": 5, "bc": "periodic", "dtype": "f32",
         "dynamic": True, "scheme": "ssf", "steps": 200, "dx": 0.125, "dt": 5e-4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: lines of 64 to 8192 points, grids of
    24 to 2048 points a side, host models up to 4000 / 400 nodes, batches of 8
    to 256 grids, split-step sizes (powers of two)."""
    kind = rng.choice(["line", "grid", "grid", "model1d", "model2d", "batch", "batch", "sweep", "ssf"])
    order = rng.choice([3, 5, 5, 5, 7])
    dtype = rng.choice(["f32", "f32", "f64"])
    bc = rng.choice(["periodic", "periodic", "ref"])
    dyn = rng.random() < (0.75 if bc == "periodic" else 0.35)
    dx = round(rng.uniform(0.05, 0.25), 4)
    dt = float("%.3g" % (rng.uniform(0.04, 0.12) * dx * dx))
    base = {"order": order, "bc": bc, "dtype": dtype, "dynamic": dyn, "scheme": "rk4", "dx": dx, "dt": dt}
    if kind == "line":
        return dict(base, kind="advance", dim=1, n=_log(rng, 64, 8192), steps=_log(rng, 100, 2000))
    if kind == "grid":
        n = _log(rng, 24, 2048)
        return dict(base, kind="advance", dim=2, n=n, steps=max(20, min(1000, _log(rng, 50, 1000), int(8e8 / (n * n)))))
    if kind == "model1d":
        return {"kind": "model", "dim": 1, "n": _log(rng, 200, 4000), "order": order, "steps": _log(rng, 300, 2000),
                "dx": dx, "dt": dt}
    if kind == "model2d":
        return {"kind": "model", "dim": 2, "n": _log(rng, 20, 400), "order": order, "steps": _log(rng, 200, 1500),
                "dx": dx, "dt": dt}
    if kind == "sweep":
        return {"kind": "sweep", "n": _log(rng, 40, 300), "order": order, "count": rng.randint(3, 24),
                "steps": _log(rng, 200, 1000), "dx": dx, "dt": dt}
    if kind == "batch":
        groups = []
        for _ in range(rng.randint(1, 4)):
            side = _log(rng, 24, 320)
            groups.append("%d*%d" % (side, rng.randint(2, max(2, min(64, int(2.5e6 / (side * side)))))))
        length = 24 * dx * 8
        return {"kind": "batch", "order": order, "bc": bc, "dtype": dtype, "dynamic": dyn, "sides": " ".join(groups),
                "length": round(length, 3), "steps": _log(rng, 60, 500),
                "dt": float("%.3g" % (rng.uniform(0.04, 0.12) * (length / 320) ** 2))}
    dim = rng.choice([1, 2, 2])
    n = 2 ** (rng.randint(6, 12) if dim == 1 else rng.randint(5, 11))
    return dict(base, kind="advance", dim=dim, n=n, order=5, bc="periodic", scheme="ssf",
                steps=_log(rng, 20, 60) if n > 600 and dim == 2 else _log(rng, 50, 500))


# ---- inputs --------------------------------------------------------------

def _coeffs(dynamic):
    """The standard workloads' model: g = 1, g_R = 2, R = 1, gamma_c = 1, gamma_R = 1.5."""
    c = np.zeros(23)
    c[2], c[3], c[4], c[5] = 0.5, 0.5, 1.0, 4.0
    c[10], c[11], c[12], c[13] = (1.0 if dynamic else 0.0), 1.0, 1.5, 1.0
    return c


def _model_coeffs():
    """The reference's derived coefficients at its default parameters, in the
    single precision of its entry points."""
    R, gamma, g, tilde_g, gamma_R = 0.0242057488654, 0.0242057488654, 0.00162178517398, 0.0169440242057, 0.242057488654
    phi0 = math.sqrt(gamma / (2.0 * g))
    n0 = 2.0 / (R * phi0)
    c = np.zeros(23)
    c[:5] = 1.0
    c[5] = 4.0 * tilde_g / R
    c[11], c[12], c[13] = 1.0 / (n0 * gamma_R), 1.0, R * phi0 ** 2 / gamma_R
    return c.astype(np.float32).astype(np.float64)


def _fields(dim, n, dx, seed, bc):
    """(psi0, P) of one solve: a Gaussian seed with complex noise and a ring
    pump whose power, radius and width come from the seed."""
    rng = np.random.default_rng(seed)
    P0, half = rng.uniform(0.5, 5.0), n * dx / 2.0
    r0, w = rng.uniform(0.15, 0.5) * half, max(rng.uniform(0.04, 0.12) * half, 2 * dx)
    x = np.linspace(0.0, n * dx, n) if (dim == 1 and bc == "ref") else -half + dx * np.arange(n)
    r = np.abs(x) if dim == 1 else np.sqrt(x[:, None] ** 2 + x[None, :] ** 2)
    noise = rng.standard_normal((2,) + r.shape)
    psi0 = 0.1 * np.exp(-r * r / (0.02 * half * half + 4.0)) + (1e-3 / math.sqrt(2.0)) * (noise[0] + 1j * noise[1])
    return psi0, P0 * np.exp(-(r - r0) ** 2 / (2.0 * w * w))


class _Gaussian(object):
    """Pumping functor of a host model: power exp(-r^2 / (2 variation^2))."""

    def __init__(self, power, variation):
        self.power, self.variation = power, variation

    def __call__(self, *axes):
        return self.power * np.exp(-sum(a * a for a in axes) / (2.0 * self.variation ** 2))


def _model_inputs(dim, n, dx, seed):
    rng = np.random.default_rng(seed)
    pump = _Gaussian(rng.uniform(5.0, 25.0), rng.uniform(0.08, 0.3) * n * dx / 2.0)
    shape = (n,) * dim
    noise = rng.standard_normal((2,) + shape)
    return pump, (0.1 + (1e-3 / math.sqrt(2.0)) * (noise[0] + 1j * noise[1])).astype(np.complex64)


class _Member(object):

    def __init__(self, n, dx, dt, dynamic, seed, bc):
        self.n, self.dx, self.dt, self.coeffs = n, dx, dt, _coeffs(dynamic)
        self.psi0, self.P = _fields(2, n, dx, seed, bc)
        self.n0 = np.zeros((n, n)) if dynamic else None


def _sides(case):
    return [int(g.split("*")[0]) for g in case["sides"].split() for _ in range(int(g.split("*")[1]))]


def _members(case, seed):
    return [_Member(n, case["length"] / n, case["dt"], case["dynamic"], 4096 * seed + i, case["bc"])
            for i, n in enumerate(_sides(case))]


def _models(case, seed):
    out = []
    for i in range(case.get("count", 1)):
        dim = case.get("dim", 2)
        pump, u0 = _model_inputs(dim, case["n"], case["dx"], 4096 * seed + i)
        out.append(Problem().model(model="%dd" % dim, dx=case["dx"], dt=case["dt"], order=case["order"],
                                   num_nodes=case["n"], num_iters=case["steps"], pumping=pump, u0=u0))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "model":
        return {"kind": kind, "model": _models(case, seed)[0]}
    if kind == "sweep":
        return {"kind": kind, "models": _models(case, seed)}
    if kind == "batch":
        return {"kind": kind, "steps": case["steps"],
                "batch": Batch(_members(case, seed), dim=2, order=case["order"], bc=case["bc"], dtype=case["dtype"])}
    desc = native.ProblemDesc.make(case["dim"], case["n"], case["order"], case["dt"], case["dx"],
                                   _coeffs(case["dynamic"]), bc=case["bc"], dtype=case["dtype"], scheme=case["scheme"])
    psi0, P = _fields(case["dim"], case["n"], case["dx"], seed, case["bc"])
    psi0 = torch.from_numpy(psi0.astype(COMPLEX[case["dtype"]])).cuda()
    P = torch.from_numpy(P.astype(REAL[case["dtype"]])).cuda()
    return {"kind": kind, "desc": desc, "steps": case["steps"], "P": P, "psi0": psi0, "psi": torch.empty_like(psi0),
            "nres": torch.empty_like(P) if case["dynamic"] else None,
            "ws": torch.empty(native.workspace_bytes(desc), dtype=torch.uint8, device="cuda")}


def run(state):
    kind = state["kind"]
    if kind == "model":
        return state["model"].solve().getSolution()
    if kind == "sweep":
        return [s.getSolution() for s in solve_models(state["models"])]
    if kind == "batch":
        b = state["batch"]
        b.reset()
        b.advance(state["steps"])
        return [b.psi, b.nres] if b.dynamic else [b.psi]
    state["psi"].copy_(state["psi0"])
    if state["nres"] is not None:
        state["nres"].zero_()
    native.advance(state["desc"], state["steps"], state["P"], state["psi"], state["nres"], state["ws"])
    return [state["psi"], state["nres"]] if state["nres"] is not None else [state["psi"]]


# ---- the work of a pass ----------------------------------------------------

def work(case):
    """Fields read and written once; the scheme's arithmetic at every point
    and step."""
    kind, order = case["kind"], case["order"]
    R = (order - 1) // 2
    dim, bc = case.get("dim", 2), case.get("bc", "ref")
    real = 8 if case.get("dtype", "f32") == "f64" else 4
    dyn = case.get("dynamic", False)
    if kind == "batch":
        pts = sum(n * n for n in _sides(case))
    else:
        pts = case["n"] ** dim * case.get("count", 1)
    point = 16 + (5 if dyn else 4)                        # |y|^2, factors, both components, reservoir
    combine = 8 + (4 if dyn else 0)                       # accumulator and next stage input
    if case.get("scheme", "rk4") == "ssf":
        per = 2 * 5 * dim * math.log2(case["n"]) + 6 + 2 * 4 * (point + combine)
    else:
        lap = 2 * (2 * order) if (dim == 1 and bc == "ref") else 2 * ((5 if dim == 2 else 3) * R + 1)
        per = 4 * (lap + point + combine)
    return {"bytes": pts * real * (2 * (2 + (1 if dyn else 0)) + 1), "flops": pts * case["steps"] * per}


# ---- the same solves in plain torch, double precision ----------------------

def _s2(order, h):
    return {3: [-2.0, 1.0], 5: [-30.0 / 12, 16.0 / 12, -1.0 / 12],
            7: [-490.0 / 180, 270.0 / 180, -27.0 / 180, 2.0 / 180]}[order], 1.0 / (h * h)


def _cartesian(dim, order, h, bc):
    w, s = _s2(order, h)
    R = len(w) - 1

    def along(y, axis):
        n = y.shape[axis]
        if bc == "periodic":
            lo, hi = y.narrow(axis, n - R, R), y.narrow(axis, 0, R)
        else:
            lo = hi = torch.zeros_like(y.narrow(axis, 0, R))
        e = torch.cat([lo, y, hi], axis)
        out = (w[0] * s) * y
        for d in range(1, R + 1):
            out.add_(e.narrow(axis, R - d, n) + e.narrow(axis, R + d, n), alpha=w[d] * s)
        return out

    return lambda y: along(y, -1) + along(y, -2) if dim == 2 else along(y, -1)


def _radial(n, order, h, device):
    """psi'' + psi'/r on r = k h with psi(-r) = psi(r), psi = 0 past the grid."""
    w, s = _s2(order, h)
    first = {3: [0.0, 0.5], 5: [0.0, 8.0 / 12, -1.0 / 12], 7: [0.0, 0.75, -0.15, 1.0 / 60]}[order]
    R = len(w) - 1
    i = np.arange(n)
    taps = []
    for d in range(-R, R + 1):
        a = abs(d)
        wt = np.full(n, w[a] * s)
        wt[1:] += math.copysign(1.0, d) * first[a] / h / (i[1:] * h)
        wt[0] *= 2.0
        j = np.abs(i + d)
        wt[j >= n] = 0.0
        taps.append((torch.from_numpy(np.minimum(j, n - 1)).to(device), torch.from_numpy(wt).to(device)))
    return lambda y: sum(wt * y[..., j] for j, wt in taps)


def _solve_rk4(lap, c, dt, steps, psi, nres, P):
    dyn = nres is not None

    def rhs(y, m):
        s = y.real * y.real + y.imag * y.imag
        decay = c[12] + c[13] * s
        r = m if dyn else c[11] * P / decay
        k = torch.complex(c[2] * r - c[3], -(c[4] * s + c[5] * r)) * y + 1j * lap(y)
        return k, (c[11] * P - decay * m) / c[10] if dyn else None

    for _ in range(steps):
        k, kn = rhs(psi, nres)
        acc, accn = k, kn
        for a, b in ((0.5, 2.0), (0.5, 2.0), (1.0, 1.0)):
            k, kn = rhs(psi + (a * dt) * k, nres + (a * dt) * kn if dyn else None)
            acc = acc + b * k
            accn = accn + b * kn if dyn else None
        psi = psi + (dt / 6.0) * acc
        nres = nres + (dt / 6.0) * accn if dyn else None
    return psi, nres


def _solve_ssf(dim, n, h, c, dt, steps, psi, nres, P):
    k = 2.0 * math.pi * torch.fft.fftfreq(n, d=h, dtype=torch.float64).to(psi.device)
    k2 = k * k if dim == 1 else k[:, None] ** 2 + k[None, :] ** 2
    phase = torch.exp(-1j * k2 * dt)
    axes = tuple(range(-dim, 0))
    for _ in range(steps):
        psi, nres = _solve_rk4(lambda y: 0.0 * y, c, 0.5 * dt, 1, psi, nres, P)
        psi = torch.fft.ifftn(torch.fft.fftn(psi, dim=axes) * phase, dim=axes)
        psi, nres = _solve_rk4(lambda y: 0.0 * y, c, 0.5 * dt, 1, psi, nres, P)
    return psi, nres


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    kind, order = case["kind"], case["order"]

    def wide(a, dtype):
        a = np.asarray(a)
        a = a.astype(COMPLEX[dtype] if np.iscomplexobj(a) else REAL[dtype])
        return torch.from_numpy(a.astype(np.complex128 if np.iscomplexobj(a) else np.float64)).to(device)

    if kind in ("model", "sweep"):
        dim, n = case.get("dim", 2), case["n"]
        dx, dt = float(np.float32(case["dx"])), float(np.float32(case["dt"]))
        psi, P = [], []
        x = np.linspace(0.0, n * case["dx"], n) if dim == 1 else np.linspace(-n * case["dx"] / 2, n * case["dx"] / 2, n)
        for i in range(case.get("count", 1)):
            pump, u0 = _model_inputs(dim, n, case["dx"], 4096 * seed + i)
            psi.append(u0)
            P.append(pump(*np.meshgrid(*([x] * dim))))
        lap = _radial(n, order, dx, device) if dim == 1 else _cartesian(2, order, dx, "ref")
        out, _ = _solve_rk4(lap, _model_coeffs(), dt, case["steps"], wide(np.stack(psi), "f32"), None,
                            wide(np.stack(P), "f32"))
        out = [o for o in out.cpu().numpy()]
        return out if kind == "sweep" else out[0]
    if kind == "batch":
        ms = _members(case, seed)
        offs, o = [], 0
        for m in ms:
            offs.append(o)
            o += -(-m.n * m.n // 64) * 64
        psi = torch.zeros(o, dtype=torch.complex128, device=device)
        nres = torch.zeros(o, dtype=torch.float64, device=device) if case["dynamic"] else None
        for n in sorted({m.n for m in ms}):
            ids = [i for i, m in enumerate(ms) if m.n == n]
            P = wide(np.stack([ms[i].P for i in ids]), case["dtype"])
            y, r = _solve_rk4(_cartesian(2, order, case["length"] / n, case["bc"]), _coeffs(case["dynamic"]),
                              case["dt"], case["steps"], wide(np.stack([ms[i].psi0 for i in ids]), case["dtype"]),
                              torch.zeros_like(P) if case["dynamic"] else None, P)
            for k, i in enumerate(ids):
                psi[offs[i]:offs[i] + n * n] = y[k].reshape(-1)
                if nres is not None:
                    nres[offs[i]:offs[i] + n * n] = r[k].reshape(-1)
        return [psi, nres] if nres is not None else [psi]
    psi, P = (wide(a, case["dtype"]) for a in _fields(case["dim"], case["n"], case["dx"], seed, case["bc"]))
    nres = torch.zeros_like(P) if case["dynamic"] else None
    c = _coeffs(case["dynamic"])
    if case["scheme"] == "ssf":
        psi, nres = _solve_ssf(case["dim"], case["n"], case["dx"], c, case["dt"], case["steps"], psi, nres, P)
    else:
        lap = (_radial(case["n"], order, case["dx"], device) if case["dim"] == 1 and case["bc"] == "ref"
               else _cartesian(case["dim"], order, case["dx"], case["bc"]))
        psi, nres = _solve_rk4(lap, c, case["dt"], case["steps"], psi, nres, P)
    return [psi, nres] if nres is not None else [psi]
