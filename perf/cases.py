"""Performance cases of the Lennard-Jones library: the calls its users make.

Each case is one kind of call through the Python entry points (which are the
C-ABI's), at sizes taken from the benchmark configurations, the task programs
and the tests:

  step   LJSystem.Integrate: `steps` device-resident time steps of one box,
         with the history rows and the state as outputs
  batch  LJBatch.integrate_hist: the same for an ensemble of boxes
  grad   a backward pass through a differentiable trajectory (ljamd.autograd)
  rdf    LJSystem.rdf: the radial-distribution histogram of one configuration
  compat copyArrayToDevice + calculateNForces + copyArrayFromDevice, the force
         call that an unchanged MDSystem makes, from and to host arrays

listed() are the cases that are timed, draw() makes others of the same ranges.
The numbers that come from 32-bit pair sums (history rows, losses, parameter
gradients) are returned as 32-bit values, since that is what they are good for.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.abspath(os.path.join("lennard-jones-cuda_amd", "python")))

import ljamd  # noqa: E402
from ljamd import _lib as _L  # noqa: E402
from ljamd.autograd import trajectory_loss  # noqa: E402
from ljamd.system import CompatArrays  # noqa: E402

_PREC = {"fp32": ljamd.PREC_FP32, "comp": ljamd.PREC_COMPENSATED, "fp64": ljamd.PREC_FP64}
_BC = {"periodic": ljamd.BC_PERIODIC, "wall": ljamd.BC_WALL, "open": ljamd.BC_NONE}
_ENS = {"evn": ljamd.EVN, "tvn": ljamd.TVN}
_RULE = {"cpu": ljamd.RDF_REF_CPU, "gpu": ljamd.RDF_REF_GPU, "rbins": ljamd.RDF_RBINS}


def _step(name, N, rho, T0, ens, bc, prec, dt, steps):
    case = {"kind": "step", "N": N, "rho": rho, "T0": T0, "ens": ens, "bc": bc, "prec": prec,
            "dt": dt, "steps": steps}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one Integrate(dt) of the CPU-runnable configuration: what a GUI or a
        # driver loop that reads the observables after every step calls
        _step("step_one_n400", 400, 0.05, 1.4, "evn", "periodic", "fp32", 0.005, 1),
        # the same configuration as its 2000-step run is made, 50 steps a call
        _step("step_n400", 400, 0.05, 1.4, "evn", "periodic", "fp32", 0.005, 50),
        # liquid of the differentiable workload's size, thermostatted
        _step("step_n2048", 2048, 0.85, 1.0, "tvn", "periodic", "fp32", 0.005, 40),
        # an odd mid-size box with hard walls
        _step("step_n5003_wall", 5003, 0.6, 1.2, "evn", "wall", "fp32", 0.005, 40),
        # the headline configuration
        _step("step_n16384", 16384, 0.85, 1.0, "tvn", "periodic", "fp32", 0.005, 40),
        # the large two-phase system, compensated sums
        _step("step_n131072_comp", 131072, 0.3, 1.0, "evn", "wall", "comp", 0.002, 1),
        # the FP64 mode, the reference of a precision study
        _step("step_n16384_fp64", 16384, 0.85, 1.0, "evn", "periodic", "fp64", 0.005, 10),
        # the 512-box ensemble, with the tiling that its autotuner settles on
        {"name": "batch_512", "kind": "batch", "boxes": 512, "nlo": 200, "nhi": 4000,
         "ens": "evn", "bc": "periodic", "sizes": 7, "tuned": True, "dt": 0.005, "steps": 20},
        # an isotherm: a handful of equal small boxes over a range of densities
        {"name": "batch_isotherm", "kind": "batch", "boxes": 16, "nlo": 400, "nhi": 400,
         "ens": "tvn", "bc": "periodic", "sizes": 7, "tuned": False, "dt": 0.005, "steps": 50},
        # the differentiable workload, a trajectory of two checkpoint intervals
        {"name": "grad_n2048", "kind": "grad", "N": 2048, "rho": 0.85, "T0": 1.0,
         "bc": "periodic", "dt": 0.005, "steps": 40, "every": 20},
        # the 500-bin g(r) of the headline configuration
        {"name": "rdf_n16384", "kind": "rdf", "N": 16384, "rho": 0.85, "bc": "periodic",
         "rule": "rbins", "nbins": 500},
        # the drop-in force call of an unchanged MDSystem at the headline size
        {"name": "compat_n16384", "kind": "compat", "N": 16384, "rho": 0.85, "bc": "periodic"},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["step", "batch", "grad", "rdf", "compat"], [10, 3, 2, 3, 3])[0]
    bc = rng.choice(["periodic", "periodic", "wall", "open"])
    rho = round(rng.uniform(0.05, 0.9), 3)
    T0 = round(rng.uniform(0.8, 2.0), 3)
    if kind == "step":
        prec = rng.choice(["fp32", "fp32", "fp32", "comp", "fp64"])
        N = _logint(rng, 100, 12000 if prec == "fp64" else 40000)
        budget = 1.5e9 if prec == "fp64" else 8e9  # ordered pairs of a pass
        steps = max(1, min(rng.choice([1, 10, 37, 64]), int(budget / N / N)))
        return _step(None, N, rho, T0, rng.choice(["evn", "tvn"]), bc, prec, 0.005, steps)
    if kind == "batch":
        boxes = _logint(rng, 4, 300)
        nlo = rng.randint(100, 600)
        nhi = rng.randint(nlo, 3000)
        pairs = boxes * (nlo * nlo + nlo * nhi + nhi * nhi) / 3
        steps = max(1, min(rng.choice([8, 20, 45]), int(2e10 / pairs)))
        return {"kind": "batch", "boxes": boxes, "nlo": nlo, "nhi": nhi,
                "ens": rng.choice(["evn", "tvn"]), "bc": bc, "sizes": rng.randint(1, 9999),
                "tuned": rng.random() < 0.5, "dt": 0.005, "steps": steps}
    if kind == "grad":
        steps = rng.choice([10, 25, 40])
        return {"kind": "grad", "N": _logint(rng, 200, 4500), "rho": rho, "T0": T0,
                "bc": rng.choice(["periodic", "open"]), "dt": 0.005, "steps": steps,
                "every": rng.choice([5, 10, 20])}
    if kind == "rdf":
        return {"kind": "rdf", "N": _logint(rng, 400, 40000), "rho": rho,
                "bc": "wall" if bc == "open" else bc, "rule": rng.choice(["cpu", "gpu", "rbins"]),
                "nbins": rng.choice([200, 256, 500, 1001])}
    return {"kind": "compat", "N": _logint(rng, 300, 40000), "rho": rho,
            "bc": "wall" if bc == "open" else bc}


# ---- inputs -----------------------------------------------------------------

def _box(N, rho):
    return (N / rho) ** (1.0 / 3.0)


def _positions(rng, N, rho):
    """Simple-cubic sites in [0, L]^3, each displaced by up to 8% of the spacing."""
    L = _box(N, rho)
    n = 1
    while n * n * n < N:
        n += 1
    k = np.arange(N)
    s = np.stack([k // (n * n), (k // n) % n, k % n], axis=1) + 0.5
    p = np.zeros((N, 4), np.float32)
    p[:, :3] = (s + rng.uniform(-0.08, 0.08, (N, 3))) * (L / n)
    return p


def _velocities(rng, N, T0):
    """Maxwell-Boltzmann velocities at exactly T0, without net momentum."""
    v = rng.normal(0.0, math.sqrt(T0), (N, 3))
    v -= v.mean(axis=0)
    v *= math.sqrt(3.0 * N * T0 / np.sum(v * v))
    o = np.zeros((N, 4), np.float32)
    o[:, :3] = v
    return o


def _batch_boxes(case):
    """N, rho and T0 of the boxes: the case's own, whatever the seed of the state."""
    rng = np.random.default_rng(case["sizes"])
    N = rng.integers(case["nlo"], case["nhi"] + 1, case["boxes"]).astype(np.int32)
    if case["nlo"] == case["nhi"]:  # an isotherm: equal boxes, the density stepped, one temperature
        return N, np.linspace(0.05, 0.8, case["boxes"]), np.full(case["boxes"], 1.4)
    return N, rng.uniform(0.05, 0.9, case["boxes"]), rng.uniform(0.8, 2.0, case["boxes"])


def _batch_state(case, rng):
    N, rho, T0 = _batch_boxes(case)
    x = [_positions(rng, int(n), r) for n, r in zip(N, rho)]
    v = [_velocities(rng, int(n), t) for n, t in zip(N, T0)]
    return N, rho, T0, x, v


class _DeviceView:
    """A context's device array as torch sees it; keeps the context alive."""

    def __init__(self, owner, address, N):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (N, 4), "typestr": "<f4", "strides": None,
                                         "data": (address, False), "version": 2}


def _views(s):
    return [torch.as_tensor(_DeviceView(s, a, s.N), device="cuda") for a in s.device_arrays()]


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "batch":
        N, rho, T0, x, v = _batch_state(case, rng)
        b = ljamd.LJBatch(N, rho, T0, canonical=_ENS[case["ens"]], boundary=_BC[case["bc"]])
        if case["tuned"]:
            b.set_tuning(1, 512, 8, 1)
        b.set_array(_L.ARRAY_POS, np.concatenate(x))
        b.set_array(_L.ARRAY_VEL, np.concatenate(v))
        b.compute_forces()
        return {"case": case, "b": b}
    N, rho = case["N"], case["rho"]
    x = _positions(rng, N, rho)
    if kind == "compat":
        return {"case": case, "x": x.reshape(-1), "L": _box(N, rho), "arrays": CompatArrays(N),
                "dr2": float(_L.lib().lj_rdf_dr2_default(N))}
    T0 = case.get("T0", 1.0)
    v = _velocities(rng, N, T0)
    if kind == "grad":
        s = ljamd.LJSystem(N, rho, T0, boundary=_BC[case["bc"]])
        dev = torch.device("cuda:0")
        return {"case": case, "s": s, "v": torch.tensor(v, device=dev),
                "x": torch.tensor(x, device=dev, requires_grad=True),
                "eps": torch.tensor(1.0, dtype=torch.float64, requires_grad=True),
                "sig": torch.tensor(1.0, dtype=torch.float64, requires_grad=True)}
    if kind == "rdf":
        s = ljamd.LJSystem(N, rho, T0, boundary=_BC[case["bc"]])
        s.set_state(x, v)
        return {"case": case, "s": s}
    s = ljamd.LJSystem(N, rho, T0, canonical=_ENS[case["ens"]], boundary=_BC[case["bc"]],
                       precision=_PREC[case["prec"]])
    s.set_state(x, v)
    s.CalculateForces()
    s.CalculateParameters()
    s.resetAveraging()
    return {"case": case, "s": s, "views": _views(s)}


# ---- one pass ---------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        s = state["s"]
        hist = s.Integrate(case["dt"], case["steps"])
        if case["prec"] == "fp64":
            return {"hist": hist, "pos": s.get_array_f64(_L.ARRAY_POS).reshape(-1, 4),
                    "vel": s.get_array_f64(_L.ARRAY_VEL).reshape(-1, 4)}
        pos, vel, force = state["views"]
        # w of the force array holds per-particle energies in some modes only
        return {"hist": hist.astype(np.float32), "pos": pos, "vel": vel, "force": force[:, :3]}
    if kind == "batch":
        b = state["b"]
        hist = b.integrate_hist(case["dt"], case["steps"])
        return {"hist": hist.astype(np.float32), "pos": b.get_array(_L.ARRAY_POS).reshape(-1, 4),
                "vel": b.get_array(_L.ARRAY_VEL).reshape(-1, 4)}
    if kind == "grad":
        loss = trajectory_loss(state["x"], state["eps"], state["sig"], state["s"], state["v"],
                               dt=case["dt"], nsteps=case["steps"],
                               checkpoint_every=case["every"])
        gx, ge, gs = torch.autograd.grad(loss, (state["x"], state["eps"], state["sig"]))
        return {"loss": loss.detach().float(), "dx": gx, "deps": ge.float(), "dsig": gs.float()}
    if kind == "rdf":
        return {"counts": state["s"].rdf(_RULE[case["rule"]], case["nbins"]).astype(np.int64)}
    force, pressure, rdf = state["arrays"].calculate(state["x"], state["L"],
                                                     case["bc"] == "periodic", state["dr2"])
    return {"force": force.reshape(-1, 4), "pressure": pressure, "rdf": rdf}


# ---- what a pass cannot do without ------------------------------------------

_PAIR_FLOPS = 30  # of an unordered pair: separation 8, (s/r)^2 2, powers 6, two forces 12, sums 2
_ADJ_FLOPS = 75   # of an unordered pair of the adjoint pass (H z, force, virial gradient, sums)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        N = _batch_boxes(case)[0].astype(float)
        pairs = float(np.sum(N * (N - 1) / 2))
        return {"flops": case["steps"] * pairs * _PAIR_FLOPS,
                "bytes": float(N.sum()) * 16 * 5 + case["steps"] * case["boxes"] * 40}
    N = float(case["N"])
    pairs = N * (N - 1) / 2
    if kind == "step":
        size = 32 if case["prec"] == "fp64" else 16
        return {"flops": case["steps"] * pairs * _PAIR_FLOPS, "bytes": N * size * 6 + 40 * case["steps"]}
    if kind == "grad":
        # forward and reverse, each state once
        return {"flops": case["steps"] * pairs * (_PAIR_FLOPS + _ADJ_FLOPS),
                "bytes": N * 16 * 3 + case["steps"] * N * 32 * 2}
    if kind == "rdf":
        return {"flops": pairs * 10, "bytes": N * 16 + 8 * case["nbins"]}
    return {"flops": pairs * (_PAIR_FLOPS + 10), "bytes": N * 32 + 1024}


# ---- the same in 64 bits ----------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _forces(x, L, periodic, eps=1.0, sig=1.0):
    """Forces, pair energies per particle (halves) and the virial sum r.f / 2,
    all pairs in double, in blocks of rows."""
    N = x.shape[0]
    rows = max(1, min(N, 60_000_000 // N))
    F, e, w = [], [], []
    for i0 in range(0, N, rows):
        d = x[i0:i0 + rows, None, :] - x[None, :, :]
        if periodic:
            d = d - L * torch.round(d.detach() / L)
        r2 = (d * d).sum(-1)
        self_pair = torch.zeros_like(r2, dtype=torch.bool)
        k = torch.arange(r2.shape[0], device=x.device)
        self_pair[k, k + i0] = True
        q = (sig * sig) / r2.masked_fill(self_pair, 1.0)
        q3 = (q * q * q).masked_fill(self_pair, 0.0)
        t = q3 * (2.0 * q3 - 1.0)
        F.append(((24.0 * eps / (sig * sig)) * t * q).unsqueeze(-1).mul(d).sum(1))
        e.append((2.0 * eps) * (q3 * q3 - q3).sum(1))
        w.append((12.0 * eps) * t.sum(1))
    return torch.cat(F), torch.cat(e), torch.cat(w)


def _trajectory(x, v, N, rho, T0, ens, bc, dt, steps):
    """`steps` velocity-Verlet steps in double: history rows, x, v, forces."""
    L = _box(N, rho)
    per = bc == "periodic"
    f, _, _ = _forces(x, L, per)
    hist = []
    for _ in range(steps):
        x = x + dt * v + 0.5 * dt * dt * f
        g, e, w = _forces(x, L, per)
        if ens == "evn":
            v = v + 0.5 * dt * (f + g)
        else:
            tf = 0.5 * (f + g)
            tv = v + 0.5 * dt * tf
            chi = torch.sqrt(T0 / ((tv * tv).sum() / (3.0 * N)))
            v = (2.0 * chi - 1.0) * v + chi * dt * tf
        f = g
        if bc == "periodic":
            x = torch.where(x < 0, x + L, x)
            x = torch.where(x > L, x - L, x)
        elif bc == "wall":
            v = torch.where(((x < 0) & (v < 0)) | ((x > L) & (v > 0)), -v, v)
        K = 0.5 * (v * v).sum()
        T = 2.0 * K / 3.0 / N
        V, W = e.sum(), w.sum()
        hist.append(torch.stack([K + V, T, K, V, (W / 3.0 + N * T) / (N / rho)]))
    return torch.stack(hist), x, v, f


def _four(a):
    return torch.nn.functional.pad(a, (0, 1))


def exact(case, seed):
    kind = case["kind"]
    if kind == "rdf":
        return None
    rng = np.random.default_rng(seed)
    dev = _device()
    if dev.type == "cpu" and case.get("N", 99999) > 3000:
        return None

    def wide(a):
        return torch.tensor(a[:, :3], dtype=torch.float64, device=dev)

    if kind == "batch":
        N, rho, T0, x, v = _batch_state(case, rng)
        out = [_trajectory(wide(a), wide(b), int(n), r, t, case["ens"], case["bc"], case["dt"],
                           case["steps"]) for n, r, t, a, b in zip(N, rho, T0, x, v)]
        return {"hist": torch.stack([o[0] for o in out], 1), "pos": _four(torch.cat([o[1] for o in out])),
                "vel": _four(torch.cat([o[2] for o in out]))}
    N, rho = case["N"], case["rho"]
    x = wide(_positions(rng, N, rho))
    if kind == "compat":
        F, e, w = _forces(x, float(np.float32(_box(N, rho))), case["bc"] == "periodic")
        # Force.w: sum over the particle's pairs of (1/r^12 - 1/r^6); pressure:
        # a third of the virial summed over ordered pairs
        return {"force": torch.cat([F, (e / 2.0).unsqueeze(1)], 1), "pressure": w.sum() / 3.0,
                "rdf": None}
    v = wide(_velocities(rng, N, case["T0"]))
    if kind == "step":
        hist, x, v, f = _trajectory(x, v, N, rho, case["T0"], case["ens"], case["bc"], case["dt"],
                                    case["steps"])
        out = {"hist": hist, "pos": _four(x), "vel": _four(v)}
        return out if case["prec"] == "fp64" else out | {"force": f}
    if N * N * case["steps"] > 4e8:
        return None
    L, per, dt, M = _box(N, rho), case["bc"] == "periodic", case["dt"], case["steps"]
    x0 = x.clone().requires_grad_(True)
    eps = torch.ones((), dtype=torch.float64, device=dev, requires_grad=True)
    sig = torch.ones((), dtype=torch.float64, device=dev, requires_grad=True)
    x, E, P = x0, 0.0, 0.0
    f, _, _ = _forces(x, L, per, eps, sig)
    for _ in range(M):
        x = x + dt * v + 0.5 * dt * dt * f
        g, e, w = _forces(x, L, per, eps, sig)
        v = v + 0.5 * dt * (f + g)
        f = g
        E = E + e.sum() / M
        P = P + (w.sum() / 3.0 + (v * v).sum() / 3.0) / L ** 3 / M
    loss = E + (P - 1.0) ** 2
    gx, ge, gs = torch.autograd.grad(loss, (x0, eps, sig))
    return {"loss": loss.detach(), "dx": _four(gx), "deps": ge, "dsig": gs}
