"""The work that a user of this framework has it do, as measurable cases.

Every case is one pass through the public objects (ProblemSolver,
PBProblemSolver): put the initial states in place, Solve (or record and
reverse the discrete adjoint), bring the results to the host and wait.
Small calls go the way the tutorials go (fill the host mirrors, upload
everything, Solve, download everything); large ensembles keep their inputs in
HBM and restore the initial states on the device.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "massively-parallel-gpu-ode-solver_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from mpgos import PB, Algorithms, PBProblemSolver, Precision, ProblemSolver  # noqa: E402
from mpgos import ListOfSolverOptions as O  # noqa: E402
from mpgos import ListOfVariables as V  # noqa: E402
from mpgos import workloads as W  # noqa: E402
from mpgos.tuning import DeviceSnapshot, apply  # noqa: E402

TWO_PI = 2.0 * math.pi
_PREC = {"f64": Precision.DOUBLE, "f32": Precision.FLOAT, "f32k": Precision.FLOAT_KAHAN}
# launch shapes that the autotuner settles on for large ensembles, and the default
_FORMS = {"default": None, "persistent": {"mode": 1, "block": 256, "round": 32},
          "relaunch": {"mode": 2, "block": 256, "relaunch": 200, "launches": 32},
          "sorted": {"mode": 3, "block": 64, "relaunch": 400}}


def listed():
    return [
        # impact dynamics tutorial: a few hundred valves, one Solve up to the next maximum of the lift; the latency of a
        # small call (uploads, one short launch, downloads)
        {"name": "valve_256", "family": "valve", "nt": 256},
        # first tutorial: double-well oscillators with two event functions, accessories and 200 points of dense output,
        # one forcing period per Solve
        {"name": "double_well_dense", "family": "double_well", "nt": 4000, "ndo": 200, "tol": 1e-9},
        # parameter scan at a fixed step: 64 forcing periods of RK4 in one Solve
        {"name": "duffing_rk4_16384", "family": "duffing_rk4", "nt": 16384, "periods": 64, "steps": 1000, "prec": "f64"},
        # adaptive ensemble of an ordinary, ragged size with the default launch
        {"name": "lorenz_50001", "family": "lorenz", "nt": 50001, "tol": 1e-10, "form": "default", "prec": "f64"},
        # the headline ensemble with the tuned launch
        {"name": "lorenz_262144_sorted", "family": "lorenz", "nt": 262144, "tol": 1e-10, "form": "sorted", "prec": "f64"},
        # single precision with compensated sums at a single-precision tolerance
        {"name": "lorenz_65536_f32k", "family": "lorenz", "nt": 65536, "tol": 1e-6, "form": "default", "prec": "f32k"},
        # uneven time scales with Poincare sections logged: horizons of two orders of magnitude
        {"name": "uneven_20000", "family": "uneven", "nt": 20000, "tol": 1e-9, "cap": 2000.0, "evcap": 64, "form": "sorted"},
        # gradients of a long fixed-step trajectory
        {"name": "adjoint_rk4_65536", "family": "adjoint", "nt": 65536, "alg": "rk4", "periods": 64, "k": 16},
        # gradients of an adaptive trajectory, ragged size
        {"name": "adjoint_rkck45_10007", "family": "adjoint", "nt": 10007, "alg": "rkck45", "periods": 4, "k": 16},
        # coupled systems: rings of 256 units with a dense coupling matrix
        {"name": "ring_4096x256", "family": "ring", "ns": 4096, "ups": 256, "periods": 4, "tol": 1e-9, "prec": "f64"},
        # the same at sizes that are no multiple of anything
        {"name": "ring_1000x100", "family": "ring", "ns": 1000, "ups": 100, "periods": 4, "tol": 1e-9, "prec": "f64"},
        # gradients of coupled systems with respect to states, unit and system parameters
        {"name": "ring_adjoint_1024x128", "family": "ring_adjoint", "ns": 1024, "ups": 128, "periods": 2, "tol": 1e-8, "k": 32},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["valve", "double_well", "duffing_rk4", "duffing_rk4", "lorenz", "lorenz", "uneven", "adjoint",
                         "adjoint", "ring", "ring", "ring_adjoint", "ring_tutorial"])
    if family == "valve":
        return {"family": family, "nt": _log(rng, 64, 20000)}
    if family == "double_well":
        return {"family": family, "nt": _log(rng, 100, 10000), "ndo": rng.choice([0, 50, 200]), "tol": 10.0 ** -rng.randint(7, 10)}
    if family == "duffing_rk4":
        return {"family": family, "nt": _log(rng, 100, 65536), "periods": _log(rng, 2, 64), "steps": rng.randint(200, 1000),
                "prec": rng.choice(["f64", "f64", "f64", "f32k"])}
    if family == "lorenz":
        prec = rng.choice(["f64", "f64", "f64", "f32", "f32k"])
        tol = 10.0 ** -rng.randint(7, 10) if prec == "f64" else 10.0 ** -rng.randint(4, 6)
        return {"family": family, "nt": _log(rng, 1000, 262144), "tol": tol, "form": rng.choice(sorted(_FORMS)), "prec": prec}
    if family == "uneven":
        return {"family": family, "nt": _log(rng, 500, 20000), "tol": 10.0 ** -rng.randint(7, 9),
                "cap": float(_log(rng, 100, 2000)), "evcap": rng.randint(0, 64), "form": rng.choice(["default", "relaunch", "sorted"])}
    if family == "adjoint":
        alg = rng.choice(["rk4", "rkck45"])
        return {"family": family, "nt": _log(rng, 500, 65536), "alg": alg, "periods": _log(rng, 2, 32), "k": rng.randint(8, 32)}
    if family == "ring":
        prec = rng.choice(["f64", "f64", "f64", "f32"])
        ups = rng.choice([32 * rng.randint(1, 8), _log(rng, 12, 250)])
        most = (4096 if ups % 32 == 0 and prec == "f64" else 800) * min(1.0, (256.0 if ups % 32 == 0 and prec == "f64" else 128.0) / ups)
        return {"family": family, "ns": _log(rng, 16, most), "ups": ups, "periods": rng.randint(1, 4),
                "tol": 10.0 ** -rng.randint(7, 9) if prec == "f64" else 1e-5, "prec": prec}
    if family == "ring_adjoint":
        return {"family": family, "ns": _log(rng, 16, 1024), "ups": 32 * rng.randint(1, 4), "periods": 1, "tol": 1e-8,
                "k": rng.randint(8, 32)}
    return {"family": family, "ns": _log(rng, 2, 400), "ups": 14, "spb": rng.choice([1, 3, 4])}


# ---------------------------------------------------------------- inputs
def _inputs(case, seed):
    """Description of the inputs (sizes, options and arrays), made from the seed."""
    f, r = case["family"], np.random.RandomState(seed % (1 << 32))
    if f == "valve":
        s = W.tutorial_relief_valve(nt=case["nt"])
        s["X"][0] = 0.2 + 0.02 * r.uniform(-1, 1, case["nt"])
        s["cPAR"][0] *= 1.0 + 0.05 * r.uniform(-1, 1, case["nt"])
        s["cPAR"][0] = np.maximum(s["cPAR"][0], 0.2)
        return s
    if f == "double_well":
        nt = case["nt"]
        s = W.new_spec("duffing_dw", Algorithms.RKCK45, nt, ndo=case["ndo"])
        s["TD"][1] = TWO_PI
        s["X"][0] = -0.5 + 0.1 * r.uniform(-1, 1, nt)
        s["X"][1] = -0.1 + 0.1 * r.uniform(-1, 1, nt)
        s["cPAR"][0] = W.linspace(0.2, 0.3, nt)
        s["sPAR"][0] = 0.3
        s["rtol"] = s["atol"] = case["tol"]
        s["edir"] = np.array([-1, 0])
        s["options"].update(dtmax=1e3, dtmin=1e-14, grow=10.0, shrink=0.2)
        return s
    if f == "duffing_rk4":
        nt = case["nt"]
        s = W.config0_duffing_rk4(nt=nt)
        s["TD"][1] = case["periods"] * TWO_PI
        s["options"]["dt0"] = TWO_PI / case["steps"]
        s["X"][0] += 0.05 * r.uniform(-1, 1, nt)
        s["cPAR"][1] *= 1.0 + 0.01 * r.uniform(-1, 1, nt)
        return s
    if f == "lorenz":
        nt = case["nt"]
        s = W.new_spec("lorenz", Algorithms.RKCK45, nt)
        s["cPAR"][0] = r.uniform(0.0, 21.0, nt)
        s["X"][:] = 10.0 + 0.1 * r.standard_normal((3, nt))
        s["TD"][1] = 10.0
        s["rtol"] = s["atol"] = case["tol"]
        return s
    if f == "uneven":
        nt = case["nt"]
        s = W.new_spec("duffing_eps", Algorithms.RKCK45, nt)
        eps = 10.0 ** r.uniform(-3.0, 0.0, nt)
        periods = np.round(2.0 ** r.uniform(4.0, 12.0, nt))
        s["cPAR"][0] = 0.2
        s["cPAR"][1] = W.linspace(0.3, 10.0, nt)
        s["cPAR"][2] = eps
        s["TD"][1] = np.minimum(periods * TWO_PI / eps, case["cap"] * 10.0 ** r.uniform(-2.0, 0.0, nt))
        s["X"][0] = -0.5
        s["X"][1] = 0.1
        s["rtol"] = s["atol"] = case["tol"]
        s["etol"] = 1e-6
        s["evcap"] = case["evcap"]
        return s
    if f == "adjoint":
        nt = case["nt"]
        alg = Algorithms.RK4 if case["alg"] == "rk4" else Algorithms.RKCK45
        s = W.config3_duffing_adjoint(nt=nt, algorithm=alg, periods=case["periods"])
        s["cPAR"][0] = 0.2 * (1.0 + r.uniform(-0.05, 0.05, nt))
        s["cPAR"][1] = W.linspace(0.3, 10.0, nt) * (1.0 + r.uniform(-0.05, 0.05, nt))
        s["TD"][1] = case["periods"] * TWO_PI
        s["lam"] = r.standard_normal((3, nt))
        # accepted steps that a user's earlier Solve has shown to suffice
        s["cap"] = case["periods"] * 500 + 1 if case["alg"] == "rk4" else case["periods"] * 420 + 200
        return s
    if f in ("ring", "ring_adjoint"):
        ns, ups = case["ns"], case["ups"]
        s = W.new_pb_spec("ring_duffing" if f == "ring" else "ring_duffing_q", Algorithms.RKCK45, ns, ups)
        C = math.sqrt(0.05 / ups) * r.standard_normal((ups, ups))
        np.fill_diagonal(C, 0.0)
        s["dense_coupling"] = C
        s["cMat"] = W.store_coupling(C, 0, 0)
        s["uPAR"][0] = 0.2
        s["sPAR"][0] = r.uniform(0.5, 5.0, ns)
        s["X"][:2] = r.uniform(-1.0, 1.0, (2, ns * ups))
        s["TD"][1] = case["periods"] * TWO_PI
        s["strength"][0] = 1.0
        s["cIndex"][0] = 1
        s["rtol"] = s["atol"] = case["tol"]
        if f == "ring_adjoint":
            s["lam"] = r.standard_normal((3, ns * ups))
            s["cap"] = case["periods"] * 420 + 200
        return s
    ns = case["ns"]
    s = W.tutorial_ring_dw(ns=25)
    t = W.new_pb_spec("ring_dw", Algorithms.RKCK45, ns, 14, cbw=1, cci=1, ndo=100)
    for k in ("options", "rtol", "atol", "edir", "cIndex", "gPAR", "cMat"):
        t[k] = s[k]
    t["TD"][1] = 10.0 * TWO_PI / 0.5
    t["strength"][:] = 0.002
    t["sACC"][:] = 1e-2
    t["uPAR"][:] = np.array([0.5, 0.24, 13.633])[:, None]
    t["X"][:] = -5.0
    t["X"][0, 11::14] = r.uniform(-8.0, 8.0, ns)
    t["X"][1, 11::14] = r.uniform(-20.0, 40.0, ns)
    t["uACC"][:2] = t["X"]
    return t


class _Owned:
    """A host mirror that keeps its solver alive as long as the array is used."""

    def __init__(self, solver, array):
        self.solver = solver
        self.__array_interface__ = array.__array_interface__


def _results(solver, variables):
    return {v.name: np.asarray(_Owned(solver, solver.host_array(v))) for v in variables if solver.host_array(v).size}


def prepare(case, seed):
    f, spec = case["family"], _inputs(case, seed)
    if "ns" in case:
        s = PBProblemSolver(spec["system"], spec["ns"], spec["ups"], spec["algorithm"], _PREC[case.get("prec", "f64")],
                            spb=case.get("spb", 1), cbw=spec["cbw"], cci=spec["cci"], ndo=spec["ndo"])
        W.load_pb(s, spec)
        state = {"solver": s, "family": f, "case": case, "spec": spec}
        if f == "ring_tutorial":
            state["inputs"] = {k: spec[n].copy() for k, n in ((PB.ActualState, "X"), (PB.UnitAccessories, "uACC"),
                                                              (PB.SystemAccessories, "sACC"))}
            state["results"] = _results(s, (PB.ActualState, PB.ActualTime, PB.UnitAccessories, PB.SystemAccessories,
                                            PB.IntegerSystemAccessories, PB.DenseIndex, PB.DenseTime, PB.DenseState,
                                            PB.AcceptedSteps, PB.RejectedSteps, PB.Status))
            return state
        state["snapshot"] = DeviceSnapshot(s, (PB.ActualState, PB.ActualTime))
        state["download"] = (PB.ActualState, PB.ActualTime, PB.AcceptedSteps, PB.RejectedSteps, PB.Status)
        state["results"] = _results(s, state["download"])
        return state
    s = ProblemSolver(spec["system"], spec["nt"], spec["algorithm"], _PREC[case.get("prec", "f64")], ndo=spec["ndo"])
    W.load(s, spec)
    if _FORMS[case.get("form", "default")]:
        apply(s, _FORMS[case["form"]])
    state = {"solver": s, "family": f, "case": case, "spec": spec}
    if f in ("valve", "double_well"):
        state["inputs"] = {V.ActualState: s.host_array(V.ActualState).copy()}
        state["results"] = _results(s, (V.ActualState, V.ActualTime, V.Accessories, V.IntegerAccessories, V.DenseIndex,
                                        V.DenseTime, V.DenseState, V.AcceptedSteps, V.RejectedSteps, V.Status,
                                        V.EventCount))
        return state
    state["snapshot"] = DeviceSnapshot(s, (V.ActualState, V.ActualTime))
    state["download"] = [V.ActualState, V.ActualTime, V.AcceptedSteps, V.RejectedSteps, V.Status]
    if f == "duffing_rk4":
        state["download"].append(V.Accessories)
    if f == "uneven":
        state["download"] += [V.EventCount] + ([V.EventLog] if spec["evcap"] else [])
    state["results"] = _results(s, state["download"])
    return state


def run(state):
    s, f = state["solver"], state["family"]
    if "inputs" in state:
        # the tutorials' sequence over the host mirrors
        for var, value in state["inputs"].items():
            s.host_array(var)[...] = value
        every = PB.All if f == "ring_tutorial" else V.All
        s.SynchroniseFromHostToDevice(every)
        s.Solve()
        s.SynchroniseFromDeviceToHost(every)
        s.InsertSynchronisationPoint()
        s.SynchroniseSolver()
        return state["results"]
    state["snapshot"].restore()
    if f == "adjoint":
        k, cap = state["case"]["k"], state["spec"]["cap"]
        gx, gp = s.adjoint(state["spec"]["lam"], k, cap // k + 2)
        return {"dx0": gx, "dpar": gp}
    if f == "ring_adjoint":
        k, cap = state["case"]["k"], state["spec"]["cap"]
        gx, gu, gs = s.adjoint(state["spec"]["lam"], k, cap // k + 2, cap)
        return {"dx0": gx, "dunit": gu, "dsys": gs}
    s.Solve()
    for var in state["download"]:
        s.SynchroniseFromDeviceToHost(var)
    s.InsertSynchronisationPoint()
    s.SynchroniseSolver()
    return state["results"]


# ---------------------------------------------------------------- what a pass cannot do without
def _steps(case):
    """Attempted steps of an instance or system (estimate from the horizon and the tolerance)."""
    f = case["family"]
    if f == "duffing_rk4":
        return case["periods"] * case["steps"]
    if f == "adjoint":
        return case["periods"] * (500 if case["alg"] == "rk4" else 195)
    scale = (1e-9 / case["tol"]) ** 0.2 if "tol" in case else 1.0
    return {"valve": 120.0, "double_well": 95.0 * scale, "lorenz": 620.0 * scale, "uneven": 2.4 * case.get("cap", 0.0) * scale,
            "ring": 286.0 * case.get("periods", 0) * scale, "ring_adjoint": 290.0 * case.get("periods", 0) * scale,
            "ring_tutorial": 90.0}[f]


def work(case):
    f, n = case["family"], _steps(case)
    word = 4 if case.get("prec", "f64") != "f64" else 8
    if "ns" in case:
        ns, ups = case["ns"], case["ups"]
        flops = ns * n * (6 * 2 * (ups * ups if f != "ring_tutorial" else 6 * ups) + 404.0 * ups)
        size = ns * ups * word * (2 * 2 + 1) + ups * ups * word + ns * 60
        if f == "ring_adjoint":
            flops, size = 3.0 * flops, size + ns * ups * 8 * 4
        if f == "ring_tutorial":
            size += ns * ups * 8 * 2 * n
        return {"bytes": size, "flops": flops}
    nt = case["nt"]
    per = {"valve": 420.0, "double_well": 430.0, "duffing_rk4": 212.0, "lorenz": 283.0, "uneven": 449.0,
           "adjoint": 229.0 if case.get("alg") == "rk4" else 505.0}[f]
    flops = nt * n * per
    size = nt * (word * 8 + 40)
    if f == "adjoint":
        flops, size = 3.0 * flops, nt * 8 * 15
    if f == "double_well":
        size += nt * 8 * 3 * min(case["ndo"], n)
    if f == "uneven":
        size += nt * 24 * case["evcap"]
    return {"bytes": size, "flops": flops}


# ---------------------------------------------------------------- the same in 64 bits, in plain torch
_A = ((1 / 5,), (3 / 40, 9 / 40), (3 / 10, -9 / 10, 6 / 5), (-11 / 54, 5 / 2, -70 / 27, 35 / 27),
      (1631 / 55296, 175 / 512, 575 / 13824, 44275 / 110592, 253 / 4096))
_C = (0.0, 1 / 5, 3 / 10, 3 / 5, 1.0, 7 / 8)
_B = (37 / 378, 0.0, 250 / 621, 125 / 594, 0.0, 512 / 1771)
_E = tuple(b - d for b, d in zip(_B, (2825 / 27648, 0.0, 18575 / 48384, 13525 / 55296, 277 / 14336, 1 / 4)))


def _combine(weights, ks):
    out = None
    for w, k in zip(weights, ks):
        if w:
            out = w * k if out is None else out + w * k
    return out


def _stages(rhs, X, t, h):
    """Cash-Karp stage states, their times and derivatives."""
    ys, ts, ks = [], [], []
    for j in range(6):
        ys.append(X if j == 0 else X + h * _combine(_A[j - 1], ks))
        ts.append(t + _C[j] * h)
        ks.append(rhs(ts[j], ys[j]))
    return ys, ts, ks


def _adaptive(rhs, X, td, tol, safety, reduce, opts, ef=None, edir=None, etol=1e-6, accepted=None, event=None, keep=None):
    """Cash-Karp with the solver's controller over all instances at once.  X is (components, ...) and the time has the
    shape that `reduce` gives a per-component quantity (instances, or systems of units)."""
    wide = (lambda v: v) if X.dim() == 2 else (lambda v: v[:, None])
    t, end = td[0].clone(), td[1]
    dt = torch.full_like(t, opts.get("dt0", 1e-2))
    dtmin, dtmax, grow, shrink = opts.get("dtmin", 1e-12), opts.get("dtmax", 1e6), opts.get("grow", 5.0), opts.get("shrink", 0.1)
    done = torch.zeros_like(t, dtype=torch.bool)
    values = ef(X) if ef else None
    it = 0
    while it % 32 or not bool(done.all()):
        it += 1
        left = end - t
        last = dt > left
        h = torch.where(last, left, dt)
        hw = wide(h)
        ys, ts, ks = _stages(rhs, X, wide(t), hw)
        nx = X + hw * _combine(_B, ks)
        err = hw * _combine(_E, ks).abs() + 1e-18
        lim = torch.clamp(tol * torch.maximum(nx.abs(), X.abs()), min=tol)
        ok = reduce((err < lim).to(torch.float64)) > 0.5
        ratio = torch.clamp(reduce(lim / err), max=1e30)
        fac = torch.clamp(safety * torch.where(ok, ratio ** 0.2, ratio ** 0.25), min=shrink, max=grow)
        new = torch.clamp(h * fac, min=dtmin, max=dtmax)
        if ef:
            cand = ef(nx)
            for i in range(len(cand)):
                cross = torch.zeros_like(ok)
                if edir[i] <= 0:
                    cross |= (values[i] > etol) & (cand[i] < -etol)
                if edir[i] >= 0:
                    cross |= (values[i] < -etol) & (cand[i] > etol)
                cross &= ok
                short = torch.where(cross, -values[i] / (cand[i] - values[i]) * h, h)
                best = short if i == 0 else torch.minimum(best, short)
                hit = cross if i == 0 else hit | cross
            hit &= best >= dtmin
            new = torch.where(hit, best, new)
            ok = ok & ~hit
        go = ok & ~done
        if keep is not None:
            keep.append((X, t, torch.where(go, h, torch.zeros_like(h)), go))
        X = torch.where(wide(go), nx, X)
        t = torch.where(go, t + h, t)
        stop = go & last
        if accepted:
            stop |= accepted(X, t, go)
        if ef:
            for i in range(len(cand)):
                found = torch.zeros_like(ok)
                if edir[i] <= 0:
                    found |= (values[i] > etol) & (cand[i].abs() < etol)
                if edir[i] >= 0:
                    found |= (values[i] < -etol) & (cand[i].abs() < etol)
                found &= go
                if event:
                    X, extra = event(i, found, X, t)
                    stop |= found & extra
            after = ef(X)
            values = [torch.where(go, a, v) for a, v in zip(after, values)]
        dt = torch.where(done, dt, new)
        done = done | stop
    return X, t


def _back(vjp, steps, lam, mu, wide, rk4=None):
    """Adjoint of the recorded steps, last to first (step sizes taken as given)."""
    for X, t, h, go in reversed(steps):
        hw, tw = wide(h), wide(t)
        if rk4:
            ys, ts, a = [X], [tw, tw + 0.5 * hw, tw + 0.5 * hw, tw + hw], (0.5, 0.5, 1.0)
            for j in range(3):
                ys.append(X + a[j] * hw * rk4(ts[j], ys[j]))
            weights, lower = (1 / 6, 1 / 3, 1 / 3, 1 / 6), (None, (0.5,), (0.0, 0.5), (0.0, 0.0, 1.0))
        else:
            ys, ts, _ = _stages(vjp.rhs, X, tw, hw)
            weights, lower = _B, (None,) + _A
        kb = [w * hw * lam for w in weights]
        total = lam
        for j in reversed(range(len(weights))):
            gx, gp = vjp(ts[j], ys[j], kb[j])
            total = total + gx
            mu = [m + g for m, g in zip(mu, gp)]
            for i in range(j):
                if lower[j][i]:
                    kb[i] = kb[i] + lower[j][i] * hw * gx
        lam = total
    return lam, mu


def exact(case, seed):
    f, spec = case["family"], _inputs(case, seed)
    single = case.get("prec", "f64") != "f64"

    def dev(a):
        a = np.asarray(a, np.float32 if single else np.float64)
        return torch.from_numpy(np.ascontiguousarray(a)).to("cuda").to(torch.float64)

    if f in ("ring", "ring_adjoint"):
        ns, ups = case["ns"], case["ups"]
        C, B, k = dev(spec["dense_coupling"]), dev(spec["sPAR"][0])[:, None], 0.2
        X = dev(spec["X"]).reshape(-1, ns, ups)

        def rhs(t, X):
            x, v = X[0], X[1]
            dv = -k * v + B * torch.cos(t) - (x + x * x * x) + x @ C.T
            return torch.stack((v, dv) if f == "ring" else (v, dv, x * x))

        def low(a):
            return a.amin(dim=(0, 2))

        if f == "ring":
            X, t = _adaptive(rhs, X, dev(spec["TD"]), case["tol"], 0.8, low, spec["options"])
            return {"ActualState": X.reshape(2, -1), "ActualTime": t, "AcceptedSteps": None, "RejectedSteps": None, "Status": None}
        if _steps(case) * ns * ups * 24 > 40e9:
            return None
        kept = []
        _adaptive(rhs, X, dev(spec["TD"]), case["tol"], 0.8, low, spec["options"], keep=kept)

        def vjp(t, X, kb):
            x, v = X[0], X[1]
            gx = torch.stack((-(1 + 3 * x * x) * kb[1] + 2 * x * kb[2] + kb[1] @ C, kb[0] - k * kb[1], torch.zeros_like(x)))
            return gx, (-v * kb[1], torch.cos(t) * kb[1])

        vjp.rhs = rhs
        lam = dev(spec["lam"]).reshape(3, ns, ups)
        lam, mu = _back(vjp, kept, lam, [torch.zeros_like(lam[0])] * 2, lambda v: v[:, None])
        return {"dx0": lam.reshape(3, -1), "dunit": mu[0].reshape(1, -1), "dsys": mu[1].sum(dim=1)[None]}
    if f == "ring_tutorial":
        return None
    X, td, par = dev(spec["X"]), dev(spec["TD"]), dev(spec["cPAR"])

    def low(a):
        return a.amin(dim=0)

    if f == "lorenz":
        def rhs(t, X):
            x, y, z = X
            return torch.stack((10 * (y - x), par[0] * x - y - x * z, x * y - 8 / 3 * z))
        X, t = _adaptive(rhs, X, td, case["tol"], 0.9, low, spec["options"])
        return {"ActualState": X, "ActualTime": t, "AcceptedSteps": None, "RejectedSteps": None, "Status": None}
    if f == "duffing_rk4":
        # long forced trajectories of this oscillator are chaotic: rounding is amplified to the size of the state
        if case["periods"] > 12 or _steps(case) > 12000:
            return None
        t, h = td[0].clone(), spec["options"]["dt0"]
        most = X[0].abs()

        def rhs(t, X):
            return torch.stack((X[1], -par[0] * X[1] + par[1] * torch.cos(t) - (X[0] + X[0] ** 3)))
        while True:
            left = td[1] - t
            last = h > left
            s = torch.where(last, left, torch.full_like(left, h))
            k1 = rhs(t, X)
            k2 = rhs(t + 0.5 * s, X + 0.5 * s * k1)
            k3 = rhs(t + 0.5 * s, X + 0.5 * s * k2)
            k4 = rhs(t + s, X + s * k3)
            X, t = X + s / 6 * (k1 + 2 * k2 + 2 * k3 + k4), t + s
            most = torch.maximum(most, X[0].abs())
            if float(t[0]) > float(td[1][0]) - 1.5 * h and bool(last.all()):
                break
        return {"ActualState": X, "ActualTime": t, "Accessories": most[None], "AcceptedSteps": None, "RejectedSteps": None, "Status": None}
    if f == "adjoint":
        if case["periods"] > 6 or case["nt"] * _steps(case) * 60 > 40e9:
            return None

        def rhs(t, X):
            return torch.stack((X[1], -par[0] * X[1] + par[1] * torch.cos(t) - (X[0] + X[0] ** 3), X[0] * X[0]))

        def vjp(t, X, kb):
            x, v = X[0], X[1]
            gx = torch.stack((-(1 + 3 * x * x) * kb[1] + 2 * x * kb[2], kb[0] - par[0] * kb[1], torch.zeros_like(x)))
            return gx, (-v * kb[1], torch.cos(t) * kb[1])
        vjp.rhs = rhs
        lam, kept = dev(spec["lam"]), []
        if case["alg"] == "rk4":
            t, h = td[0].clone(), spec["options"]["dt0"]
            while True:
                left = td[1] - t
                last = h > left
                s = torch.where(last, left, torch.full_like(left, h))
                kept.append((X, t, s, None))
                k1 = rhs(t, X)
                k2 = rhs(t + 0.5 * s, X + 0.5 * s * k1)
                k3 = rhs(t + 0.5 * s, X + 0.5 * s * k2)
                k4 = rhs(t + s, X + s * k3)
                X, t = X + s / 6 * (k1 + 2 * k2 + 2 * k3 + k4), t + s
                if bool(last.all()):
                    break
        else:
            _adaptive(rhs, X, td, spec["rtol"], 0.9, low, spec["options"], keep=kept)
        lam, mu = _back(vjp, kept, lam, [torch.zeros_like(lam[0])] * 2, lambda v: v, rhs if case["alg"] == "rk4" else None)
        return {"dx0": lam, "dpar": torch.stack(mu)}
    if f == "uneven":
        # about 35 steps per unit of time in the largest oscillations
        if case["cap"] * (1e-9 / case["tol"]) ** 0.2 > 350.0:
            return None
        n, hits = torch.zeros(case["nt"], dtype=torch.int64, device="cuda"), spec["evcap"]
        log = torch.zeros((hits + 1, 3, case["nt"]), dtype=torch.float64, device="cuda")

        def rhs(t, X):
            return torch.stack((X[1], -par[0] * X[1] + par[1] * torch.cos(par[2] * t) - (X[0] + X[0] ** 3)))

        def event(i, found, X, t):
            row = torch.clamp(n, max=hits)
            entry = torch.stack((t, X[0], X[1]))
            at = row[None, None, :].expand(1, 3, -1)
            log.scatter_(0, at, torch.where(found[None], entry, log.gather(0, at)[0])[None])
            n.add_(found)
            return X, torch.zeros_like(found)
        X, t = _adaptive(rhs, X, td, case["tol"], 0.9, low, spec["options"], ef=lambda X: [X[1]], edir=[0], event=event)
        out = {"ActualState": X, "ActualTime": t, "AcceptedSteps": None, "RejectedSteps": None, "Status": None, "EventCount": None}
        return dict(out, EventLog=log[:hits]) if hits else out
    if f == "double_well":
        B, ndo, nt = 0.3, case["ndo"], case["nt"]
        acc = torch.stack((X[0], X[1], X[0]))
        n = torch.zeros(nt, dtype=torch.int64, device="cuda")
        at = torch.ones(nt, dtype=torch.int64, device="cuda")
        dense = torch.zeros((ndo + 1, 3, nt), dtype=torch.float64, device="cuda")
        dense[0] = torch.cat((td[0][None], X))

        def rhs(t, X):
            return torch.stack((X[1], X[0] - X[0] ** 3 - par[0] * X[1] + B * torch.cos(t)))

        def accepted(X, t, go):
            acc[2] = torch.where(go, torch.maximum(acc[2], X[0]), acc[2])
            row = torch.clamp(at, max=ndo)[None, None, :].expand(1, 3, -1)
            dense.scatter_(0, row, torch.where(go[None], torch.cat((t[None], X)), dense.gather(0, row)[0])[None])
            at.add_(go)
            return torch.zeros_like(go)

        def event(i, found, X, t):
            acc[0] = torch.where(found, torch.maximum(acc[0], X[0]), acc[0])
            if i == 1:
                n.add_(found)
                acc[1] = torch.where(found & (n == 2), X[1], acc[1])
            return X, torch.zeros_like(found)
        X, t = _adaptive(rhs, X, td, case["tol"], 0.9, low, spec["options"], ef=lambda X: [X[1], X[0]], edir=[-1, 0],
                         accepted=accepted, event=event)
        out = {"ActualState": X, "ActualTime": t, "Accessories": acc, "IntegerAccessories": None, "DenseIndex": None,
               "AcceptedSteps": None, "RejectedSteps": None, "Status": None, "EventCount": None}
        return dict(out, DenseTime=dense[:ndo, 0], DenseState=dense[:ndo, 1:]) if ndo else out
    kappa, delta, beta, bounce = (float(v) for v in spec["sPAR"])
    acc, still = torch.stack((X[0], X[0], X[0])), torch.zeros(case["nt"], dtype=torch.int64, device="cuda")

    def rhs(t, X):
        return torch.stack((X[1], -kappa * X[1] - (X[0] + delta) + X[2], beta * (par[0] - X[0] * torch.sqrt(X[2]))))

    def accepted(X, t, go):
        acc[0] = torch.where(go, torch.minimum(acc[0], X[0]), acc[0])
        acc[1] = torch.where(go, torch.maximum(acc[1], X[0]), acc[1])
        rest = (X[0] - acc[2]).abs() < 1e-6
        still.add_(go & rest)
        acc[2] = torch.where(go & ~rest, X[0], acc[2])
        return go & (still == 50)

    def event(i, found, X, t):
        if i == 0:
            return X, torch.ones_like(found)
        return torch.stack((X[0], torch.where(found, -bounce * X[1], X[1]), X[2])), torch.zeros_like(found)
    X, t = _adaptive(rhs, X, td, 1e-10, 0.9, low, spec["options"], ef=lambda X: [X[1], X[0]], edir=[-1, -1],
                     accepted=accepted, event=event)
    return {"ActualState": X, "ActualTime": t, "Accessories": acc, "IntegerAccessories": None, "AcceptedSteps": None,
            "RejectedSteps": None, "Status": None, "EventCount": None, "DenseIndex": None}
