"""Timed cases of the solver: the calls a user of this package makes, over the range of sizes it serves.

A case names one public call and its sizes.  ``prepare`` builds what a program holds before the call (vector field,
initial value, grid, or a linear model on the GPU), ``run`` is one pass, ``exact`` is what it returns, from a plain
NumPy square-root filter and smoother that steps through time (the parallel scan solves the same linear problem in
every iteration).

What ``run`` returns.  A posterior of this method is a mean and a covariance; the library hands the covariance out as a
factor L, and programs use ``L L^T`` (a band, a marginal).  The columns of L carry the signs of Householder pivots
which, with noiseless observations, are rounding noise, so the product and not the factor is what the inputs determine.
The factor is also scaled by the calibration ``sigma_squared``, a mean of whitened residuals that depends on those same
signs and, on fine grids, is a sum of cancelled digits (it moves by up to per cents when ``y0`` moves in its last bit).
The covariance therefore comes back per unit of it, except in the cases marked ``calibrated``, coarse grids on which it is
determined to many digits: they return it and the calibrated covariance.  The log likelihood comes back where it is
determined (solves that run to convergence, the single-pass smoother, the linear model); after a few iterations on a fine
grid it is a sum over residuals that have cancelled.

The spans and starts are those on which the first iterates are determined as well: linearised at a constant trajectory,
a chaotic system amplifies the last bit of its inputs by the exponential of the span.
"""
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "parallel-in-time-ode-filters_amd"))

import pof.batch  # noqa: E402
import pof.ivp  # noqa: E402
import pof.parallel_filtsmooth  # noqa: E402
import pof.solver  # noqa: E402
from pof.observations import AffineModel  # noqa: E402
from pof.transitions import IWP, TransitionModel, preconditioned_discretize  # noqa: E402
from pof.utils import MVNSqrt  # noqa: E402

MAXITERS = 200


# ------------------------------------------------------------------------------------------------------------- cases
def _solve(name, problem, steps, order, tmax, iters, init="constant", d=0, calibrated=False):
    c = {"call": "solve", "problem": problem, "steps": steps, "order": order, "tmax": tmax, "iters": iters,
         "init": init, "d": d, "calibrated": calibrated}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: a short grid, the default initial trajectory, run to convergence
        _solve("logistic 63", "logistic", 63, 2, 10.0, 0, "prior", calibrated=True),
        # an oscillator on a coarse grid, run to convergence (order 3: D = 8)
        _solve("fitzhughnagumo 299", "fitzhughnagumo", 299, 3, 20.0, 0),
        # an ordinary system on an ordinary grid, to convergence (D = 12)
        _solve("rigid_body 1000", "rigid_body", 1000, 3, 20.0, 0),
        # the benchmark's grid and state dimension (D = 12, 65536 steps), ten iterations
        _solve("rigid_body 65536", "rigid_body", 65536, 3, 20.0, 10),
        # the largest order of the batched workload (D = 15), ragged length
        _solve("lorenz63 q4 10007", "lorenz63", 10007, 4, 0.25, 5),
        # a small state on the longest grid (D = 4): levels of the scan bound by launches and latency
        _solve("logistic 65536", "logistic", 65536, 3, 10.0, 10),
        # two equations, low order (D = 6), the default initial trajectory, odd length
        _solve("fhn_classic 20001", "fhn_classic", 20001, 2, 5.0, 6, "prior"),
        # many small IVPs of mixed dimension, order and length solved together
        {"name": "batch 96", "call": "batch", "count": 96, "min_steps": 256, "max_steps": 8192, "iters": 5},
        # a high-dimensional system (D = 128) on the large-state engine
        _solve("lorenz96 d32 8192", "lorenz96", 8192, 3, 0.2, 2, d=32),
        # the same engine where each level is small (D = 24)
        _solve("lorenz96 d8 511", "lorenz96", 511, 2, 0.2, 3, d=8),
        # the sequential extended Kalman smoother of the README figure
        {"name": "eks fitzhughnagumo 299", "call": "eks", "problem": "fitzhughnagumo", "steps": 299, "order": 3,
         "tmax": 100.0, "calibrated": True},
        # one linear smoothing problem with noisy observations on device tensors, full states (D = 12)
        {"name": "filtsmooth 16384", "call": "filtsmooth", "d": 3, "order": 3, "steps": 16384},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """One more case: the same calls, sizes spread over the logarithm of their ranges."""
    kind = rng.choice(["solve", "solve", "solve", "solve", "converge", "batch", "large", "eks", "filtsmooth"])
    if kind == "solve":
        problem, tmax = rng.choice([("logistic", 10.0), ("fhn_classic", 5.0), ("rigid_body", 20.0),
                                    ("lorenz63", 0.25), ("lorenz96", 0.2)])
        order = rng.randint(1, 3 if problem == "lorenz96" else 4)
        return _solve(None, problem, _log(rng, 64, 65536), order, tmax, rng.randint(4, 8),
                      rng.choice(["constant", "prior"]) if problem in ("logistic", "fhn_classic") else "constant",
                      4 if problem == "lorenz96" else 0)
    if kind == "converge":
        problem, tmax = rng.choice([("logistic", 10.0), ("rigid_body", 20.0)])
        return _solve(None, problem, _log(rng, 64, 4096), rng.randint(2, 3), tmax, 0)
    if kind == "batch":
        lo = _log(rng, 64, 512)
        return {"call": "batch", "count": _log(rng, 8, 96), "min_steps": lo, "max_steps": _log(rng, 1024, 8192),
                "iters": rng.randint(4, 5)}
    if kind == "large":
        d = rng.choice([6, 8, 16, 32])
        return _solve(None, "lorenz96", _log(rng, 64, 4096), rng.randint(2, 3) if d < 32 else 3, 0.2, 2, d=d)
    if kind == "eks":
        problem, tmax = rng.choice([("fitzhughnagumo", 50.0), ("logistic", 10.0), ("rigid_body", 10.0)])
        return {"call": "eks", "problem": problem, "steps": _log(rng, 64, 2048), "order": rng.randint(2, 4),
                "tmax": tmax, "calibrated": False}
    return {"call": "filtsmooth", "d": rng.randint(1, 3), "order": rng.randint(1, 4), "steps": _log(rng, 64, 32768)}


# ------------------------------------------------------------------------------------------------------------ inputs
def _ivp(problem, rng, d=0):
    """A problem near the package's default one: parameters and initial value moved by some per cent."""
    s = 1.0 + 0.02 * rng.standard_normal(8)
    if problem == "logistic":
        return pof.ivp.logistic(r=float(s[0]), K=1.0, y0=[0.01 * s[1]])
    if problem == "fitzhughnagumo":
        return pof.ivp.fitzhughnagumo(y0=[s[0], s[1]])
    if problem == "fhn_classic":
        return pof.ivp.fhn_classic(a=0.2 * s[0], b=0.2 * s[1], c=3.0 * s[2], y0=[-s[3], s[4]])
    if problem == "rigid_body":
        return pof.ivp.rigid_body(y0=[s[0], 0.1 * (s[1] - 1.0), 0.9 * s[2]])
    if problem == "lorenz63":
        return pof.ivp.lorenz63(rho=28.0 * s[0], y0=[s[1], s[2], s[3]])
    if problem == "lorenz96":
        return pof.ivp.lorenz96(d=d, y0=8.0 + 0.1 * rng.standard_normal(d))
    raise ValueError(problem)


def _mixed(case, rng):
    """The members of a batch: problem, order and length of each."""
    out = []
    for _ in range(case["count"]):
        problem, tmax = [("logistic", 10.0), ("fhn_classic", 5.0), ("lorenz63", 0.25)][int(rng.integers(3))]
        order = int(rng.integers(1, 5))
        steps = int(round(math.exp(rng.uniform(math.log(case["min_steps"]), math.log(case["max_steps"])))))
        out.append((_ivp(problem, rng), np.linspace(0.0, tmax, steps + 1), order))
    return out


def _linear_model(case, rng):
    """A linear-Gaussian model: IWP transition, random noisy observations of every state."""
    d, D, n = case["d"], case["d"] * (case["order"] + 1), case["steps"]
    H = rng.standard_normal((n, d, D))
    c = rng.standard_normal((n, d))
    R = np.tril(rng.standard_normal((n, d, d))) * 0.3 + 0.5 * np.eye(d)
    return rng.standard_normal(D), np.tril(rng.standard_normal((D, D))), H, c, R


def prepare(case, seed):
    # the sizes of a batch come from the case alone, so that every seed has the same work
    rng = np.random.default_rng(seed)
    if case["call"] == "batch":
        sizes = np.random.default_rng(case["count"] * 100003 + case["max_steps"])
        members = _mixed(case, sizes)
        probs = []
        for ivp, ts, order in members:
            y0 = ivp.y0 * (1.0 + 0.02 * rng.standard_normal(ivp.y0.shape))
            probs.append(pof.batch.Problem(ivp.f, y0, ts, order, "constant"))
        return {"case": case, "problems": probs}
    if case["call"] == "filtsmooth":
        m0, L0, H, c, R = _linear_model(case, rng)
        F, QL = preconditioned_discretize(IWP(case["d"], case["order"]))
        dev = torch.device("cuda", torch.cuda.current_device())
        obs = AffineModel(*(torch.as_tensor(x, device=dev) for x in (H, c, R)))
        return {"case": case, "x0": MVNSqrt(m0, L0), "model": TransitionModel(F, QL), "obs": obs}
    ivp = _ivp(case["problem"], rng, case.get("d", 0))
    return {"case": case, "f": ivp.f, "y0": ivp.y0, "ts": np.linspace(0.0, case["tmax"], case["steps"] + 1)}


# --------------------------------------------------------------------------------------------------------------- run
def _posterior(ys, info, power, calibrated=False):
    """Mean and covariance of a solution whose factor is scaled by ``sigma_squared ** (power / 2)``."""
    cov = ys.chol @ ys.chol.transpose(-1, -2)
    if calibrated:
        return {"mean": ys.mean, "cov": cov, "sigma_squared": info["sigma_squared"]}
    return {"mean": ys.mean, "cov": cov / info["sigma_squared"] ** power}


def run(state):
    case = state["case"]
    if case["call"] == "batch":
        res = pof.batch.solve_batch(state["problems"], fixed_iters=case["iters"])
        outs = [_posterior(ys, info, 2) for ys, info in res]
        return {"mean": torch.cat([o["mean"].reshape(-1) for o in outs]),
                "cov": torch.cat([o["cov"].reshape(-1) for o in outs])}
    if case["call"] == "filtsmooth":
        out, nll, obj, _ = pof.parallel_filtsmooth.linear_filtsmooth(state["x0"], state["model"], state["obs"])
        return {"mean": out.mean, "cov": out.chol @ out.chol.transpose(-1, -2), "nll": nll, "obj": obj}
    if case["call"] == "eks":
        ys, info = pof.solver.sequential_eks_solve(f=state["f"], y0=state["y0"], ts=state["ts"], order=case["order"])
        return dict(_posterior(ys, info, 1, case["calibrated"]), nll=info["nll"])
    ys, info = pof.solver.solve(f=state["f"], y0=state["y0"], ts=state["ts"], order=case["order"], init=case["init"],
                                fixed_iters=case["iters"] or None, maxiters=MAXITERS)
    out = _posterior(ys, info, 2, case["calibrated"])
    if not case["iters"]:
        out["iterations"] = int(info["iterations"])
        out["nll"] = info["nll"]
    return out


# -------------------------------------------------------------------------------------------------------------- work
def _iteration_flops(n, D, d):
    """One iteration at the counts of the method's formulas: element, two scans of combines, smoother element."""
    return n * (74.3 * D**3 + (4.0 / 3.0) * (D + d) ** 3)


_DIMS = {"logistic": 1, "fitzhughnagumo": 2, "fhn_classic": 2, "rigid_body": 3, "lorenz63": 3}
_TYPICAL_ITERS = {"logistic": 10, "fitzhughnagumo": 48, "rigid_body": 10}


def work(case):
    if case["call"] == "batch":
        sizes = np.random.default_rng(case["count"] * 100003 + case["max_steps"])
        total = {"bytes": 0.0, "flops": 0.0}
        for ivp, ts, order in _mixed(case, sizes):
            n, d = len(ts) - 1, len(ivp.y0)
            D = d * (order + 1)
            total["flops"] += case["iters"] * _iteration_flops(n, D, d)
            total["bytes"] += 8.0 * (n + 1) * (1 + d + d * D)
        return total
    n = case["steps"]
    if case["call"] == "filtsmooth":
        d, D = case["d"], case["d"] * (case["order"] + 1)
        return {"bytes": 8.0 * n * (d * D + d + d * d + D + D * D), "flops": _iteration_flops(n, D, d)}
    d = case.get("d") or _DIMS[case["problem"]]
    D = d * (case["order"] + 1)
    io = 8.0 * (n + 1) * (1 + d + d * D)
    if case["call"] == "eks":
        # predict, update and smooth of every step: QRs of D x 2D, (d + D) x (D + d), 2D x 2D and D x 2D
        return {"bytes": io, "flops": n * (25.0 * D**3 + (4.0 / 3.0) * (D + d) ** 3)}
    iters = case["iters"] or _TYPICAL_ITERS[case["problem"]]
    return {"bytes": io, "flops": iters * _iteration_flops(n, D, d)}


# ------------------------------------------------------------------------------------- the same in plain NumPy, 64 bit
def _field(name, p):
    """f(y) and its Jacobian at one point."""
    if name == "logistic":
        return lambda y: np.array([p[0] * y[0] * (1 - y[0] / p[1])]), lambda y: np.array([[p[0] * (1 - 2 * y[0] / p[1])]])
    if name == "fitzhughnagumo":
        return (lambda y: np.array([y[0] - y[0] ** 3 / 3 - y[1] + p[3], p[2] * (y[0] + p[0] - p[1] * y[1])]),
                lambda y: np.array([[1 - y[0] ** 2, -1.0], [p[2], -p[2] * p[1]]]))
    if name == "fhn_classic":
        return (lambda y: np.array([p[2] * (y[0] - y[0] ** 3 / 3 + y[1]), -(y[0] - p[0] + p[1] * y[1]) / p[2]]),
                lambda y: np.array([[p[2] * (1 - y[0] ** 2), p[2]], [-1 / p[2], -p[1] / p[2]]]))
    if name == "rigid_body":
        return (lambda y: np.array([p[0] * y[1] * y[2], p[1] * y[0] * y[2], p[2] * y[0] * y[1]]),
                lambda y: np.array([[0, p[0] * y[2], p[0] * y[1]], [p[1] * y[2], 0, p[1] * y[0]],
                                    [p[2] * y[1], p[2] * y[0], 0]]))
    if name == "lorenz63":
        return (lambda y: np.array([p[0] * (y[1] - y[0]), y[0] * (p[1] - y[2]) - y[1], y[0] * y[1] - p[2] * y[2]]),
                lambda y: np.array([[-p[0], p[0], 0], [p[1] - y[2], -1, -y[0]], [y[1], y[0], -p[2]]]))

    def f96(y):
        return (np.roll(y, -1) - np.roll(y, 2)) * np.roll(y, 1) - y + p[0]

    def j96(y):
        d = len(y)
        J = -np.eye(d)
        for i in range(d):
            J[i, (i + 1) % d] += y[i - 1]
            J[i, i - 2] -= y[i - 1]
            J[i, i - 1] += y[(i + 1) % d] - y[i - 2]
        return J

    return f96, j96


def _derivatives(name, p, y0, q):
    """y^(k)(0), k = 0..q, of a quadratic or cubic field from its Taylor coefficients."""
    d = len(y0)
    a = np.zeros((q + 1, d))
    a[0] = y0

    def mul(u, v, k):
        return sum(u[j] * v[k - j] for j in range(k + 1))

    for k in range(q):
        y = [a[: k + 1, i] for i in range(d)]
        one = 1.0 if k == 0 else 0.0
        if name == "logistic":
            c = [p[0] * (y[0][k] - mul(y[0], y[0], k) / p[1])]
        elif name in ("fitzhughnagumo", "fhn_classic"):
            sq = [mul(y[0], y[0], j) for j in range(k + 1)]
            cube = mul(sq, y[0], k)
            if name == "fhn_classic":
                c = [p[2] * (y[0][k] - cube / 3 + y[1][k]), -(y[0][k] - p[0] * one + p[1] * y[1][k]) / p[2]]
            else:
                c = [y[0][k] - cube / 3 - y[1][k] + p[3] * one, p[2] * (y[0][k] + p[0] * one - p[1] * y[1][k])]
        elif name == "rigid_body":
            c = [p[0] * mul(y[1], y[2], k), p[1] * mul(y[0], y[2], k), p[2] * mul(y[0], y[1], k)]
        elif name == "lorenz63":
            c = [p[0] * (y[1][k] - y[0][k]), p[1] * y[0][k] - mul(y[0], y[2], k) - y[1][k],
                 mul(y[0], y[1], k) - p[2] * y[2][k]]
        else:
            c = [mul(y[(i + 1) % d], y[i - 1], k) - mul(y[i - 2], y[i - 1], k) - y[i][k] + p[0] * one
                 for i in range(d)]
        a[k + 1] = np.array(c) / (k + 1)
    return a * np.array([math.factorial(k) for k in range(q + 1)], float)[:, None]


def _tria(M):
    return np.linalg.qr(M.T, mode="r").T


def _iwp(d, q):
    """Preconditioned integrated Wiener process: transition and noise factor."""
    n = q + 1
    A = np.array([[math.comb(q - i, j - i) if j >= i else 0 for j in range(n)] for i in range(n)], float)
    Q = np.array([[1.0 / (2 * q + 1 - i - j) for j in range(n)] for i in range(n)])
    return np.kron(np.eye(d), A), np.kron(np.eye(d), np.linalg.cholesky(Q))


def _filter_smoother(F, QL, m, L, observe, n):
    """Square-root Kalman filter and RTS smoother; ``observe(k, mp)`` gives (H, c, R) of step k.
    Returns the means, the factors, -log likelihood, and the whitened sum of the observations."""
    D = len(m)
    fm, fL, nll, white = [m], [L], 0.0, 0.0
    for k in range(n):
        mp, Lp = F @ m, _tria(np.hstack([F @ L, QL]))
        H, c, R = observe(k, mp)
        d = len(c)
        S = _tria(np.block([[H @ Lp, R], [Lp, np.zeros((D, d))]]))
        z = np.linalg.solve(S[:d, :d], -(H @ mp + c))
        m, L = mp + S[d:, :d] @ z, S[d:, d:]
        nll += 0.5 * z @ z + np.log(np.abs(np.diag(S)[:d])).sum() + 0.5 * d * math.log(2 * math.pi)
        white += z @ z
        fm.append(m)
        fL.append(L)
    sm, sL = [m], [L]
    for k in range(n - 1, -1, -1):
        T = _tria(np.block([[F @ fL[k], QL], [fL[k], np.zeros((D, D))]]))
        E = np.linalg.solve(T[:D, :D].T, T[D:, :D].T).T
        sm.append(fm[k] + E @ (sm[-1] - F @ fm[k]))
        sL.append(_tria(np.hstack([T[D:, D:], E @ sL[-1]])))
    return np.array(sm[::-1]), np.array(sL[::-1]), nll, white


def _exact_ode(ivp, name, ts, q, init, iters, eks=False, calibrated=False):
    p, y0 = ivp.f.params, np.asarray(ivp.y0, float)
    d, n = len(y0), len(ts) - 1
    D, h = d * (q + 1), ts[1] - ts[0]
    f, jac = _field(name, p)
    F, QL = _iwp(d, q)
    e = np.arange(q, -1, -1) + 0.5
    fact = np.array([math.factorial(q - i) for i in range(q + 1)], float)
    P1 = h**e / fact
    P = np.tile(P1, d)
    der = _derivatives(name, p, y0, q)
    i0, i1 = np.arange(d) * (q + 1), np.arange(d) * (q + 1) + 1
    x0 = der.T.reshape(-1) / P
    zero = np.zeros((d, d))

    def ek1(m):
        y = P[i0] * m[i0]
        J = jac(y)
        H = np.zeros((d, D))
        H[np.arange(d), i1] = P[i1]
        H[:, i0] -= J * P[i0]
        return H, J @ y - f(y), zero

    if init == "prior":
        # the Taylor polynomial at every time point, not preconditioned (the solver's default start)
        T = np.array([[[t ** (j - i) / math.factorial(j - i) if j >= i else 0.0 for j in range(q + 1)]
                       for i in range(q + 1)] for t in ts])
        lin = np.einsum("tij,jd->tdi", T, der).reshape(n + 1, D)
    else:
        row = np.zeros((d, q + 1))
        row[:, 0], row[:, 1] = y0, f(y0)
        lin = np.tile(row.reshape(-1) / P, (n + 1, 1))
    obj, k = 0.0, 0
    while True:
        m, L, nll, white = _filter_smoother(F, QL, x0, np.zeros((D, D)),
                                            (lambda j, mp: ek1(mp)) if eks else (lambda j, mp: ek1(lin[j + 1])), n)
        k += 1
        r = np.linalg.solve(QL, (m[:-1] - m[1:] @ F.T).T)
        old, obj = obj, float((r * r).sum())
        close = bool((np.abs(lin - m) <= 1e-8 + 1e-13 * np.abs(m)).all())
        lin = m
        if eks or (iters and k >= iters):
            break
        if not iters and (abs(old - obj) <= 1e-9 + 1e-6 * abs(obj) or close or k > MAXITERS):
            break
    C = P[i0][:, None] * L[:, i0]
    out = {"mean": m[:, i0] * P[i0], "cov": C @ C.transpose(0, 2, 1)}
    if eks or not iters:
        out["nll"] = -nll if eks else nll
    if calibrated and d == 1:
        out["sigma_squared"] = white / n
        out["cov"] = out["cov"] * out["sigma_squared"] ** (1 if eks else 2)
    elif calibrated:
        # a system's sigma_squared depends on the signs of the factors, which no other factorisation shares
        out["sigma_squared"] = out["cov"] = None
    if not iters and not eks:
        out["iterations"] = k
    return out


def exact(case, seed):
    rng = np.random.default_rng(seed)
    if case["call"] == "batch":
        if case["iters"] * sum(len(p.ts) for p in prepare(case, seed)["problems"]) > 30_000:
            return None
        names = {1: "logistic", 2: "fhn_classic", 3: "lorenz63"}
        outs = [_exact_ode(pof.ivp.IVP(p.f, 0.0, p.ts[-1], p.y0), names[len(p.y0)], p.ts, p.order, p.init, case["iters"])
                for p in prepare(case, seed)["problems"]]
        return {"mean": np.concatenate([o["mean"].reshape(-1) for o in outs]),
                "cov": np.concatenate([o["cov"].reshape(-1) for o in outs])}
    if case["call"] == "filtsmooth":
        if case["steps"] > 40_000:
            return None
        m0, L0, H, c, R = _linear_model(case, rng)
        F, QL = _iwp(case["d"], case["order"])
        m, L, nll, _ = _filter_smoother(F, QL, m0, L0, lambda k, mp: (H[k], c[k], R[k]), case["steps"])
        r = np.linalg.solve(QL, (m[:-1] - m[1:] @ F.T).T)
        return {"mean": m, "cov": L @ L.transpose(0, 2, 1), "nll": nll, "obj": float((r * r).sum())}
    ivp = _ivp(case["problem"], rng, case.get("d", 0))
    D = len(ivp.y0) * (case["order"] + 1)
    iters = case.get("iters", 1) or _TYPICAL_ITERS[case["problem"]] + 10
    if case["steps"] * iters > (40_000 if D <= 16 else 4_000 if D <= 32 else 300):
        return None
    ts = np.linspace(0.0, case["tmax"], case["steps"] + 1)
    return _exact_ode(ivp, case["problem"], ts, case["order"], case.get("init", "constant"), case.get("iters", 1),
                      case["call"] == "eks", case["calibrated"])
