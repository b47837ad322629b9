"""The extended Kalman filter with a caller's prior factor and transition noise factor that are not lower triangular.

A factor L stands for L L^T, whichever square root it is: symmetric, upper, a triangular one times a rotation.
``extended_kalman_filter`` / ``filtsmooth`` (pof/sequential_filtsmooth/filter.py:9-30, __init__.py:5-10) are compared
with the oracle, which multiplies the full matrices, at one state dimension per kernel family (row-per-lane kernels of odd,
even and full rows, and D = 20 of the whole-wavefront ones).  Tolerances: 20 times the oracle's own change when its
inputs move by 1e-15 relative, and at least 1e-12 (normwise; scalars relative).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PROBLEMS = [("logistic", {}, 2), ("fitzhughnagumo", {}, 3), ("rigid_body", {}, 3), ("lorenz96", {"d": 4}, 3),
            ("lorenz96", {"d": 4}, 4)]
# (prior factor, noise factor)
FACTORS = [("full", "lower"), ("lower", "full"), ("full", "full"), ("upper", "lower"), ("lower", "lower"), ("zero", "full")]


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def cov(c):
    return np.einsum("nij,nkj->nik", c, c)


def _prior(form, D, rng):
    A = rng.standard_normal((D, D)) * 0.1
    return {"full": A, "lower": np.tril(A), "upper": np.triu(A), "zero": np.zeros((D, D))}[form]


@pytest.mark.parametrize("name,kw,q", PROBLEMS, ids=[f"{n}-q{q}" for n, _, q in PROBLEMS])
def test_ekf_with_factors_of_any_form(gpu, name, kw, q):
    import torch

    import pof.convenience as pc
    import pof.ivp
    import pof.sequential_filtsmooth as sfs
    from oracle import model as om
    from oracle import problems as op
    from oracle import sequential as oseq
    from pof.transitions import TransitionModel
    from pof.utils import MVNSqrt

    ivp, oivp = getattr(pof.ivp, name)(**kw), getattr(op, name)(**kw)
    ts = np.linspace(0.0, 0.5, 35)
    Ns = len(ts) - 1
    setup = pc.set_up_solver(f=ivp.f, y0=ivp.y0, ts=ts, order=q)
    os_ = om.set_up_solver(oivp, ts, q)
    D = os_.F.shape[0]
    rng = np.random.default_rng(D)
    rot, _ = np.linalg.qr(rng.standard_normal((D, D)))
    for prior, noise in FACTORS:
        print(f"D={D} prior={prior} noise={noise}", flush=True)
        L0 = _prior(prior, D, rng)
        QL = os_.QL @ rot if noise == "full" else os_.QL
        x0 = MVNSqrt(np.asarray(os_.x0.mean), L0)
        dtm = TransitionModel(np.broadcast_to(os_.F, (Ns, D, D)), np.broadcast_to(QL, (Ns, D, D)))
        filt, nll, ssq = sfs.extended_kalman_filter(x0, dtm, setup["om"])
        out, nll2, obj, _ = sfs.filtsmooth(x0, dtm, setup["om"])
        torch.cuda.synchronize()

        def oracle(e=0.0):
            x = om.MVNSqrt(os_.x0.mean, L0 * (1 + e))
            fi, nl, ss = oseq.extended_kalman_filter(x, os_.F, QL * (1 - e), os_, Ns)
            sm, ob = oseq.smoothing(os_.F, QL * (1 - e), fi)
            # sigma_squared whitens with I^T and depends on the factor's column signs beyond one equation
            s = [np.array(ss)] if os_.x0.mean.size == q + 1 else []
            return [fi.mean, cov(fi.chol), np.array(nl), sm.mean, cov(sm.chol), np.array(ob)] + s

        ref = oracle()
        tol = [max(1e-12, 20 * max(rel(a, b) for a in x)) for *x, b in zip(*(oracle(e) for e in (1e-15, -1e-15, 3e-15)), ref)]
        got = [filt.mean.cpu().numpy(), cov(filt.chol.cpu().numpy()), np.array(nll), out.mean.cpu().numpy(),
               cov(out.chol.cpu().numpy()), np.array(obj)] + [np.array(ssq)]
        for k, (a, b, t) in enumerate(zip(got, ref, tol)):
            print(f"  result {k}: {rel(a, b):.1e} of {t:.1e}", flush=True)
            assert rel(a, b) <= t, (prior, noise, k)
        assert nll2 == nll
        # state 0 is the prior as the caller gave it
        np.testing.assert_array_equal(filt.chol.cpu().numpy()[0], L0)
