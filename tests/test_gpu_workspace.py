"""Workspaces that a call leaves for the next one: calls of many shapes in turn against calls on a context of their own.

A context serves one thread, so a call made on a new thread finds no workspace.  The same call has to give the same
bits either way, whatever ran before it: smaller and larger grids, other state dimensions, the sequential form, the
smoother alone and the extended filter, a call that failed.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _calls():
    rng = np.random.default_rng(7)
    out = []
    for d, q, n, seq, noise in [(3, 3, 300, False, True), (3, 3, 40, False, False), (3, 3, 41, True, True), (1, 2, 700, False, True),
                                (2, 1, 64, True, False), (2, 4, 90, False, True), (4, 2, 33, False, True), (3, 3, 900, False, True)]:
        D = d * (q + 1)
        R = np.tril(rng.standard_normal((n, d, d))) * 0.3 + 0.5 * np.eye(d) if noise else None
        out.append((d, q, seq, rng.standard_normal((n, d, D)), rng.standard_normal((n, d)), R, rng.standard_normal(D),
                    np.tril(rng.standard_normal((D, D)))))
    return out


def _run(call):
    import torch

    import pof.parallel_filtsmooth as pfs
    import pof.sequential_filtsmooth as sfs
    from oracle import model as om
    from pof.observations import AffineModel
    from pof.transitions import TransitionModel
    from pof.utils import MVNSqrt

    d, q, seq, H, c, R, m0, L0 = call
    F, QL = om.preconditioned_discretize(om.IWP(d, q))
    t = [None if x is None else torch.as_tensor(x, device="cuda") for x in (H, c, R)]
    fs = sfs if seq else pfs
    out, nll, obj, ssq = fs.linear_filtsmooth(MVNSqrt(m0, L0), TransitionModel(F, QL), AffineModel(*t))
    torch.cuda.synchronize()
    return [out.mean.cpu().numpy(), out.chol.cpu().numpy(), np.array([nll, obj, ssq])]


def _alone(call):
    from pof import _lib

    res = []

    def work():
        for key in [k for k in _lib._ctx if k[0] == threading.get_ident()]:
            del _lib._ctx[key]  # an ended thread's, whose identity this one has
        res.append(_run(call))

    t = threading.Thread(target=work)
    t.start()
    t.join()
    return res[0]


def test_calls_in_turn_equal_calls_alone(gpu):
    from pof import _lib
    import pof.parallel_filtsmooth as pfs
    from pof.transitions import TransitionModel
    from pof.observations import AffineModel
    from pof.utils import MVNSqrt

    calls = _calls()
    want = [_alone(c) for c in calls]
    order = [0, 1, 2, 0, 3, 4, 5, 6, 7, 1, 0, 5, 2, 7, 3]
    for k, i in enumerate(order):
        print(f"call {i} (d={calls[i][0]} q={calls[i][1]} steps={len(calls[i][4])})", flush=True)
        if k == 6:  # a refused call in between
            with pytest.raises((ValueError, NotImplementedError, _lib.PofError)):
                pfs.linear_filtsmooth(MVNSqrt(np.zeros(7), np.eye(7)), TransitionModel(np.eye(7), np.eye(7)),
                                      AffineModel(np.zeros((3, 1, 7)), np.zeros((3, 1)), None))
        for a, b in zip(_run(calls[i]), want[i]):
            np.testing.assert_array_equal(a, b)


def test_threads_have_a_workspace_each(gpu):
    calls = _calls()
    want = [_alone(c) for c in calls]
    bad = []

    def work(first):
        for i in range(first, first + 6):
            k = i % len(calls)
            for a, b in zip(_run(calls[k]), want[k]):
                if not np.array_equal(a, b):
                    bad.append(k)

    ts = [threading.Thread(target=work, args=(f,)) for f in (0, 3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def _filters_and_smoothers():
    """Calls that share workspaces of one (D, d): extended filters of other fields, parameters, priors and transition models,
    smoothers over given filtered states, both forms, and linear models in between."""
    import torch

    import pof.convenience as pc
    import pof.ivp
    import pof.parallel_filtsmooth as pfs
    import pof.sequential_filtsmooth as sfs
    from pof.observations import AffineModel
    from pof.transitions import TransitionModel
    from pof.utils import MVNSqrt

    def arrays(*xs):
        torch.cuda.synchronize()
        return [x.cpu().numpy() if hasattr(x, "cpu") else np.array(x) for x in xs]

    out = []
    for q, ivps in [(3, [pof.ivp.fitzhughnagumo(), pof.ivp.vanderpol(), pof.ivp.fhn_classic(a=0.3, b=0.1, c=2.0)]),
                    (3, [pof.ivp.rigid_body(), pof.ivp.lorenz63(), pof.ivp.rigid_body(y0=[0.9, 0.1, 1.1])])]:
        for k, (ivp, n) in enumerate(zip(ivps, (60, 23, 41))):
            s = pc.set_up_solver(f=ivp.f, y0=ivp.y0, ts=np.linspace(0.0, 0.5, n + 1), order=q)
            F, QL = np.asarray(s["dtm"].F)[0], np.asarray(s["dtm"].QL)[0]
            D = F.shape[0]
            d = D // (q + 1)
            rng = np.random.default_rng(100 * D + k)
            rot, _ = np.linalg.qr(rng.standard_normal((D, D)))

            def model(QL_, F_=F, n_=n, D_=D):
                return TransitionModel(np.broadcast_to(F_, (n_, D_, D_)), np.broadcast_to(QL_, (n_, D_, D_)))

            def ekf(x0=s["x0"], dtm=s["dtm"], om=s["om"]):
                f, nll, ssq = sfs.extended_kalman_filter(x0, dtm, om)
                return arrays(f.mean, f.chol, nll, ssq)

            x1 = MVNSqrt(np.asarray(s["x0"].mean), 0.1 * rng.standard_normal((D, D)))
            fm = torch.as_tensor(rng.standard_normal((n + 1, D)), device="cuda")
            fL = torch.as_tensor(rng.standard_normal((n + 1, D, D)), device="cuda")

            def smooth(fn, dtm, m=fm, L=fL):
                o, obj = fn(dtm, MVNSqrt(m, L))
                return arrays(o.mean, o.chol, obj)

            H, c = rng.standard_normal((n, d, D)), rng.standard_normal((n, d))

            def linear(fs, dtm, H_=H, c_=c, x0=x1):
                t = [torch.as_tensor(x, device="cuda") for x in (H_, c_)]
                o, nll, obj, ssq = fs.linear_filtsmooth(x0, dtm, AffineModel(*t, None))
                return arrays(o.mean, o.chol, nll, obj, ssq)

            out += [ekf, lambda e=ekf, x=x1, m=model(QL @ rot): e(x0=x, dtm=m), lambda f=smooth, m=model(QL): f(pfs.smoothing, m),
                    lambda f=linear, m=model(1.5 * QL): f(pfs, m), lambda f=smooth, m=model(QL @ rot): f(sfs.smoothing, m),
                    lambda f=linear, m=model(QL @ rot): f(sfs, m)]
    return out


def test_filters_and_smoothers_in_turn_equal_calls_alone(gpu):
    """As above for every call that takes a kept workspace: what one leaves in it (model, field, parameters, flags) is not
    what the next one uses."""
    from pof import _lib

    calls = _filters_and_smoothers()

    def alone(call):
        res = []

        def work():
            for key in [k for k in _lib._ctx if k[0] == threading.get_ident()]:
                del _lib._ctx[key]
            res.append(call())

        t = threading.Thread(target=work)
        t.start()
        t.join()
        return res[0]

    want = [alone(c) for c in calls]
    order = np.random.default_rng(5).permutation(np.repeat(np.arange(len(calls)), 2))
    for i in order:
        print(f"call {i}", flush=True)
        for a, b in zip(calls[i](), want[i]):
            np.testing.assert_array_equal(a, b)


def test_trim_gives_the_memory_back(gpu):
    import torch

    from pof import _lib

    _lib.context()
    _lib.trim()
    free = torch.cuda.mem_get_info()[0]
    call = _calls()[0]
    first = _run(call)
    assert torch.cuda.mem_get_info()[0] <= free
    assert _lib.trim() > 0
    assert _lib.trim() == 0
    for a, b in zip(_run(call), first):
        np.testing.assert_array_equal(a, b)
