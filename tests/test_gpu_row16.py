"""Scan combines with one matrix row per lane (state dimensions D <= 16) against the oracle.

A random linear-Gaussian model with observation noise, so that every factor is well defined, for each state
dimension the kernels exist for, on grids around the places where the work can go wrong: a single element,
levels of odd length, fewer combines than a wavefront's four workers, one more and one less than a full block, stages of
several levels over one block and over many (a block's first prefix comes from the block before), several stages.
Both sides run the same scan in float64.  How far rounding may take two such runs apart is the model's conditioning,
which ranges over six orders of magnitude here (order 5: 3e-10 between the oracle's own parallel and sequential
filters): the tolerance of each result is 20 times the oracle's own change when its inputs move by 1e-15 relative, and
at least 1e-12 (normwise; scalar terms relative).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PAIRS = [(1, 1), (1, 2), (1, 3), (1, 4), (1, 5), (2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3), (3, 4),
         (4, 1), (4, 2), (4, 3)]
STEPS = [1, 2, 3, 4, 5, 7, 8, 9, 31, 33, 130, 515, 1100]


def gram(c):
    return c @ np.swapaxes(c, -1, -2)


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("d,q", PAIRS)
def test_linear_model_against_oracle(gpu, d, q):
    import torch

    import pof.parallel_filtsmooth as pfs
    from oracle import model as om
    from oracle import parallel as opar
    from pof.observations import AffineModel
    from pof.transitions import TransitionModel
    from pof.utils import MVNSqrt

    D = d * (q + 1)
    F, QL = om.preconditioned_discretize(om.IWP(d, q))
    for n in STEPS:
        rng = np.random.default_rng(1000 * D + n)
        H, c = rng.standard_normal((n, d, D)), rng.standard_normal((n, d))
        R = np.tril(rng.standard_normal((n, d, d))) * 0.3 + 0.5 * np.eye(d)
        m0, L0 = rng.standard_normal(D), np.tril(rng.standard_normal((D, D)))
        print(f"D={D} d={d} steps={n}", flush=True)
        t = [torch.as_tensor(x, device="cuda") for x in (H, c, R)]
        out, nll, obj, ssq = pfs.linear_filtsmooth(MVNSqrt(m0, L0), TransitionModel(F, QL), AffineModel(*t))
        filt, _, _, _ = pfs.linear_noiseless_filtering(MVNSqrt(m0, L0), TransitionModel(F, QL), AffineModel(*t))
        torch.cuda.synchronize()
        def oracle(e=0.0):
            x0, mod = om.MVNSqrt(m0, L0 * (1 + e)), om.AffineModel(H * (1 - e), c, R)
            sm, nll, obj, _ = opar.linear_filtsmooth(x0, F, QL, mod)
            fi, _, _, _ = opar.linear_noiseless_filtering(x0, F, QL, mod)
            return [sm.mean, gram(sm.chol), fi.mean, gram(fi.chol), np.array(nll), np.array(obj)]

        ref = oracle()
        tol = [max(1e-12, 20 * max(rel(a, b) for a in x)) for *x, b in zip(*(oracle(e) for e in (1e-15, -1e-15, 3e-15)), ref)]
        got = [out.mean.cpu().numpy(), gram(out.chol.cpu().numpy()), filt.mean.cpu().numpy(),
               gram(filt.chol.cpu().numpy()), np.array(nll), np.array(obj)]
        for a, b, t in zip(got, ref, tol):
            assert rel(a, b) <= t
        # the filtered factors are lower triangular, their strict upper part stored as zeros
        assert not np.triu(filt.chol.cpu().numpy()[1:], 1).any()


@pytest.mark.parametrize("d,q", PAIRS)
def test_sequential_linear_model_against_oracle(gpu, d, q):
    """The sequential filter and smoother, one problem per row: one step, and the sixteen steps between two writes of the
    scalar terms less, exactly and more, with a prior factor that is not triangular.  Tolerances as above."""
    import torch

    import pof.sequential_filtsmooth as sfs
    from oracle import model as om
    from oracle import sequential as oseq
    from pof.observations import AffineModel
    from pof.transitions import TransitionModel
    from pof.utils import MVNSqrt

    D = d * (q + 1)
    F, QL = om.preconditioned_discretize(om.IWP(d, q))
    for n in [1, 2, 15, 16, 17, 33]:
        rng = np.random.default_rng(2000 * D + n)
        H, c = rng.standard_normal((n, d, D)), rng.standard_normal((n, d))
        R = np.tril(rng.standard_normal((n, d, d))) * 0.3 + 0.5 * np.eye(d)
        m0, L0 = rng.standard_normal(D), rng.standard_normal((D, D))
        print(f"D={D} d={d} steps={n}", flush=True)
        t = [torch.as_tensor(x, device="cuda") for x in (H, c, R)]
        out, nll, obj, ssq = sfs.linear_filtsmooth(MVNSqrt(m0, L0), TransitionModel(F, QL), AffineModel(*t))
        filt, _, _ = sfs.linear_noiseless_filter(MVNSqrt(m0, L0), TransitionModel(F, QL), AffineModel(*t))
        torch.cuda.synchronize()

        def oracle(e=0.0):
            x0, mod = om.MVNSqrt(m0, L0 * (1 + e)), om.AffineModel(H * (1 - e), c, R)
            sm, nll, obj, _ = oseq.linear_filtsmooth(x0, F, QL, mod)
            fi, _, _ = oseq.linear_noiseless_filter(x0, F, QL, mod)
            return [sm.mean, gram(sm.chol), fi.mean, gram(fi.chol), np.array(nll), np.array(obj)]

        ref = oracle()
        tol = [max(1e-12, 20 * max(rel(a, b) for a in x)) for *x, b in zip(*(oracle(e) for e in (1e-15, -1e-15, 3e-15)), ref)]
        got = [out.mean.cpu().numpy(), gram(out.chol.cpu().numpy()), filt.mean.cpu().numpy(),
               gram(filt.chol.cpu().numpy()), np.array(nll), np.array(obj)]
        for a, b, t in zip(got, ref, tol):
            assert rel(a, b) <= t


@pytest.mark.parametrize("d,q", [(1, 2), (2, 3)])
def test_one_and_two_workers_per_combine(gpu, d, q):
    """D <= 8: the up-sweep's widest launch with 256 blocks of 16 combines (two workers each) and with 257 (one each), against
    the oracle's parallel filter.  Tolerances as above."""
    import torch

    import pof.parallel_filtsmooth as pfs
    from oracle import model as om
    from oracle import parallel as opar
    from pof.observations import AffineModel
    from pof.transitions import TransitionModel
    from pof.utils import MVNSqrt

    D = d * (q + 1)
    F, QL = om.preconditioned_discretize(om.IWP(d, q))
    for n in (8193, 8194):
        rng = np.random.default_rng(3000 * D + n)
        H, c = rng.standard_normal((n, d, D)), rng.standard_normal((n, d))
        R = np.tril(rng.standard_normal((n, d, d))) * 0.3 + 0.5 * np.eye(d)
        m0, L0 = rng.standard_normal(D), np.tril(rng.standard_normal((D, D)))
        print(f"D={D} d={d} steps={n}", flush=True)
        t = [torch.as_tensor(x, device="cuda") for x in (H, c, R)]
        filt, _, _, _ = pfs.linear_noiseless_filtering(MVNSqrt(m0, L0), TransitionModel(F, QL), AffineModel(*t))
        torch.cuda.synchronize()

        def oracle(e=0.0):
            fi, _, _, _ = opar.linear_noiseless_filtering(om.MVNSqrt(m0, L0 * (1 + e)), F, QL, om.AffineModel(H * (1 - e), c, R))
            return [fi.mean, gram(fi.chol)]

        ref = oracle()
        tol = [max(1e-12, 20 * max(rel(a, b) for a in x)) for *x, b in zip(*(oracle(e) for e in (1e-15, -1e-15, 3e-15)), ref)]
        for a, b, t in zip([filt.mean.cpu().numpy(), gram(filt.chol.cpu().numpy())], ref, tol):
            assert rel(a, b) <= t
