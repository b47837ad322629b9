"""A call on a stream that the program is capturing into a HIP graph is refused, and leaves the capture as it is."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_calls_are_refused_while_their_stream_is_captured(gpu):
    import torch

    import pof.ivp
    import pof.parallel_filtsmooth as pfs
    import pof.solver
    from oracle import model as om
    from pof import _lib
    from pof.observations import AffineModel
    from pof.transitions import TransitionModel
    from pof.utils import MVNSqrt

    ivp = pof.ivp.rigid_body()
    ts = np.linspace(0.0, 1.0, 65)
    F, QL = om.preconditioned_discretize(om.IWP(3, 3))
    rng = np.random.default_rng(3)
    dom = AffineModel(torch.as_tensor(rng.standard_normal((64, 3, 12)), device="cuda"),
                      torch.as_tensor(rng.standard_normal((64, 3)), device="cuda"), None)
    x0 = MVNSqrt(rng.standard_normal(12), np.eye(12))

    def solve():
        return pof.solver.solve(f=ivp.f, y0=ivp.y0, ts=ts, order=3, init="constant", fixed_iters=3)[0]

    def smooth():
        return pfs.linear_filtsmooth(x0, TransitionModel(F, QL), dom)[0]

    want = [solve(), smooth()]
    x = torch.arange(4.0, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = x + 1.0
        for call in (solve, smooth):
            with pytest.raises(_lib.PofError, match="captured"):
                call()
        z = y * 2.0
    for k in range(3):
        x.fill_(float(k))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, torch.full((4,), 2.0 * (k + 1.0), device="cuda"))
        got = [solve(), smooth()]
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a.mean, b.mean) and torch.equal(a.chol, b.chol)
