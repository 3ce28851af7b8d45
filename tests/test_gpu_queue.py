"""GPU: how many iterations a solve queues ahead of the host (CLOWNS_POLL)
changes neither the results nor the iteration count, in five launches an
iteration and in single kernels, FP64 and mixed."""
import os

import numpy as np
import pytest

from _systems import box_system

pytestmark = pytest.mark.gpu


def _solve(s, env, maxiters):
    import torch
    from clowns3d import Solver
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    os.environ.update(env)
    try:
        sol = Solver(0)  # reads the switches at creation
    finally:
        for k in env:
            del os.environ[k]
    sol.set_matrix(t(s["AL"].T), t(s["LL"].T), t(s["D"]))
    b = t(s["B"])
    out = []
    for m in maxiters:
        for mixed in (False, True):
            x, i = sol.solve(b, eps=1e-10, maxiter=m, mixed=mixed)
            torch.cuda.synchronize()
            out.append((m, mixed, i["iters"], i["ier"], x.cpu().numpy()))
    sol.close()
    return out


@pytest.mark.parametrize("small", ["0", "1"], ids=["single-kernels", "five-launches"])
@pytest.mark.parametrize("poll", ["0", "1", "2", "16", "64"])
def test_iterations_ahead(poll, small):
    s = box_system(24, 16, 10, seed=3)
    calls = (1, 2, 3, 5000)
    ref = _solve(s, {"CLOWNS_SMALL": small}, calls)
    got = _solve(s, {"CLOWNS_SMALL": small, "CLOWNS_POLL": poll}, calls)
    assert ref[-1][3] == 0 and ref[0][3] == 3000
    for g, r in zip(got, ref):
        assert g[:4] == r[:4]
        assert np.array_equal(g[4], r[4])
