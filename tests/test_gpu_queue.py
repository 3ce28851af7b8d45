"""GPU: how many iterations a solve queues ahead of the host (CLOWNS_POLL) and
how many it may take (maxiter, up to the largest int) change neither the
results nor the iteration count, in five launches an iteration and in single
kernels, FP64 and mixed."""
import os

import numpy as np
import pytest

from _systems import box_system

pytestmark = pytest.mark.gpu

INT_MAX = 2**31 - 1


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


@pytest.mark.parametrize("small", ["0", "1"], ids=["single-kernels", "five-launches"])
def test_largest_maxiter(small):
    s = box_system(24, 16, 10, seed=3)
    ref, ref32, got, got32 = _solve(s, {"CLOWNS_SMALL": small}, (5000, INT_MAX))
    for g, r in ((got, ref), (got32, ref32)):
        assert g[2:4] == r[2:4] and r[3] == 0
        assert np.array_equal(g[4], r[4])


def test_largest_maxiter_dropin():
    import clowns3d
    s = box_system(12, 10, 8, seed=4)
    out = []
    for m in (5000, INT_MAX):
        AL, LL, D, B = (np.array(s[k], order="F") for k in ("AL", "LL", "D", "B"))
        X = np.zeros(s["N"] + 64)
        r = clowns3d.pcgpme(AL, 6, s["NA"], LL, D, s["N"], 64, B, X, np.array([1e-10, 0.0]), 5.0, m)
        out.append((r, X.copy()))
    print(out[0][0], out[1][0])
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
