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


@pytest.mark.parametrize("small", ["0", "1"], ids=["single-kernels", "five-launches"])
def test_solve_after_one_left_by_an_error(small):
    """A solve that an error ends (here one that the host program left behind)
    waits for the kernels it had queued: while the GPU is still busy with other
    work, their word that a zero right-hand side is done must not end the next
    solve."""
    import ctypes
    import torch
    from clowns3d import ClownsError, Solver
    s = box_system(24, 16, 10, seed=3)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    os.environ["CLOWNS_SMALL"] = small
    try:
        sol = Solver(0)  # reads the switch at creation
    finally:
        del os.environ["CLOWNS_SMALL"]
    sol.set_matrix(t(s["AL"].T), t(s["LL"].T), t(s["D"]))
    b = t(s["B"])
    zero, x0, x = torch.zeros_like(b), torch.zeros_like(b), torch.zeros_like(b)  # torch itself stops at such an error
    ref, iref = sol.solve(b, eps=1e-10)
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    a = torch.ones((8192, 8192), device="cuda:0")
    torch.cuda.synchronize()
    for _ in range(20):
        a @ a
    assert hip.hipSetDevice(9999) != 0
    with pytest.raises(ClownsError) as e:
        sol.solve(zero, x0, eps=1e-10)
    assert e.value.code == 4004
    x, i = sol.solve(b, x, eps=1e-10)
    torch.cuda.synchronize()
    assert (i["iters"], i["ier"]) == (iref["iters"], 0) and torch.equal(x, ref)
    sol.close()
