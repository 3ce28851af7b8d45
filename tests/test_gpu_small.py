"""GPU: the small kernels (k_small_spmv, k_small_pm, k_small_update), an
iteration in five launches, or nine with the column kernels' PM.  They repeat
work to save launches but keep every value and the order of operations, so
solves must be bit-identical to the single kernels': sizes around the
wavefronts, row blocks and workgroups, both precisions and coefficient widths,
warm starts, runs that end at the first iterations, zero and non-finite
right-hand sides, slots without a neighbour that carry a coefficient, and the
solve that does not allocate."""
import os

import numpy as np
import pytest

from _systems import box_system

pytestmark = pytest.mark.gpu


def _solver(env):
    from clowns3d import Solver
    os.environ.update(env)
    try:
        return Solver(0)  # reads the switches at creation
    finally:
        for k in env:
            del os.environ[k]


def _runs(env, s, b, calls):
    import torch
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    sol = _solver(env)
    sol.set_matrix(t(s["AL"].T), t(s["LL"].T), t(s["D"]))
    b = t(b)
    out = []
    for kind, kw in calls:
        kw = dict(kw)
        if kind == "noalloc":
            x, i = sol.solve_noalloc(b, torch.zeros_like(b), **kw)
        elif kind == "transpose":
            x, i = sol.solve_transpose(b, **kw)
        else:
            x0 = t(np.linspace(-1.0, 1.0, b.numel())) if kind == "warm" else None
            x, i = sol.solve(b, x0, warm=kind == "warm", **kw)
        torch.cuda.synchronize()
        out.append((kind, kw, x.cpu().numpy(), i["iters"], i["ier"]))
    sol.close()
    return out


def _check(s, b, calls, on=("1", "2", "-1")):
    ref = _runs({"CLOWNS_SMALL": "0", "CLOWNS_RUNS": "0"}, s, b, calls)
    for form in on:
        got = _runs({"CLOWNS_SMALL": form}, s, b, calls)
        for g, r in zip(got, ref):
            assert g[3:] == r[3:], (form, g[0], g[1])
            assert np.array_equal(g[2], r[2], equal_nan=True), (form, g[0], g[1])
    return ref


ITERS = [("solve", dict(eps=1e-14, maxiter=m, mixed=mixed)) for m in (1, 2, 3, 7) for mixed in (False, True)]
WHOLE = [("solve", dict(eps=1e-10)), ("solve", dict(eps=1e-10, mixed=True)), ("warm", dict(eps=1e-10)),
         ("warm", dict(eps=1e-10, mixed=True)), ("noalloc", dict(eps=1e-10)),
         ("noalloc", dict(eps=1e-10, mixed=True)), ("transpose", dict(eps=1e-10))]


@pytest.mark.parametrize("shape", [(1, 1, 2), (2, 1, 2), (9, 7, 2), (127, 1, 2), (128, 1, 2), (43, 3, 2), (17, 15, 2),
                                   (16, 16, 2), (57, 3, 3), (32, 16, 2), (41, 5, 5), (31, 29, 3), (24, 16, 10),
                                   (43, 41, 7), (61, 45, 37)])
def test_sizes(shape):
    s = box_system(*shape, seed=sum(shape))
    ref = _check(s, s["B"], ITERS + WHOLE)
    # (two rows converge exactly: iterations forced past that divide 0 by 0)
    assert all(np.all(np.isfinite(r[2])) for r in ref if s["N"] > 4 or r[1].get("maxiter") == 1)


def test_single_precision_coefficients_of_the_inner_solve():
    s = box_system(33, 31, 9, seed=5)
    env = {"CLOWNS_PM_HALF": "0"}
    a = _runs(dict(env, CLOWNS_SMALL="0"), s, s["B"], WHOLE)
    for form in ("1", "2"):
        for g, r in zip(_runs(dict(env, CLOWNS_SMALL=form), s, s["B"], WHOLE), a):
            assert g[3:] == r[3:] and np.array_equal(g[2], r[2])


@pytest.mark.parametrize("bed", ["wavy", "bathymetry"])
def test_assembled_with_patterns(bed):
    """Past the size from which the operator has row patterns."""
    import torch
    from clowns3d import DeviceGrid, configs
    if bed == "wavy":
        g = configs.config_wavy_box(129, 125, 36, (60, 100, 50, 80, 0, 14))
    else:
        g = configs.config_bathymetry(131, 127, 36, nbumps=12)
    dg = DeviceGrid(g)
    out = []
    for env in ({"CLOWNS_SMALL": "0"}, {"CLOWNS_SMALL": "1"}, {"CLOWNS_SMALL": "2"}, {}):
        sol = _solver(env)
        b = dg.assemble_into(sol, keep_raw=True)
        r = [sol.solve(b, eps=1e-10), sol.solve(b, eps=1e-10, mixed=True), sol.solve_transpose(b, eps=1e-10)]
        torch.cuda.synchronize()
        out.append(([x.cpu().numpy() for x, _ in r], [(i["iters"], i["ier"]) for _, i in r]))
        sol.close()
    for o in out[1:]:
        assert o[1] == out[0][1]
        assert all(np.array_equal(a, b) for a, b in zip(o[0], out[0][0]))


def test_coefficients_without_a_neighbour_and_exits():
    """Ghost slots stay zero whatever their coefficient and whatever an earlier
    solve left; a zero and a non-finite right-hand side end a run at once."""
    s = box_system(24, 20, 10, seed=42)
    N = s["N"]
    for k in range(6):
        m = s["LL"][:N, k] == 0
        s["AL"][:N, k][m] = -0.01
    calls = [("solve", dict(eps=1e-10, mixed=mixed)) for mixed in (False, True)]
    ref = _check(s, s["B"] * 1e300, calls + ITERS)
    assert ref[0][4] == 4001
    ref = _check(s, np.zeros(N), calls)
    assert all(r[3] == 0 and r[4] == 0 for r in ref)
    _check(s, s["B"], calls + ITERS)
