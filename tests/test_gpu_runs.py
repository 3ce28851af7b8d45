"""GPU: row runs (k_spmv_run, k_pm_pair_run, k_pm_dot_run).  Operators with row
patterns run by tasks of 128-row windows, lists and records; values and the
order of operations are the column kernels', so solves must be bit-identical
to those with the runs switched off: on assembled grids (uniform and stretched
spacing orders, both block orders, both coefficient widths) and on synthetic
operators whose runs are cut at every length, with odd and even offsets,
ghosts in any slot, rows of their own coefficients, slots that lead elsewhere,
and last slots that are or are not the adjacent rows."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(env):
    from clowns3d import Solver
    os.environ.update(env)
    try:
        return Solver(0)  # reads the switches at creation
    finally:
        for k in env:
            del os.environ[k]


def _equal(setup, env, eps, maxiter, transpose=False):
    """Solutions with runs on and off; returns whether they ran by runs."""
    import torch
    out = []
    for runs in ("1", "0"):
        sol = _solver(dict(env, CLOWNS_RUNS=runs))
        b = setup(sol)
        r = [sol.solve(b, eps=eps, maxiter=maxiter), sol.solve(b, eps=eps, maxiter=maxiter, mixed=True)]
        if transpose:
            r.append(sol.solve_transpose(b, eps=eps, maxiter=maxiter))
        torch.cuda.synchronize()
        out.append(([x.cpu().numpy() for x, _ in r], [(i["iters"], i["ier"]) for _, i in r],
                    sol.tuning()["index64"] == 0))
        sol.close()
    for a, b in zip(out[0][0], out[1][0]):
        assert np.all(np.isfinite(b)) and np.any(b != 0)
        assert np.array_equal(a, b)
    assert out[0][1] == out[1][1]
    assert not out[1][2]
    return out[0][2]


@pytest.mark.parametrize("env", [{}, {"CLOWNS_BLOCK_ORDER": "0"}, {"CLOWNS_PM_HALF": "0"}],
                         ids=["default", "natural-order", "pm-single"])
@pytest.mark.parametrize("bed,dy", [("wavy", 1.0), ("wavy", 0.8), ("wavy", 1.25), ("bathymetry", 1.0),
                                    ("bathymetry", 0.8), ("bathymetry", 1.25)])
def test_assembled(bed, dy, env):
    """dy decides which direction's neighbours the sorted slots name last."""
    from clowns3d import DeviceGrid, configs
    if bed == "wavy":
        g = configs.config_wavy_box(161, 127, 40, (60, 100, 50, 80, 0, 14))
    else:
        g = configs.config_bathymetry(193, 159, 40, nbumps=12)
    g.h = (g.h[0], g.h[1] * dy, g.h[2])
    dg = DeviceGrid(g)
    assert _equal(lambda sol: dg.assemble_into(sol, keep_raw=True), env, 1e-10, 4000, transpose=True)


# relative sizes of the six coefficients of the table rows: those of one row
# differ, so the sort's order (z, y, x pairs) is the generator's
TABLE = np.array([[.30, .28, .20, .18, .10, .08], [.26, .24, .19, .17, .09, .07], [.33, .29, .21, .16, .12, .05]])


def synthetic(N, seed, own, far, adjacent, longest):
    """Rows along lines of 1 .. longest cells; strides of y and z that change
    now and then (odd and even); own: share of the segments with their own
    coefficients, far: of rows with a slot that leads to any row."""
    rng = np.random.default_rng(seed)
    cut = np.cumsum(rng.integers(1, longest + 1, size=2 * N // longest + 64))
    cut = cut[cut < N]
    while cut[-1] < N - longest:
        cut = np.append(cut, cut[-1] + longest)
    first = np.zeros(N, bool)
    first[0] = True
    first[cut] = True
    last = np.append(first[1:], True)
    seg = np.cumsum(first) - 1
    nseg = seg[-1] + 1
    block = np.arange(N) // 5003
    sy = rng.integers(200, 264, size=block[-1] + 1)[block]
    sz = rng.integers(9000, 9064, size=block[-1] + 1)[block]
    r = np.arange(N)
    pairs = [(-sz, sz), (-sy, sy), (-np.ones(N, int), np.ones(N, int))]
    if not adjacent:
        pairs = [pairs[2], pairs[0], pairs[1]]
    LL = np.zeros((N, 6), np.int64)
    for p, (a, b) in enumerate(pairs):
        LL[:, 2 * p] = r + a + 1
        LL[:, 2 * p + 1] = r + b + 1
    p = 2 if adjacent else 0
    LL[first, 2 * p] = 0
    LL[last, 2 * p + 1] = 0
    LL[(LL < 1) | (LL > N)] = 0
    ghost = rng.random(nseg)[seg] < 0.05  # segments without one of their slots
    slot = rng.integers(0, 6, size=nseg)[seg]
    LL[r[ghost], slot[ghost]] = 0
    coef = -TABLE[np.where(rng.random(nseg) < 0.9, 0, rng.integers(1, 3, size=nseg))[seg]]
    mine = (rng.random(nseg) < own)[seg]
    coef[mine] *= rng.uniform(0.99, 1.01, size=(mine.sum(), 6))
    away = np.flatnonzero(rng.random(N) < far)
    LL[away, rng.integers(0, 6, size=away.size)] = rng.integers(1, N + 1, size=away.size)
    coef = np.where(LL == 0, 0.0, coef)
    D = np.full(N, 1.5)
    return LL.astype(np.int32), coef, D


@pytest.mark.parametrize("N,own,far,adjacent,longest", [
    (262144, 0.0, 0.0, True, 400), (262145, 0.05, 0.0, True, 400), (262657, 0.0, 0.001, True, 600),
    (270001, 0.08, 0.002, True, 900), (262399, 0.05, 0.0005, False, 600),
    (300007, 0.3, 0.0, True, 700),  # more records than the two-term form takes
    (262271, 0.0, 0.0, True, 30),  # mostly too short for tasks: the column kernels
])
def test_synthetic(N, own, far, adjacent, longest):
    import torch
    LL, coef, D = synthetic(N, N + longest, own, far, adjacent, longest)
    dev = torch.device("cuda:0")
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    b = t(np.random.default_rng(N).uniform(-1.0, 1.0, size=N))
    al, ll, d = t(coef.T), t(LL.T), t(D)

    def setup(sol):
        sol.set_matrix(al, ll, d)
        return b

    used = _equal(setup, {}, 1e-9, 40)
    assert used == (longest > 30)
