"""GPU: the forms of operators in row runs (test_gpu_runs.py has the runs
themselves): grids whose widest spacing is in y, x or z, so that the sorted slots
end in another direction's neighbours and stage 5/6 runs by runs or by columns.
Every form keeps values and the order of operations: solves are bit-identical to
those without runs."""
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


def _solve(sol, b, **kw):
    import torch
    out = []
    for mixed in (False, True):
        x, i = sol.solve(b, mixed=mixed, **kw)
        torch.cuda.synchronize()
        out.append((x.cpu().numpy(), i["iters"], i["ier"]))
    return out


def _same(got, ref):
    for g, r in zip(got, ref):
        assert g[1:] == r[1:]
        assert np.array_equal(g[0], r[0], equal_nan=True)


def _grid(bed, scale):
    """A box with the spacings (1, 1, 0.5) scaled."""
    from clowns3d import DeviceGrid, configs
    if bed == "wavy":
        g = configs.config_wavy_box(161, 127, 40, (60, 100, 50, 80, 0, 14))
    else:
        g = configs.config_bathymetry(193, 159, 40, nbumps=12)
    for l in range(3):
        g.dx[l] *= scale[l]
        g.xf[l] *= scale[l]
    return DeviceGrid(g)


@pytest.mark.parametrize("scale", [(1, 0.8, 1), (1, 1.25, 1), (1, 1, 4)], ids=["x-widest", "y-widest", "z-widest"])
@pytest.mark.parametrize("bed", ["wavy", "bathymetry"])
def test_spacings(bed, scale, capfd):
    # (the bathymetry has more partial cells than stage 5/6 by runs takes records)
    by = "runs" if bed == "wavy" and scale[1] < 1 else "columns"
    dg = _grid(bed, scale)
    ref = None
    forms = [{"CLOWNS_RUNS": "0"}, {}] + [{"CLOWNS_PM_PAT": p, "CLOWNS_LL8": c} for p in "01" for c in "01"]
    for env in forms:
        capfd.readouterr()
        sol = _solver(dict({"CLOWNS_RUNS": "1", "CLOWNS_VERBOSE": "1"}, **env))
        b = dg.assemble_into(sol)
        got = _solve(sol, b, eps=1e-10, maxiter=4000)
        err = capfd.readouterr().err
        runs = env.get("CLOWNS_RUNS") != "0"
        assert ("stage 5/6 by " + by in err) == runs
        if runs:  # 8-bit codes are built only where a kernel reads them
            assert ("8-bit neighbour codes" in err) == (by == "columns" and env.get("CLOWNS_LL8") == "1")
        sol.close()
        if ref is None:
            ref = got
            assert all(r[2] == 0 for r in ref)
        else:
            _same(got, ref)


def _orders(N):
    """The natural order of the 512-row blocks, a permutation, and back."""
    import torch
    G = ((N + 511) // 512 + 7) // 8 * 8
    perm = np.random.default_rng(N).permutation(G).astype(np.int32)
    return [None, torch.from_numpy(perm).to("cuda:0"), None]


@pytest.mark.parametrize("stream", ["0", "1"], ids=["cached", "streamed"])
@pytest.mark.parametrize("scale", [(1, 0.8, 1), (1, 1.25, 1)], ids=["runs", "columns"])
def test_streams_and_block_orders(scale, stream):
    dg = _grid("wavy", scale)
    sol = _solver({"CLOWNS_RUNS": "0", "CLOWNS_STREAM": stream})
    ref = _solve(sol, dg.assemble_into(sol), eps=1e-10, maxiter=4000)
    sol.close()
    sol = _solver({"CLOWNS_RUNS": "1", "CLOWNS_STREAM": stream})
    b = dg.assemble_into(sol)
    for order in _orders(dg.N):
        sol.set_block_order(order)
        _same(_solve(sol, b, eps=1e-10, maxiter=4000), ref)
        t = sol.tuning()
        assert t["index64"] == 0 and t["stream64"] == t["stream32"] == int(stream)
    sol.close()


def _arrays(N, adjacent, ghost):
    """Runs of every kind (test_gpu_runs.synthetic), coefficients `ghost` on the
    slots that have no neighbour."""
    import torch
    from test_gpu_runs import synthetic
    LL, coef, D = synthetic(N, 11, 0.05, 0.0005, adjacent, 600)
    coef = np.where(LL == 0, ghost, coef)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    return t(coef.T), t(LL.T), t(D)


@pytest.mark.parametrize("adjacent", [True, False], ids=["adjacent", "not-adjacent"])
def test_ghost_coefficients_orders_and_exits(adjacent):
    """Ghost slots stay zero whatever their coefficient; a zero and a non-finite
    right-hand side end a run at once, as by the column kernels."""
    import torch
    N = 262657
    op = _arrays(N, adjacent, -0.01)
    rng = np.random.default_rng(5)
    b = rng.uniform(-1.0, 1.0, size=N)
    nan, inf = b.copy(), b.copy()
    nan[N // 3] = np.nan
    inf[N - 1] = np.inf
    rhs = [torch.from_numpy(v).to("cuda:0") for v in (b, b * 1e300, np.zeros(N), nan, inf)]
    out = []
    for runs in "01":
        sol = _solver({"CLOWNS_RUNS": runs})
        sol.set_matrix(*op)
        got = []
        for order in _orders(N):
            sol.set_block_order(order)
            for v in rhs:
                got += _solve(sol, v, eps=1e-9, maxiter=25)
        assert (sol.tuning()["index64"] == 0) == (runs == "1")
        sol.close()
        out.append(got)
    _same(out[1], out[0])
    first = out[0][:2 * len(rhs)]
    assert np.all(np.isfinite(first[0][0])) and first[0][1] > 1
    assert first[2][2] == 4001 and first[4][1:] == (0, 0)


@pytest.mark.parametrize("cfg,rows", [(2, 2449992), (3, 13066133)])
def test_full_size_default(cfg, rows):
    """The forms that the solver takes by default at full size, the grid's block
    order among them, against the column kernels."""
    from clowns3d import DeviceGrid, configs
    dg = DeviceGrid(configs.CONFIGS[cfg]())
    assert dg.N == rows
    out = []
    for env in ({}, {"CLOWNS_RUNS": "0"}):
        sol = _solver(env)
        b = dg.assemble_into(sol)
        out.append(_solve(sol, b, eps=1e-10))
        assert (sol.tuning()["index64"] == 0) == (env == {})
        sol.close()
    _same(out[0], out[1])
    assert all(r[2] == 0 for r in out[0])


def test_natural_order_again():
    """set_block_order(None) takes the tasks back too, not the index arrays
    alone: the SpMV is as fast as before the order that slowed it."""
    from clowns3d import DeviceGrid, configs
    dg = DeviceGrid(configs.config2())
    sol = _solver({"CLOWNS_BLOCK_ORDER": "0"})
    dg.assemble_into(sol)
    times = []
    for order in _orders(dg.N):
        sol.set_block_order(order)
        times.append(min(sol.time_kernel(0, 50) for _ in range(3)))
    sol.close()
    print(times)
    # (13.1, 17.6 and 17.6 us before, the last now as the first)
    if times[1] < 1.15 * times[0]:
        pytest.skip("the permuted order costs too little here to tell")
    assert times[2] < 0.5 * (times[0] + times[1])
