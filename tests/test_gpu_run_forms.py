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
