"""GPU: the drop-in's host copies.  Columns that fit a pinned chunk together
travel as one copy, larger ones by chunks, and host threads help from 1 MB on:
the arrays that come back (AL, LL, D scaled and sorted in place, rows past N
untouched) are the oracle's bit for bit on both sides of each line, with a
caller's stride larger than N and N off the device's 64-row stride."""
import numpy as np
import pytest

from conftest import call_oracle, copy_system
from _systems import box_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,extra", [
    ((1, 1, 2), 1), ((9, 7, 1), 0), ((16, 4, 1), 5), ((13, 5, 1), 64), ((61, 45, 37), 7),
    ((256, 256, 2), 0), ((257, 255, 2), 3),       # 1 MB a column: 131,072 and 131,070 rows
    ((128, 128, 42), 1), ((131, 107, 50), 2),     # 32 MB of AL: 688,128 and 700,850 rows
])
def test_arrays_come_back(shape, extra):
    import clowns3d
    s = box_system(*shape, seed=sum(shape), na_extra=extra)
    c = copy_system(s)
    N = c["N"]
    tail = {k: c[k][N:].copy() for k in ("AL", "LL")}
    X = np.zeros(N + 64)
    it, ier = clowns3d.pcgpme(c["AL"], 6, c["NA"], c["LL"], c["D"], N, 64, c["B"], X, np.array([1e-10, 0.0]), 5.0, 1)
    o = call_oracle(s, iters=1)
    for k in ("AL", "LL"):
        assert np.array_equal(c[k][:N], o[k][:N])
        assert np.array_equal(c[k][N:], tail[k])
    assert np.array_equal(c["D"][:N], o["D"][:N])
    if shape[2] == 1:  # one layer of surface rows: near the identity, its exit is a matter of rounding
        return
    assert (it, ier) == (o["ITER"], o["IER"])
    assert np.linalg.norm(X[:N] - o["X"][:N]) <= 1e-12 * np.linalg.norm(o["X"][:N])
    assert np.linalg.norm(c["B"][:N] - o["B"][:N]) <= 1e-12 * max(np.linalg.norm(o["B"][:N]), 1e-300)
