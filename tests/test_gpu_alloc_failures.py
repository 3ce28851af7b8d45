"""GPU: device allocations that fail, one at a time, while an operator is set up
and solved on a handle that held another operator.  A call whose allocation
fails either does without (the column kernels stand in for records and row runs:
the same results bit for bit) or returns CLOWNS_ENOMEM; after a failed set-up the
handle holds no operator and refuses to solve; either way the same call made
again gives what a new solver gives, and so does the smaller operator set again.

The failures come from a hipMalloc of its own in front of the runtime's, which
counts the solver library's calls: a process of its own, since it has to be
loaded before the library is."""
import ctypes
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <link.h>
#include <string.h>
static int (*real)(void **, size_t);
static int left = 0, seen = 0;
static int find(struct dl_phdr_info *i, size_t n, void *p) {
    if (!strstr(i->dlpi_name, "libamdhip64")) return 0;
    void *h = dlopen(i->dlpi_name, RTLD_LAZY | RTLD_NOLOAD);
    if (h) real = (int (*)(void **, size_t))dlsym(h, "hipMalloc");
    return real != 0;
}
void shim_arm(int k) { left = k; seen = 0; } /* the k-th call from now on fails */
int shim_seen(void) { return seen; }
int hipMalloc(void **p, size_t n) {
    Dl_info d;
    if (!real) dl_iterate_phdr(find, 0);
    if (dladdr(__builtin_return_address(0), &d) && strstr(d.dli_fname, "libclowns_pcg")) {
        ++seen;
        if (left > 0 && --left == 0) {
            *p = 0;
            return 2; /* hipErrorOutOfMemory */
        }
    }
    return real(p, n);
}
"""

CASES = ["small", "nine", "runs", "runs-codes"]


@pytest.mark.parametrize("case", CASES)
def test_allocation_failures(case, tmp_path):
    src, so = tmp_path / "shim.c", tmp_path / "libshim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(so), str(src), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), str(so), case], timeout=110)
    assert r.returncode == 0


def _system(case):
    """A system (AL (6, N), LL (6, N), D, B) of the size whose forms the case is about."""
    import numpy as np
    from _systems import box_system
    from test_gpu_runs import synthetic
    if case.startswith("runs"):
        N = 262145
        LL, AL, D = synthetic(N, 7, 0.05, 0.0005, case == "runs", 600)
        return AL.T, LL.T, D, np.random.default_rng(N).uniform(-1.0, 1.0, size=N)
    s = box_system(*((31, 29, 13) if case == "small" else (71, 53, 37)), seed=9)
    N = s["N"]
    return s["AL"][:N].T, s["LL"][:N].T, s["D"], s["B"]


def _child(path, case):
    shim = ctypes.CDLL(path, ctypes.RTLD_GLOBAL)  # before the library and torch
    here = os.path.dirname(os.path.abspath(__file__))
    sys.path[:0] = [here, os.path.join(os.path.dirname(here), "2clowns-3d_amd")]
    import numpy as np
    import torch
    from _systems import box_system
    from clowns3d import ClownsError, Solver
    from clowns3d._lib import CLOWNS_EBADARG, CLOWNS_ENOMEM
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    s = box_system(24, 16, 10, seed=3)
    first = [t(a) for a in (s["AL"][:s["N"]].T, s["LL"][:s["N"]].T, s["D"], s["B"])]
    then = [t(a) for a in _system(case)]

    def solver():
        os.environ["CLOWNS_RUNS"] = "1" if case.startswith("runs") else "-1"
        sol = Solver(0)  # reads the switch at creation
        del os.environ["CLOWNS_RUNS"]
        return sol

    def steps(sol, op):
        b = op[3]
        kw = dict(eps=1e-10, maxiter=30)
        yield lambda: sol.set_matrix(*op[:3])
        yield lambda: sol.solve(b, **kw)
        yield lambda: sol.solve(b, mixed=True, **kw)
        if not case.startswith("runs"):  # whose patterns are not symmetric
            yield lambda: sol.solve_transpose(b, **kw)

    def keep(r):
        return None if r is None else (r[0].cpu().numpy(), r[1]["iters"], r[1]["ier"])

    def same(a, b):
        return all(x is y or (np.array_equal(x[0], y[0]) and x[1:] == y[1:]) for x, y in zip(a, b))

    def whole(op):
        sol = solver()
        out = [keep(f()) for f in steps(sol, op)]
        print(case, sol.N, "rows", sol.tuning(), [r[1:] for r in out[1:]], flush=True)
        sol.close()
        return out

    ref_first, ref_then = whole(first), whole(then)
    k, failed, without = 0, 0, 0
    while True:
        k += 1
        sol = solver()
        assert same([keep(f()) for f in steps(sol, first)], ref_first)
        shim.shim_arm(k)
        out, errors = [], 0
        for n, f in enumerate(steps(sol, then)):
            try:
                out.append(keep(f()))
            except ClownsError as e:
                assert e.code == CLOWNS_ENOMEM, e
                errors += 1
                if n == 0:
                    for g in list(steps(sol, then))[1:]:
                        try:
                            g()
                            raise AssertionError("solved without an operator")
                        except ClownsError as e2:
                            assert e2.code == CLOWNS_EBADARG, e2
                out.append(keep(f()))
        seen = shim.shim_seen()
        shim.shim_arm(0)
        torch.cuda.synchronize()
        print(case, "allocation", k, "of", seen, "refused" if errors else "done without", sol.tuning(), flush=True)
        assert same(out, ref_then), k
        assert same([keep(f()) for f in steps(sol, first)], ref_first), k
        sol.close()
        failed += errors
        if seen < k:  # none failed
            assert errors == 0
            break
        without += errors == 0
    assert failed > 0 and without > 0
    print(case, "ok", flush=True)


if __name__ == "__main__":
    _child(sys.argv[1], sys.argv[2])
