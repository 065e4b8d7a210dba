"""Which matrices are solved directly, and up to which cost (host work only,
no device): a box whose tables would not fit keeps the Krylov solver, and is
refused before any table is made."""
import os
import subprocess
import sys

import numpy as np
import pytest
import scipy.sparse as sp

from higflow_amd import native

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _line(n):
    t = sp.diags([-np.ones(n - 1), 2.0 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1], format="lil")
    t[0, 0] = t[n - 1, n - 1] = 1.0
    return t.tocsr()


def _box(*sizes):
    """Neumann box, first dimension fastest, first unknown held by an added diagonal."""
    a = sp.csr_matrix((int(np.prod(sizes)),) * 2)
    for d, n in enumerate(sizes):
        left, right = int(np.prod(sizes[d + 1:])), int(np.prod(sizes[:d]))
        a = a + sp.kron(sp.kron(sp.identity(left), _line(n)), sp.identity(right), format="csr")
    a = a.tolil()
    a[0, 0] += 1.0
    a = a.tocsr()
    a.sort_indices()
    return a


def _plan(a, max_ops=0.0):
    return native.direct_plan(a.indptr, a.indices, a.data, max_ops)


@pytest.mark.parametrize("sizes, direct", [
    ((100000, 3), False), ((3, 100000), False), ((8193, 3), False), ((8192, 3), True), ((3, 8192), True),
    ((8193, 3, 3), False), ((300, 200), True), ((40, 30, 20), True)])
def test_sides_of_a_box(sizes, direct):
    kind, entries = _plan(_box(*sizes))
    assert kind == ("fdm" if direct else None)
    assert entries == 2 * sum(n * n for n in set(sizes))


def test_factors_within_the_operations_allowed():
    a = _box(40, 31)
    a.data = a.data * (1.0 + 0.1 * np.random.default_rng(0).random(a.nnz))  # no Kronecker form
    assert _plan(a) == (None, 0)
    kind, entries = _plan(a, 1e9)
    assert kind == "nd" and entries > a.nnz
    assert _plan(a, 1e3) == (None, entries)


def test_matrices_that_are_none_are_refused():
    with pytest.raises(native.HipError, match="column"):
        native.direct_plan([0, 1], [1], [1.0])
    with pytest.raises(native.HipError, match="row pointers"):
        native.direct_plan([0, 2, 1], [0, 0], [1.0, 1.0])
    assert native.direct_plan([0], [], []) == (None, 0)


_SHORT_OF_MEMORY = """
import resource, sys
import numpy as np
import scipy.sparse as sp
sys.path.insert(0, %r)
from higflow_amd import native
n = 300
t = sp.diags([-np.ones(n - 1), 2.0 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1])
a = (sp.kron(sp.identity(n), t) + sp.kron(t, sp.identity(n)) + 0.1 * sp.identity(n * n)).tocsr()
a.sort_indices()
a.data = a.data * (1.0 + 0.1 * np.random.default_rng(0).random(a.nnz))
plan = lambda: native.direct_plan(a.indptr, a.indices, a.data, 1e12)[0]
native.load()
size = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
soft, hard = resource.getrlimit(resource.RLIMIT_AS)
resource.setrlimit(resource.RLIMIT_AS, (size + int(sys.argv[1]), hard))
first = plan()
resource.setrlimit(resource.RLIMIT_AS, (soft, hard))
print(first, plan())
"""


def test_factors_that_do_not_fit_the_memory():
    """The factors of 90,000 unknowns (95 MB) under a limit on the
    address space: no plan, and with the limit gone the factors are made."""
    env = dict(os.environ, HFH_SETUP_THREADS="1")
    r = subprocess.run([sys.executable, "-c", _SHORT_OF_MEMORY % ROOT, str(64 << 20)], env=env, cwd=ROOT,
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stderr[-500:])
    assert r.stdout.split() == ["None", "nd"]


_THREADS = """
#include <atomic>
#include <cstdio>
#include <new>
#include "hfh_parallel.hpp"
int main() {
    for (int nt : {0, 1, 2, 8})
        for (int bad = -1; bad < 64; bad += 13) {  // the item that fails (-1: none)
            std::atomic<int> next{0}, done{0};
            bool caught = false;
            try {
                hfh::run_parallel(nt, [&](int) {
                    for (int i; (i = next++) < 64;) {
                        if (i == bad) throw std::bad_alloc();
                        done++;
                    }
                });
            } catch (const std::bad_alloc &) {
                caught = true;
            }
            // every item but the failing one, or those up to it on one thread
            if (caught != (bad >= 0) || (bad < 0 && done != 64) || (nt <= 1 && bad >= 0 && done != bad)) return 1;
        }
    return 0;
}
"""


def test_exceptions_of_the_factor_threads_reach_the_caller(tmp_path):
    src, exe = tmp_path / "threads.cpp", tmp_path / "threads"
    src.write_text(_THREADS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "higflow_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True, timeout=120)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0
