"""Direct solves of Kronecker-sum systems (hfh_fdm.hpp) through the solver
engine, against a dense solve: every pair of end rows, box sizes around the
32-wide tiles and the 4-deep k-steps, the special unknowns (eliminated with
and without its column, added diagonal), 2D and 3D; and matrices one entry
away from the form, which keep the Krylov solver.

Tolerance: the engine stops at ||b - A x|| <= rtol ||b||, so the error is at
most cond(A) rtol of ||x||; rtol is 1e-12 and cond(A) is computed."""
import itertools

import numpy as np
import pytest

from higflow_amd import native

pytestmark = pytest.mark.gpu

RTOL = 1e-12
ENDS = {"N": 1.0, "D": 0.0, "H": -1.0}  # Neumann, Dirichlet at a node, Dirichlet at half a cell


def _line(n, b, ends):
    t = 2.0 * np.eye(n) - np.eye(n, k=1) - np.eye(n, k=-1)
    t[0, 0] -= ENDS[ends[0]]
    t[-1, -1] -= ENDS[ends[1]]
    return b * t


def _box(sizes, ends, shift=0.0):
    """sum over the dimensions of I x T_d x I, first dimension fastest."""
    n = int(np.prod(sizes))
    a = shift * np.eye(n)
    for d in range(len(sizes)):
        left = np.eye(int(np.prod(sizes[d + 1:], dtype=int)))
        right = np.eye(int(np.prod(sizes[:d], dtype=int)))
        a += np.kron(np.kron(left, _line(sizes[d], 1.0 + 0.5 * d, ends[d])), right)
    return a


def _solve(a, b, impose=None):
    n = len(b)
    s = native.LinearSolver(0, n)
    s.set_tolerances(RTOL, 0.0, 20000)
    for i in range(n):
        c = np.nonzero(a[i])[0]
        s.set_Ai(i, c, a[i, c])
        s.set_bi(i, b[i])
    if impose is not None:
        s.impose_value(impose, b[impose])
    s.assemble()
    s.solve()
    return s.get_x(), s.stats()


def _check(a, b, impose=None, direct=True):
    x, (_, iters, _) = _solve(a, b, impose)
    full = a.copy()
    if impose is not None:
        full[impose] = 0.0
        full[impose, impose] = 1.0
    xd = np.linalg.solve(full, b)
    assert np.linalg.norm(x - xd) <= np.linalg.cond(full) * RTOL * np.linalg.norm(xd)
    assert (iters <= 4) == direct, iters


@pytest.mark.parametrize("ends", ["".join(e) for e in itertools.product("NDH", repeat=2)])
def test_end_rows(ends):
    b = np.random.default_rng(1).normal(size=9 * 7)
    _check(_box((9, 7), (ends, ends[::-1]), shift=0.4), b)


@pytest.mark.parametrize("sizes", [(3, 3), (4, 5), (15, 17), (31, 33), (32, 32), (33, 3), (3, 64), (65, 20),
                                   (3, 3, 3), (5, 4, 6), (11, 33, 3), (33, 3, 9),
                                   # one workgroup up to 2048 rows, tiles of many above
                                   (64, 32), (45, 46), (33, 65), (8, 16, 16), (12, 12, 15)])
def test_box_sizes(sizes):
    b = np.random.default_rng(2).normal(size=int(np.prod(sizes)))
    _check(_box(sizes, ["NH", "DD", "HN"][:len(sizes)], shift=0.1), b)


@pytest.mark.parametrize("sizes", [(8, 6), (33, 12), (5, 6, 7), (49, 43), (13, 12, 14)])
@pytest.mark.parametrize("mode", ["eliminated", "imposed", "shifted"])
@pytest.mark.parametrize("where", ["first", "inside", "last"])
def test_special_unknown(sizes, mode, where):
    n = int(np.prod(sizes))
    p = {"first": 0, "inside": n // 3, "last": n - 1}[where]
    a = _box(sizes, ["NN"] * len(sizes))
    b = np.random.default_rng(3).normal(size=n)
    if mode == "shifted":
        a[p, p] += 0.7
        _check(a, b)
    elif mode == "imposed":
        _check(a, b, impose=p)
    else:
        a[p] = a[:, p] = 0.0
        a[p, p] = 1.5
        _check(a, b)


@pytest.mark.parametrize("what", ["coupling", "diagonal", "wrap", "definite_pin"])
def test_other_matrices_keep_the_krylov_solver(what):
    a = _box((12, 10), ["ND", "HN"], shift=0.2)
    if what == "coupling":
        a[30, 31] *= 1.0 + 1e-6
    elif what == "diagonal":
        a[30, 30] *= 1.1
    elif what == "wrap":
        a[11, 12] = a[12, 11] = -1.0
    else:
        a[40] = a[:, 40] = 0.0
        a[40, 40] = 1.0
    _check(a, np.random.default_rng(4).normal(size=120), direct=False)
