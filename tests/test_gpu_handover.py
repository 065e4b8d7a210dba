"""What a direct solve leaves behind when a right-hand side is not finite, or
when some systems of a batch end before others: the next solves and the other
systems are, to the bit, what they are without it."""
import numpy as np
import pytest

from higflow_amd import cases, native

pytestmark = pytest.mark.gpu

TOL = dict(rtol=1e-11, atol=1e-11, maxit=50000)


def _engine(nx, ny):
    """Five-point Helmholtz rows on nx x ny, solved directly."""
    s = native.LinearSolver(0, nx * ny)
    s.set_tolerances(1e-12, 0.0, 20000)
    for r in range(nx * ny):
        i, j = r % nx, r // nx
        c = [r + o for o, ok in ((-1, i > 0), (1, i < nx - 1), (-nx, j > 0), (nx, j < ny - 1)) if ok]
        s.set_Ai(r, c + [r], [-1.0] * len(c) + [len(c) + 0.3])
    s.assemble()
    return s


def _set(s, b, x0):
    for r in range(len(b)):
        s.set_bi(r, b[r])
        s.set_xi(r, x0[r])


# one workgroup; tiles
@pytest.mark.parametrize("nx, ny", [(20, 17), (70, 40)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_right_hand_side_that_is_not_finite(nx, ny, bad):
    rng = np.random.default_rng(0)
    b, x0 = rng.normal(size=nx * ny), rng.normal(size=nx * ny)
    fresh = _engine(nx, ny)
    _set(fresh, b, x0)
    fresh.solve()
    assert fresh.stats()[0] == 1 and fresh.stats()[1] <= 4
    s = _engine(nx, ny)
    worse = b.copy()
    worse[nx * ny // 2] = bad
    _set(s, worse, x0)
    s.solve()
    assert s.stats()[0] == 0
    # x stays what it was, and the next solve is a direct one from there
    assert np.array_equal(s.get_x(), x0)
    _set(s, b, s.get_x())
    s.solve()
    assert s.stats()[:2] == fresh.stats()[:2]
    assert np.array_equal(s.get_x(), fresh.get_x())


def _batch(sides, dim, precision):
    # couplings of the velocity systems strong enough for the direct solve
    return native.Batch([cases.cavity(n, dim=dim, Re=re if dim == 2 else 0.1 * re, dt=1e-3,
                                      tempdiscrtype=cases.SEMI_IMPLICIT_EULER, **TOL)
                         for n, re in zip(sides, (1.0, 3.0, 2.0))], precision=precision, inner_rtol=1e-5)


# every system in one workgroup; tiles; 3D
@pytest.mark.parametrize("sides, dim", [((24, 17, 32), 2), ((24, 50, 65), 2), ((6, 9, 8), 3)])
@pytest.mark.parametrize("precision", [0, 1])
def test_members_beside_one_that_is_not_finite(sides, dim, precision):
    a, b = _batch(sides, dim, precision), _batch(sides, dim, precision)
    for s in (a, b):
        s.advance(3)
    same = lambda ms: [(m, f, c) for m in ms for f, c in [(1, 0), (2, 0)] + [(f, d) for f in (0, 3) for d in range(dim)]
                       if not np.array_equal(a.get(m, f, c), b.get(m, f, c))]
    assert not same(range(3))
    state = [(f, c, a.get(1, f, c)) for f, c in [(1, 0), (2, 0)] + [(f, d) for f in (0, 3) for d in range(dim)]]
    u = state[2][2].copy()
    u[len(u) // 2] = np.nan
    a.set(1, 1, 0, state[0][2])  # both runs start again from their own states
    b.set(1, 0, 0, u)
    for k in range(3):
        a.step()
        b.step()
        assert not same([0, 2])
        assert all(b.solve_stats(m, w)["iters"] <= 4 for m in (0, 2) for w in range(dim + 1))
        # its momentum has no finite right-hand side (later steps may: u* has
        # kept the guess)
        assert k > 0 or not all(b.solve_stats(1, w)["converged"] for w in range(1, dim + 1))
    # the member is given a good state again: as if nothing had happened
    for s in (a, b):
        for f, c, v in state:
            s.set(1, f, c, v)
    for _ in range(2):
        a.step()
        b.step()
        assert not same(range(3))
