"""Direct solves that are not the last word: right-hand sides that are not
finite, systems of a batch that end before others, passes that run out.  The
next solves and the other systems are, to the bit, what they are without it."""
import numpy as np
import pytest

from higflow_amd import cases, native

pytestmark = pytest.mark.gpu

TOL = dict(rtol=1e-11, atol=1e-11, maxit=50000)


def _engine(nx, ny, pinned=False):
    """Five-point rows on nx x ny, solved directly: Helmholtz, or Neumann with
    the first unknown imposed."""
    s = native.LinearSolver(0, nx * ny)
    s.set_tolerances(1e-12, 0.0, 20000)
    for r in range(nx * ny):
        i, j = r % nx, r // nx
        c = [r + o for o, ok in ((-1, i > 0), (1, i < nx - 1), (-nx, j > 0), (nx, j < ny - 1)) if ok]
        s.set_Ai(r, c + [r], [-1.0] * len(c) + [len(c) + (0.0 if pinned else 0.3)])
    if pinned:
        s.impose_value(0, 0.0)
    s.assemble()
    return s


def _set(s, b, x0):
    for r in range(len(b)):
        s.set_bi(r, b[r])
        s.set_xi(r, x0[r])


# one workgroup; tiles
@pytest.mark.parametrize("nx, ny", [(20, 17), (70, 40)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("pinned", [False, True])
def test_right_hand_side_that_is_not_finite(nx, ny, bad, pinned):
    rng = np.random.default_rng(0)
    b, x0 = rng.normal(size=nx * ny), rng.normal(size=nx * ny)
    fresh = _engine(nx, ny, pinned)
    _set(fresh, b, x0)
    fresh.solve()
    assert fresh.stats()[1] <= 4
    s = _engine(nx, ny, pinned)
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


@pytest.mark.parametrize("make", [
    lambda: cases.contraction(levels=2, h0=0.25, length=8.0, dt=1e-5, tempdiscrtype=cases.EXPLICIT_EULER, **TOL),
    lambda: cases.wall_layer_cavity(4, levels=1, dt=1e-4, **TOL)])
def test_refined_mesh_after_a_state_that_is_not_finite(make):
    case = make()
    dim = case["dim"]
    a, b = native.Flow(case), native.Flow(case)
    for s in (a, b):
        s.advance(2)
    state = [(1, 0), (2, 0)] + [(f, d) for f in (0, 3) for d in range(dim)]
    if case["params"].get("flowtype") == cases.VISCOELASTIC:
        state += [(6, i * dim + j) for i in range(dim) for j in range(i, dim)]
    state = [(f, c, a.get(f, c)) for f, c in state]
    u = state[2][2].copy()
    u[len(u) // 2] = np.nan
    b.set(0, 0, u)
    b.step()
    # no finite right-hand side: the increment stays the guess
    assert not b.solve_stats(0)["converged"] and np.isfinite(b.get(2)).all()
    for s in (a, b):
        for f, c, v in state:
            s.set(f, c, v)
        s.advance(2)
        assert s.solve_stats(0)["iters"] in range(1, 5)
    assert all(np.array_equal(a.get(f, c), b.get(f, c)) for f, c, _ in state)


def _far(nx, ny):
    """A right-hand side and a guess so far away that the first correction
    leaves a residual of about 2^-53 |A| |x0| = 1e-9 of ||b||."""
    rng = np.random.default_rng(1)
    return rng.normal(size=nx * ny), 1e6 * rng.normal(size=nx * ny)


def _dense(nx, ny):
    s1 = lambda n: 2.0 * np.eye(n) - np.eye(n, k=1) - np.eye(n, k=-1) - np.diag(np.eye(n)[0] + np.eye(n)[-1])
    return np.kron(np.eye(ny), s1(nx)) + np.kron(s1(ny), np.eye(nx)) + 0.3 * np.eye(nx * ny)


@pytest.mark.parametrize("nx, ny", [(20, 17), (70, 40)])
def test_iterations_stay_within_maxit(nx, ny, monkeypatch):
    b, x0 = _far(nx, ny)
    for passes, maxit, converged in ((None, 1, 0), (None, 2, 1), ("1", 1, 0), ("1", 3, None)):
        if passes:
            monkeypatch.setenv("HFH_DIRECT_PASSES", passes)
        s = _engine(nx, ny)
        s.set_tolerances(1e-12, 0.0, maxit)
        _set(s, b, x0)
        s.solve()
        assert s.stats()[1] <= maxit
        assert converged is None or s.stats()[0] == converged


# error at most cond(A) rtol of ||x||, as the stopping test allows
@pytest.mark.parametrize("nx, ny", [(20, 17), (70, 40)])
def test_krylov_goes_on_where_the_passes_end(nx, ny, monkeypatch):
    b, x0 = _far(nx, ny)
    monkeypatch.setenv("HFH_DIRECT_PASSES", "1")
    s = _engine(nx, ny)
    _set(s, b, x0)
    s.solve()
    assert s.stats()[0] == 1 and s.stats()[1] > 4
    a = _dense(nx, ny)
    x = np.linalg.solve(a, b)
    assert np.linalg.norm(s.get_x() - x) <= np.linalg.cond(a) * 1e-12 * np.linalg.norm(x)


def test_member_that_ends_before_another(monkeypatch):
    # to 1e-13 the 16^2 cavity needs one pass and the 96^2 cavity, in the same
    # launches, a second one or (with one pass allowed) the Krylov solver
    runs = []
    for passes in ("4", "1"):
        monkeypatch.setenv("HFH_DIRECT_PASSES", passes)
        b = native.Batch([cases.cavity(n, Re=1.0, dt=1e-3, tempdiscrtype=cases.SEMI_IMPLICIT_EULER, rtol=1e-13,
                                       atol=0.0, maxit=200) for n in (16, 96)])
        for _ in range(3):
            b.step()
            assert all(b.solve_stats(0, w)["iters"] == 1 and b.solve_stats(0, w)["converged"] for w in range(2))
        assert b.solve_stats(1)["iters"] in range(2, 5) if passes == "4" else b.solve_stats(1)["iters"] > 4
        runs.append([b.get(0, f, c) for f, c in ((0, 0), (0, 1), (1, 0), (2, 0))])
    assert all(np.array_equal(p, q) for p, q in zip(*runs))


# the projection and divergence rows are enqueued behind the first pass and run
# again when that was not the last word; with stage timing on they run once,
# after the solve
@pytest.mark.parametrize("make", [
    lambda **kw: cases.cavity(24, Re=1.0, dt=1e-4, **kw),
    lambda **kw: cases.cavity(96, Re=1.0, dt=1e-3, tempdiscrtype=cases.SEMI_IMPLICIT_EULER, **kw),
    lambda **kw: cases.contraction(levels=2, h0=0.25, length=8.0, dt=1e-5, tempdiscrtype=cases.EXPLICIT_EULER, **kw)])
@pytest.mark.parametrize("passes", ["4", "1"])
def test_work_enqueued_behind_a_pass_that_was_not_the_last(make, passes, monkeypatch):
    monkeypatch.setenv("HFH_DIRECT_PASSES", passes)
    runs = []
    for timing in (False, True):
        s = native.Flow(make(rtol=1e-15, atol=0.0, maxit=40))
        s.set_timing(timing)
        for _ in range(3):
            s.step()
            assert s.solve_stats(0)["iters"] > 1
        runs.append([s.get(f, c) for f, c in ((0, 0), (0, 1), (1, 0), (2, 0), (3, 0), (3, 1))])
    assert all(np.array_equal(p, q) for p, q in zip(*runs))


def test_engine_that_asks_for_the_v_cycle_gets_it(monkeypatch):
    b, x0 = _far(70, 40)
    monkeypatch.setenv("HFH_SLV_AMG", "1")
    runs = []
    for direct in (None, "0"):
        if direct:
            monkeypatch.setenv("HFH_DIRECT", direct)
        s = _engine(70, 40)
        _set(s, b, x0)
        s.solve()
        runs.append((s.stats(), s.get_x()))
    assert runs[0][0] == runs[1][0] and np.array_equal(runs[0][1], runs[1][1])
