"""Nested-dissection solves of the systems of refined meshes (hfh_nd.hpp)
against the Krylov solver on the same right-hand side: the first step from
rest solves A dp = b (and, semi-implicit, H u* = c) with b, c that no solve
has touched.  With the true residuals ra, rb (over ||b||) that the solves
report, the solutions differ by at most cond(A) (ra + rb); cond(A) is
estimated in the 1-norm from the assembled operator's factors, with sqrt(n)
for the change of norm on either side.  The direct residual passes the
stopping test, or is at the rounding of b - A x and below the Krylov one."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as sla

from higflow_amd import cases, native

pytestmark = pytest.mark.gpu

RTOL = 1e-11


def _cond(flow, which):
    rp, ci, v, _ = flow.operator(which)
    a = sp.csc_matrix(sp.csr_matrix((v, ci, rp)))
    lu = sla.splu(a)
    inv = sla.LinearOperator(a.shape, matvec=lu.solve, rmatvec=lambda y: lu.solve(y, "T"))
    return sla.onenormest(a) * sla.onenormest(inv) * a.shape[0]


def _pair(case, monkeypatch, **kw):
    a = native.Flow(case, **kw)
    monkeypatch.setenv("HFH_DIRECT", "0")
    b = native.Flow(case, **kw)
    monkeypatch.delenv("HFH_DIRECT")
    a.step()
    b.step()
    return a, b


# one leaf (all rows in one front); a few heights; pivots and fronts on
# either side of 256 (16 and 64 lanes per row); two trees joined in 2D, the
# dense rows of a 3D wall layer
@pytest.mark.parametrize("which", ["leaf", "contraction", "contraction3", "wall", "wall2"])
def test_pressure_of_a_refined_mesh(which, monkeypatch):
    kw = dict(rtol=RTOL, atol=0.0, maxit=50000)
    expl = dict(tempdiscrtype=cases.EXPLICIT_EULER, dt=1e-5, **kw)
    case = {
        "leaf": lambda: cases.wall_layer_cavity(8, dim=2, levels=1, layer=0.05, dt=1e-4, **kw),
        "contraction": lambda: cases.contraction(levels=1, h0=0.5, length=8.0, **expl),
        "contraction3": lambda: cases.contraction(levels=3, h0=0.25, length=10.0, graded=True, **expl),
        "wall": lambda: cases.wall_layer_cavity(4, levels=1, dt=1e-4, **kw),
        "wall2": lambda: cases.wall_layer_cavity(6, levels=2, dt=1e-4, **kw),
    }[which]()
    a, b = _pair(case, monkeypatch)
    sa, sb = a.solve_stats(0), b.solve_stats(0)
    assert sa["iters"] <= 4 < sb["iters"] and sa["resid"] <= max(RTOL, sb["resid"])
    x, y = a.get(2), b.get(2)
    assert np.linalg.norm(x - y) <= _cond(a, 0) * (sa["resid"] + sb["resid"]) * np.linalg.norm(y)


# the same in the residuals, where no condition number enters (on the 3D meshes
# it makes the bound above loose): ||A (x - y)|| <= (ra + rb) ||b|| and, for
# either residual as computed, its rounding (len + 2) u || |A||x| + |b| ||, with
# ||b|| <= ||A y|| / (1 - rb) and |b| <= |A||x| but for ra
@pytest.mark.parametrize("make", [lambda **kw: cases.wall_layer_cavity(4, levels=1, dt=1e-4, **kw),
                                  lambda **kw: cases.wall_layer_cavity(6, levels=2, dt=1e-4, **kw),
                                  lambda **kw: cases.contraction(levels=2, h0=0.25, length=8.0, dt=1e-5,
                                                                 tempdiscrtype=cases.EXPLICIT_EULER, **kw)])
def test_residual_of_the_difference(make, monkeypatch):
    a, b = _pair(make(rtol=RTOL, atol=0.0, maxit=50000), monkeypatch)
    rp, ci, v, _ = a.operator(0)
    m = sp.csr_matrix((v, ci, rp))
    x, y = a.get(2), b.get(2)
    ra, rb = a.solve_stats(0)["resid"], b.solve_stats(0)["resid"]
    bn = np.linalg.norm(m @ y) / (1.0 - rb)
    rounding = np.linalg.norm((np.diff(rp) + 3) * 2.0 ** -53 * (abs(m) @ np.maximum(abs(x), abs(y))))
    assert np.linalg.norm(m @ (x - y)) <= (ra + rb) * bn + 2 * rounding


def test_velocity_blocks_of_a_large_mixed_run(monkeypatch):
    case = cases.contraction(levels=4, graded=True, h0=0.05, dt=1e-5, rtol=RTOL, atol=0.0, maxit=50000)
    a, b = _pair(case, monkeypatch, precision=1, inner_rtol=1e-5)
    # the component that the inflow drives (the other's right-hand side is
    # zero at rest)
    sa, sb = a.solve_stats(1), b.solve_stats(1)
    assert sa["iters"] <= 4 < sb["iters"] and sa["resid"] <= max(RTOL, sb["resid"])
    x, y = a.get(3, 0), b.get(3, 0)
    assert np.linalg.norm(x - y) <= _cond(a, 1) * (sa["resid"] + sb["resid"]) * np.linalg.norm(y)
    assert not a.get(3, 1).any() and not b.get(3, 1).any()


def test_uniform_mesh_with_weak_coupling_keeps_jacobi_pcg():
    # dt / (Re h^2) = 0.0065: no direct solve, and no factors either
    case = cases.cavity(256, Re=1000.0, dt=1e-4, tempdiscrtype=cases.SEMI_IMPLICIT_EULER, rtol=RTOL, atol=0.0, maxit=1000)
    a = native.Flow(case, precision=0)
    b = native.Flow(case, precision=1, inner_rtol=1e-5)
    a.step()
    b.step()
    # a first solve of the mixed form is the FP64 one: the same iterations
    assert a.solve_stats(1)["iters"] == b.solve_stats(1)["iters"] > 1
    assert np.array_equal(a.get(3, 0), b.get(3, 0))
