"""The interpolation rows as wave tasks (k_interp_t: one template per wave,
column-by-column rows, long rows on 16 lanes) against the same rows on L
lanes each (k_interp_l, forced by HFH_INTERP_LANES).

A row is a sum of at most 120 products, so two orders of summation differ by
at most 2 * 120 * eps * sum |w x|; the weights of a row add up to less than
100 times the value's scale (difference rows over a stretched stencil), hence
5e-12 of each field's scale for everything that is computed before a solve."""
import numpy as np
import pytest

from higflow_amd import cases, native

pytestmark = pytest.mark.gpu

TOL = 5e-12
KW = dict(rtol=1e-10, atol=1e-10, maxit=2000)
VE = dict(flowtype=cases.VISCOELASTIC, De=1.0, beta=0.5)


CASES = {
    # whole waves and remainders of each template; rows of fewer than 64
    "cavity": lambda: cases.cavity(70, Re=10.0, dt=1e-5, **KW),
    "cavity_small": lambda: cases.cavity(9, Re=10.0, dt=1e-4, **KW),
    "ve_cavity": lambda: cases.ve_cavity(33, dt=1e-5, **KW),
    # level jumps: many rows without a common template
    "contraction": lambda: cases.contraction(levels=2, h0=0.25, length=8.0, dt=1e-5,
                                             tempdiscrtype=cases.EXPLICIT_EULER, **KW),
    # rows of up to 120 entries
    "wall3d": lambda: cases.wall_layer_cavity(6, levels=1, dt=1e-4, **KW),
    "ve_cavity3d": lambda: cases.cavity(6, dim=3, Re=10.0, dt=1e-4, **VE, **KW),
}


@pytest.mark.parametrize("which", sorted(CASES))
@pytest.mark.parametrize("lanes", ["1", "8"])
def test_rows_match_lane_groups(which, lanes, monkeypatch):
    case = CASES[which]()
    dim, ve = case["dim"], case["params"].get("flowtype") == cases.VISCOELASTIC
    a = native.Flow(case)
    monkeypatch.setenv("HFH_INTERP_LANES", lanes)
    b = native.Flow(case)
    rng = np.random.default_rng(7)
    state = [(0, d) for d in range(dim)] + [(1, 0)]
    if ve:
        state += [(6, i * dim + j) for i in range(dim) for j in range(i, dim)]
    for f, c in state:
        v = 0.3 * rng.normal(size=a.size(f, c)) + (1.0 if f == 6 and c % (dim + 1) == 0 else 0.0)
        a.set(f, c, v)
        b.set(f, c, v)
    a.step()
    b.step()
    fields = [(3, d) for d in range(dim)]
    if ve:
        fields += [(f, i * dim + j) for f in (6, 7, 8) for i in range(dim) for j in range(i, dim)]
    for f, c in fields:
        x, y = a.get(f, c), b.get(f, c)
        assert np.all(np.isfinite(y))
        assert np.abs(x - y).max() <= TOL * np.abs(y).max(), (f, c)
