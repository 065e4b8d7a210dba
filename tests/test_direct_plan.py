"""Which matrices are solved directly, and up to which cost (host work only,
no device): a box whose tables would not fit keeps the Krylov solver, and is
refused before any table is made."""
import numpy as np
import pytest
import scipy.sparse as sp

from higflow_amd import native


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
