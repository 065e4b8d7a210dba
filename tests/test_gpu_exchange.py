"""Field exchange through the pinned buffer (4 MiB, writes in chunks of 2,
reads of 4): what is written is read back, whatever was enqueued before."""
import numpy as np
import pytest

from higflow_amd import cases, native

pytestmark = pytest.mark.gpu

KW = dict(rtol=1e-10, atol=1e-10, maxit=100)


def _values(f, field, comp, seed):
    return np.random.default_rng(seed).normal(size=f.size(field, comp))


def test_writes_past_the_end_of_the_buffer():
    # 60 fields of 128 KB between two waits
    f = native.Flow(cases.cavity(128, dt=1e-4, **KW))
    want = {}
    for k in range(60):
        field, comp = [(0, 0), (0, 1), (1, 0), (2, 0), (3, 0), (3, 1), (4, 0)][k % 7]
        want[field, comp] = _values(f, field, comp, k)
        f.set(field, comp, want[field, comp])
    for (field, comp), v in want.items():
        assert np.array_equal(f.get(field, comp), v)


def test_fields_larger_than_a_chunk():
    # 4.2 MiB: more than a whole buffer to read, more than two chunks to write
    f = native.Flow(cases.cavity(742, dt=1e-6, **KW))
    assert 8 * f.size(1) > 4 << 20
    a, b = _values(f, 1, 0, 1), _values(f, 2, 0, 2)
    f.set(1, 0, a)
    f.set(2, 0, b)
    assert np.array_equal(f.get(1), a) and np.array_equal(f.get(2), b)
    f.set(1, 0, b)
    assert np.array_equal(f.get(2), b) and np.array_equal(f.get(1), b)


def test_solver_closed_with_writes_on_their_way():
    case = cases.cavity(96, dt=1e-4, **KW)
    keep = native.Flow(case)
    v = _values(keep, 1, 0, 0)
    keep.set(1, 0, v)
    for k in range(8):
        f = native.Flow(cases.cavity(16, dt=1e-4, **KW))
        for q in range(20):
            f.set(1, 0, _values(f, 1, 0, q))
        f.close()
    assert np.array_equal(keep.get(1), v)
