"""Small matrix products: every way an operand can lie in memory, split reductions, few rows, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(chx, a, b, A, B):
    got = chx.dot(A, B).get().astype(np.float64)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    scale = np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64))
    tol = 2e-6 if a.dtype == np.float32 else 1e-3
    assert np.all(np.abs(got - ref) <= tol * scale + 1e-30), np.abs(got - ref).max()


@pytest.mark.parametrize('dt', ['float16', 'float32'])
@pytest.mark.parametrize('m,k,n', [(1, 8, 1), (1, 784, 1000), (2, 333, 65), (4, 2048, 33), (5, 9, 31), (20, 650, 2600), (20, 2600, 650), (33, 65, 97),
                                   (128, 650, 2600), (100, 1000, 10), (3, 6001, 5), (31, 10007, 40), (650, 700, 650), (64, 63, 64), (40, 97, 1300)])
def test_layouts(dt, m, k, n):
    import chainer_amd as chx
    rng = np.random.default_rng(m * 31 + k * 7 + n)
    a = (rng.standard_normal((m, k)) / np.sqrt(k)).astype(dt)
    b = rng.standard_normal((k, n)).astype(dt)
    at, bt = np.ascontiguousarray(a.T), np.ascontiguousarray(b.T)
    for A in (chx.array(a), chx.array(at).T):
        for B in (chx.array(b), chx.array(bt).T):
            _check(chx, a, b, A, B)
    # rows inside a larger array whose other elements are not numbers
    wide = np.full((m, k + 5), np.nan, dt)
    wide[:, 3:3 + k] = a
    tall = np.full((n, k + 3), np.inf, dt)
    tall[:, 1:1 + k] = bt
    _check(chx, a, b, chx.array(wide)[:, 3:3 + k], chx.array(tall)[:, 1:1 + k].T)
