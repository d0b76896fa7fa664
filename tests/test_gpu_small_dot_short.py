"""Products of fewer than 64 terms: ends of the reduction in every piece of a load, edges of tiles, and the limits of the kernels' choice, in every layout."""
import numpy as np
import pytest

import chainer_amd as chx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt', ['float16', 'float32'])
@pytest.mark.parametrize('k', [1, 2, 3, 4, 7, 8, 9, 15, 16, 17, 31, 32, 33, 48, 63])
@pytest.mark.parametrize('m,n', [(1, 1), (4, 33), (64, 64), (65, 31), (33, 1000), (1030, 16)])
def test_few_terms(dt, m, n, k):
    _check(dt, m, n, k)


@pytest.mark.parametrize('dt', ['float16', 'float32'])
@pytest.mark.parametrize('m,n,k', [(128, 128 * 127 + 1, 16), (257, 128 * 85, 33), (257, 128 * 85 + 1, 34), (128 * 255, 3, 8), (128 * 255 + 1, 5, 63)])
def test_limits_of_the_choice(dt, m, n, k):
    _check(dt, m, n, k)


def _check(dt, m, n, k):
    """Whole numbers whose sums (at most 63 * 4 * 4) every type and order holds exactly, among others' elements that are not numbers."""
    rng = np.random.default_rng(m + 3 * n + 7 * k)

    def layouts(a):
        wide = np.full((a.shape[0], k + 3), np.nan, dt)
        wide[:, 2:2 + k] = a
        tall = np.full((k, a.shape[0] + 1), np.inf, dt)
        tall[:, :-1] = a.T
        return chx.array(a), chx.array(np.ascontiguousarray(a.T)).T, chx.array(wide)[:, 2:2 + k], chx.array(tall)[:, :-1].T

    a, b = (rng.integers(-4, 5, (rows, k)).astype(dt) for rows in (m, n))
    ref = a.astype(np.float32) @ b.astype(np.float32).T
    if m > 1000:  # rows from the last to the first
        np.testing.assert_array_equal(chx.dot(chx.array(np.ascontiguousarray(a[::-1]))[::-1], chx.array(b).T).get(), ref.astype(dt))
    for x in layouts(a):
        for y in layouts(b):
            np.testing.assert_array_equal(chx.dot(x, y.T).get(), ref.astype(dt))
