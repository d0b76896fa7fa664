"""float32 products of two operands that lie k by k in 64 x 64 tiles (SmallDotColumnsKernel): edges of tiles, of pieces of four and of 16-term chunks, and
what lies behind an operand's rows."""
import numpy as np
import pytest

import chainer_amd as chx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('m,k,n', [(1000, 64, 833), (897, 65, 961), (2601, 130, 258), (1283, 700, 701), (777, 1003, 1030)])
def test_operands_that_lie_k_by_k(m, k, n):
    rng = np.random.default_rng(k)

    def wide(cols):
        a = np.full((k, cols + 3), np.nan, np.float32)
        a[:, :cols] = rng.integers(-3, 4, (k, cols))
        return a

    a, b = wide(m), wide(n)
    got = chx.dot(chx.array(a)[:, :m].T, chx.array(b)[:, :n]).get()
    np.testing.assert_array_equal(got, a[:, :m].T @ b[:, :n])  # whole numbers: exact in any order
