"""Large float16 products whose operands lie k by k (GemmPpKernel's transposing reads): edges of the 256 x 256 tiles, of 32-wide chunks and of 8-element
pieces, one slice and several, and what lies behind an operand's columns."""
import numpy as np
import pytest

import chainer_amd as chx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('cols_a,cols_b', [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize('m,k,n', [(1030, 1002, 1041), (1283, 1024, 770), (650, 4481, 1300), (2049, 130, 2300), (515, 9000, 513)])
def test_operands_that_lie_k_by_k(cols_a, cols_b, m, k, n):
    rng = np.random.default_rng(k)

    def operand(lines, cols):
        shape = (k, lines) if cols else (lines, k)
        wide = np.full((shape[0], shape[1] + 3 + shape[1] % 2 * 3), np.nan, np.float16)  # rows of an even number of elements, NaN behind them
        wide = wide[:, :wide.shape[1] // 2 * 2]
        wide[:, :shape[1]] = rng.integers(-2, 3, shape)
        dev = chx.array(wide)[:, :shape[1]]
        mat = wide[:, :shape[1]].astype(np.float32)
        return (dev.T, mat.T) if cols else (dev, mat)

    a, am = operand(m, cols_a)
    bt, btm = operand(n, cols_b)
    expected = am @ btm.T  # whole numbers below 2^24: exact in any order
    np.testing.assert_array_equal(chx.dot(a, bt.T).get(), expected.astype(np.float16))
