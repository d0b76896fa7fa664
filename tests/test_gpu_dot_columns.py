"""Large float16 products whose operands lie k by k (GemmPpKernel's transposing reads) and those of short reductions (tiles of 256 x 128): edges of the
tiles, of 32-wide chunks and of 8-element pieces, one slice and several, and what lies behind an operand's rows or columns."""
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


@pytest.mark.parametrize('m,k,n', [(2050, 66, 2306), (1300, 130, 1701), (4100, 450, 700), (1030, 512, 2051), (20000, 64, 130), (130, 95, 17000)])
def test_short_reductions(m, k, n):
    rng = np.random.default_rng(k)

    def wide(lines):
        a = np.full((lines, k + 3 - k % 2), np.nan, np.float16)[:, :(k + 3 - k % 2) // 2 * 2]
        a[:, :k] = rng.integers(-2, 3, (lines, k))
        return a

    x, w, b = wide(m), wide(n), rng.integers(-8, 9, n).astype(np.float16)
    got = chx.linear(chx.array(x)[:, :k], chx.array(w)[:, :k], chx.array(b)).get()
    np.testing.assert_array_equal(got, (x[:, :k].astype(np.float32) @ w[:, :k].T.astype(np.float32) + b).astype(np.float16))  # exact in any order
