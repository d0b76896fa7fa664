"""Large float16 products on 256 x 256 tiles: remainders of tiles and chunks of the reduction, split reductions, operands in every layout, rows
of the result at any address, a bias, and what lies behind an operand's rows."""
import numpy as np
import pytest

import chainer_amd as chx

pytestmark = pytest.mark.gpu


def _operand(values, layout):
    """values as an array whose rows (r), columns (c) or neither (n) are dense; 'w': rows of a wider array full of NaN."""
    if layout == 'c':
        return chx.array(np.ascontiguousarray(values.T)).T
    if layout == 'r':
        return chx.array(values)
    wide = np.full((values.shape[0], values.shape[1] * (2 if layout == 'n' else 1) + 6), np.nan, values.dtype)
    step = 2 if layout == 'n' else 1
    wide[:, :values.shape[1] * step:step] = values
    return chx.array(wide)[:, :values.shape[1] * step:step]


@pytest.mark.parametrize('a_layout,b_layout', [('r', 'c'), ('r', 'r'), ('c', 'r'), ('n', 'c'), ('w', 'c')])
@pytest.mark.parametrize('m,k,n', [(2048, 2050, 2306), (1793, 650, 2563), (520, 9999, 516), (4096, 4095, 64), (1100, 6007, 777), (2560, 1024, 2560)])
def test_layouts(m, k, n, a_layout, b_layout):
    rng = np.random.default_rng(m + n)
    a = rng.integers(-2, 3, (m, k)).astype(np.float16)
    b = rng.integers(-2, 3, (k, n)).astype(np.float16)
    a[:, k // 3:] *= rng.integers(0, 2, k - k // 3).astype(np.float16)  # sums that float16 holds exactly
    expected = a.astype(np.float32) @ b.astype(np.float32)
    got = chx.to_numpy(chx.dot(_operand(a, a_layout), _operand(b.T, 'w' if b_layout == 'w' else ('r' if b_layout == 'c' else 'c')).T))
    np.testing.assert_array_equal(got, expected.astype(np.float16))


@pytest.mark.parametrize('m,k,n', [(2048, 2050, 2306), (520, 9999, 516), (1792, 642, 2563)])
def test_bias(m, k, n):
    rng = np.random.default_rng(k)
    x = rng.integers(-2, 3, (m, k)).astype(np.float16)
    w = rng.integers(-2, 3, (n, k)).astype(np.float16)
    bias = rng.integers(-50, 51, n).astype(np.float16)
    expected = x.astype(np.float32) @ w.T.astype(np.float32) + bias
    got = chx.to_numpy(chx.linear(chx.array(x), chx.array(w), chx.array(bias)))
    np.testing.assert_allclose(got.astype(np.float32), expected, rtol=1e-3)


@pytest.mark.parametrize('dt,rows', [('float32', 2500000), ('float16', 4300000)])  # 65535 tiles of rows are 2097120 and 4194240
@pytest.mark.parametrize('layout', ['r', 'c'])
def test_more_rows_to_lay_out_anew_than_a_launch_takes(dt, rows, layout):
    period = 100
    rng = np.random.default_rng(7)
    x = rng.integers(-2, 3, (period, 65)).astype(dt)  # 65 columns: rows that the matrix kernels do not read as they are
    w = rng.integers(-2, 3, (64, 65)).astype(dt)
    X = chx.array(x)[None].broadcast_to((rows // period, period, 65)).copy().reshape((rows, 65))
    if layout == 'c':
        X = X.T.copy().T
    got = chx.linear(X, chx.array(w))
    expected = (x.astype(np.float32) @ w.T.astype(np.float32)).astype(dt)
    cut = 65535 * 128 // x.itemsize
    for lo, hi in ((0, 150), (cut // 2 - 75, cut // 2 + 75), (cut - 75, cut + 75), (rows - 150, rows)):
        np.testing.assert_array_equal(got[lo:hi].get(), expected[np.arange(lo, hi) % period])
