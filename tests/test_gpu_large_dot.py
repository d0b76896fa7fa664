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
