"""Reductions along one strided axis (the column kernels): bit for bit the oracle's tree at the edges of chunks, slices and vectors."""
import numpy as np
import pytest

from oracle import native as O
from helpers import assert_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt', ['float16', 'float32', 'float64', 'int32', 'int8'])
@pytest.mark.parametrize('rows,cols', [(32, 5), (33, 64), (35, 65), (127, 1001), (131, 3), (512, 130), (515, 17), (517, 260), (16 * 512 + 31, 33),
                                       (40000, 7), (70001, 2)])
def test_axis0(dt, rows, cols):
    import chainer_amd as chx
    rng = np.random.default_rng(rows + cols)
    x = rng.standard_normal((rows, cols)).astype(dt) if dt[0] == 'f' else rng.integers(-5, 6, (rows, cols)).astype(dt)
    if dt[0] == 'f':
        x[rows // 2, 0] = np.nan
    X = chx.array(x)
    with np.errstate(all='ignore'):
        assert_exact(chx.sum(X, 0).get(), O.sum(x, 0), 'sum')
        assert_exact(chx.amax(X, 0).get(), O.amax(x, 0), 'amax')
        assert_exact(chx.argmax(X, 0).get(), O.argmax(x, 0), 'argmax')


@pytest.mark.parametrize('dt', ['float16', 'float32'])
def test_middle_axis_and_views(dt):
    import chainer_amd as chx
    rng = np.random.default_rng(3)
    x = rng.standard_normal((5, 600, 37)).astype(dt)
    X = chx.array(x)
    assert_exact(chx.sum(X, 1).get(), O.sum(x, 1), 'middle axis')
    assert_exact(chx.argmax(X, 1).get(), O.argmax(x, 1), 'middle axis')
    y, Y = x[0], X[0]
    assert_exact(chx.sum(Y[:, 3:30], 0).get(), O.sum(y[:, 3:30], 0), 'rows off every alignment')
    assert_exact(chx.sum(Y[::-1, ::2], 0).get(), O.sum(y[::-1, ::2], 0), 'strided outputs, reversed axis')
    assert_exact(chx.sum(Y, 0, True).get(), O.sum(y, 0, True), 'keepdims')
