"""Reductions of short rows, several of which share a workgroup: bit for bit the oracle's tree."""
import numpy as np
import pytest

from oracle import native as O
from helpers import assert_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt', ['float16', 'float32', 'float64', 'int32', 'int8', 'bool'])
@pytest.mark.parametrize('rows,n', [(9, 8), (8193, 19), (8200, 20), (70, 31), (33, 32), (77, 35), (31, 255), (255, 256), (257, 256), (1023, 257), (1025, 257),
                                    (1030, 1023), (1024, 1024), (2049, 1025), (2050, 2047), (2048, 2048), (2048, 2049)])
def test_rows(dt, rows, n):
    import chainer_amd as chx
    rng = np.random.default_rng(rows + n)
    if dt == 'bool':
        x = rng.random((rows, n)) > 0.9
    elif dt[0] == 'f':
        x = rng.standard_normal((rows, n)).astype(dt)
        x[::3] = rng.integers(0, 3, x[::3].shape)  # ties
        x[1::3][rng.random(x[1::3].shape) < 2 / n] = np.nan
        x[0], x[2, -1] = np.nan, np.inf
    else:
        x = rng.integers(-100, 100, (rows, n)).astype(dt)
    X = chx.array(x)
    with np.errstate(all='ignore'):
        for op in ('sum', 'amax', 'argmax'):
            assert_exact(getattr(chx, op)(X, 1).get(), getattr(O, op)(x, 1), op)
            assert_exact(getattr(chx, op)(X[:, 1:n - 2], 1).get(), getattr(O, op)(x[:, 1:n - 2], 1), op + ' of rows that start anywhere')
        assert_exact(chx.sum(X[::2], 1, True).get(), O.sum(x[::2], 1, True), 'every other row')
        assert_exact(chx.argmax(X[::-1], 1).get(), O.argmax(x[::-1], 1), 'rows in reverse')


def test_outputs_of_two_axes():
    import chainer_amd as chx
    x = np.random.default_rng(1).standard_normal((21, 100, 301)).astype('float32')
    X = chx.array(x)
    assert_exact(chx.sum(X, 2).get(), O.sum(x, 2), 'sum')
    assert_exact(chx.argmax(X[:, 3:90, 5:], 2).get(), O.argmax(x[:, 3:90, 5:], 2), 'argmax of a slice')
