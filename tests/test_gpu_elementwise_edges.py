"""Element-wise kernels at widths and offsets that no vector divides: the overlapping last vector of a row, in place too."""
import numpy as np
import pytest

from helpers import assert_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt', ['float16', 'float32', 'float64', 'int8', 'bool'])
@pytest.mark.parametrize('rows,cols', [(1, 1), (1, 3), (1, 7), (1, 8), (1, 17), (3, 15), (5, 33), (333, 1001), (2, 262147), (7, 300001)])
def test_odd_widths(dt, rows, cols):
    import chainer_amd as chx
    rng = np.random.default_rng(rows * 7 + cols)
    x = rng.integers(-4, 5, (rows, cols)).astype(dt)
    b = rng.integers(-4, 5, cols).astype(dt)
    X, B = chx.array(x), chx.array(b)
    add = (lambda p, q: p | q) if dt == 'bool' else (lambda p, q: p + q)
    assert_exact(chx.add(X, B).get(), add(x, b), 'row broadcast')
    assert_exact(chx.add(X, X[:, :1]).get(), add(x, x[:, :1]), 'column broadcast')
    assert_exact(chx.add(X[:, 1:], X[:, :-1]).get(), add(x[:, 1:], x[:, :-1]), 'shifted views')
    assert_exact(chx.multiply(X, B).get(), (x & b) if dt == 'bool' else x * b, 'multiply')
    assert_exact(X[:, ::-1].copy().get(), x[:, ::-1], 'reversed')
    Y = X.copy()
    Y += B
    assert_exact(Y.get(), add(x, b), 'in place')
    Z = X.copy()
    V = Z[:, 1:]
    V += X[:, 1:]
    z = x.copy()
    z[:, 1:] = add(x[:, 1:], x[:, 1:])
    assert_exact(Z.get(), z, 'in place on a misaligned view, nothing written outside')
    if dt[0] == 'f':
        assert_exact(chx.relu(X).get(), np.maximum(x, 0).astype(dt), 'relu')
        assert_exact(X.astype('float32').get(), x.astype('float32'), 'cast')
        assert_exact(chx.where(chx.greater(X, B), X, 1).get(), np.where(x > b, x, np.array(1, dt)), 'bool condition')
