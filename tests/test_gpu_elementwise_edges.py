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


def test_more_elements_than_a_launch_counts():
    """2^32 vectors in two rows that the operands walk apart: cut between the rows, then inside each."""
    import torch
    import chainer_amd as chx
    cols = (1 << 35) + 5
    if torch.cuda.mem_get_info()[0] < 3 * cols:
        pytest.skip('needs %d bytes of device memory' % (3 * cols))
    out = None
    try:
        out = chx.array(np.array([[3], [-7]], 'int8')).broadcast_to((2, cols)).copy()
        for row, value in enumerate((3, -7)):
            for lo in (0, cols // 4 - 500, cols // 2 - 500, 3 * (cols // 4) - 500, cols - 1000):
                assert_exact(out[row, lo:lo + 1000].get(), np.full(1000, value, 'int8'), 'row %d from %d' % (row, lo))
    finally:
        del out
        chx.synchronize()
        chx.free_unused_blocks()
