"""Reductions and log-softmax of short rows: several rows to a workgroup, or a wave or workgroup that holds one in registers.

Reductions are bit for bit the oracle's tree.  log-softmax is x - (m + log(sum exp(x - m))): the chain of the same type on the oracle differs by the rounding of
its own steps, which the float tolerance of the other log-softmax tests covers."""
import numpy as np
import pytest

from oracle import native as O
from helpers import assert_close, assert_exact

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


@pytest.mark.parametrize('dt', ['float16', 'float32', 'float64'])
@pytest.mark.parametrize('rows,n', [(5, 129), (2047, 255), (2048, 257), (2049, 511), (2050, 1023), (2048, 1025), (2051, 2047), (2048, 4095), (3, 4097), (70, 10241),
                                    (64, 16385), (65, 16385), (1, 32769), (2, 70001)])
def test_log_softmax(dt, rows, n):
    import chainer_amd as chx
    x = (np.random.default_rng(rows + n).standard_normal((rows, n + 1)) * 3).astype(dt)
    x[rows // 2, n // 3] = 60000 if dt == 'float16' else 1e30
    X = chx.array(x)
    assert_close(chx.log_softmax_fused(X).get(), O.log_softmax(x, 1), None, 'rows')
    x = x[:, 1:]
    assert_close(chx.log_softmax_fused(X[:, 1:]).get(), O.log_softmax(x, 1), None, 'rows that start anywhere')


def test_log_softmax_in_place_and_in_a_smaller_workspace():
    import chainer_amd as chx
    rng = np.random.default_rng(4)
    for rows, n in ((2100, 1001), (3, 2001), (2, 20001), (1, 100003)):
        x = rng.standard_normal((rows, n)).astype('float32')
        X = chx.array(x)
        ref = chx.log_softmax_fused(X).get()
        need = -(-n // (64 * 1024 // 4)) * rows * 2 * 4 if n > 16384 else 0  # what segments of 64 KiB take
        ws = chx.empty((max(need, 1),), 'uint8')
        chx._lib.call('hipcx_log_softmax', X.desc(), X.desc(), ws.data_ptr if need else None, need, chx.routines.current_stream())
        # other segments add the exponentials in another order: a few roundings of a sum, of which the logarithm is taken
        assert_close(X.get(), ref, 1e-5, 'in place %d x %d' % (rows, n))
