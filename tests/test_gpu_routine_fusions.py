"""Routines that run as one kernel instead of the reference's chain (Linear's bias, Sigmoid, LogSoftmax of short rows, softmax cross
entropy) against the oracle's chains, at the sizes where their dispatch changes."""
import numpy as np
import pytest

from oracle import native as O
from helpers import assert_close, assert_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt', ['float16', 'float32', 'float64'])
@pytest.mark.parametrize('rows,cols', [(1, 1), (100, 10), (3, 16), (129, 17), (1000, 16), (257, 64), (70, 129), (40, 5000)])
def test_softmax_cross_entropy(dt, rows, cols):
    import chainer_amd as chx
    rng = np.random.default_rng(rows * 10007 + cols)
    x = (3 * rng.standard_normal((rows, cols))).astype(dt)
    t = rng.integers(0, cols, rows).astype('int32')
    if rows > 2:
        t[1] = -1  # selects nothing and does not count
    got = chx.softmax_cross_entropy(chx.array(x), chx.array(t)).get()
    ref = O.softmax_cross_entropy(x, t)
    assert got.shape == () and got.dtype == x.dtype
    assert_close(got.reshape(1), np.asarray(ref).reshape(1), what='softmax_cross_entropy')
    if cols > 1:
        x[0, (t[0] + 1) % cols] = -np.inf  # 0 * -inf in the masked sum
        assert np.isnan(chx.softmax_cross_entropy(chx.array(x), chx.array(t)).get())


@pytest.mark.parametrize('t_dtype', ['int8', 'uint8', 'int64'])
def test_softmax_cross_entropy_label_dtypes(t_dtype):
    import chainer_amd as chx
    rng = np.random.default_rng(5)
    for cols in (127, 300):  # 300 classes do not fit the 8-bit labels: the chain
        x = rng.standard_normal((20, cols)).astype('float32')
        t = rng.integers(0, 100, 20).astype(t_dtype)
        ref = O.softmax_cross_entropy(x, t)
        assert_close(chx.softmax_cross_entropy(chx.array(x), chx.array(t)).get().reshape(1), np.asarray(ref).reshape(1), what=t_dtype)


@pytest.mark.parametrize('cols', [1, 2])
def test_softmax_cross_entropy_float_labels(cols):
    """The chain compares labels of any numeric dtype with Arange(n) of that dtype."""
    import chainer_amd as chx
    x = np.random.default_rng(6).standard_normal((20, cols)).astype('float32')
    t = np.array([0, 1] * 10).astype('float32')
    ref = O.softmax_cross_entropy(x, t)
    assert_close(chx.softmax_cross_entropy(chx.array(x), chx.array(t)).get().reshape(1), np.asarray(ref).reshape(1), what='float labels')


@pytest.mark.parametrize('dt', ['float16', 'float32', 'float64'])
@pytest.mark.parametrize('cols', [1, 4, 16, 17, 64, 65, 128, 129])
def test_log_softmax_short_rows(dt, cols):
    import chainer_amd as chx
    x = (4 * np.random.default_rng(cols).standard_normal((131, cols))).astype(dt)
    x[5] = -np.inf
    if cols > 2:
        x[7, 1] = np.nan
        x[8, 2] = -np.inf
    with np.errstate(all='ignore'):
        ref = O.log_softmax(x, 1)
    got = chx.log_softmax(chx.array(x), 1).get()
    fine = np.isfinite(ref)
    assert np.array_equal(fine, np.isfinite(got))
    assert_close(got[fine], ref[fine], what='log_softmax')


@pytest.mark.parametrize('dt', ['float16', 'float32', 'float64'])
def test_sigmoid_equals_its_chain(dt):
    import chainer_amd as chx
    x = np.concatenate([np.linspace(-20, 20, 4097), [np.inf, -np.inf, np.nan, 0.0, -0.0, 60000.0, -60000.0]]).astype(dt)
    X = chx.array(x)
    chain = chx.reciprocal(chx.add(chx.exp(chx.negative(X)), 1))
    assert_exact(chx.sigmoid(X).get(), chain.get(), 'sigmoid')


@pytest.mark.parametrize('dt', ['float16', 'float32', 'float64', 'int32'])
@pytest.mark.parametrize('m,k,n', [(1, 784, 10), (33, 65, 97), (100, 1000, 1000), (3, 8, 5), (130, 2048, 1000), (300, 4096, 64), (2100, 650, 2085)])
def test_linear_bias_in_the_product(dt, m, k, n):
    import chainer_amd as chx
    if dt in ('float64', 'int32') and m * k * n > 5e7:
        pytest.skip('size meant for the float16 / float32 kernels')
    rng = np.random.default_rng(m + k + n)
    draw = (lambda *s: rng.integers(-3, 4, s).astype(dt)) if dt == 'int32' else (lambda *s: (rng.standard_normal(s) / np.sqrt(s[-1])).astype(dt))
    x, w, b = draw(m, k), draw(n, k), draw(2 * n)
    X, W, B = chx.array(x), chx.array(w), chx.array(b)
    got = chx.linear(X, W, B[::2])  # strided bias
    ref = chx.add(chx.dot(X, W.T), B[::2])
    assert_close(got.get(), ref.get(), 0 if dt == 'int32' else None, 'linear')
