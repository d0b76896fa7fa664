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


@pytest.mark.parametrize('dt', ['float16', 'float32', 'float64'])
@pytest.mark.parametrize('rows,cols', [(64, 100), (65, 100), (256, 16), (257, 16), (5, 511), (5, 513), (3, 1024), (3, 1025), (2, 2049), (70, 2051),
                                       (1, 16385), (2, 40003), (255, 3000), (256, 3001), (258, 33001), (1, 700001),
                                       (1030, 1025), (1030, 2047), (1030, 2049), (512, 10), (513, 10), (256, 40), (257, 40), (64, 256), (65, 256), (32, 257),
                                       (33, 257)])
def test_softmax_cross_entropy_of_long_rows(dt, rows, cols):
    """Rows in a wave's registers, in a workgroup's, in segments of several; rows that start anywhere, labels at their ends."""
    import chainer_amd as chx
    rng = np.random.default_rng(rows * 31 + cols)
    wide = np.full((rows, cols + 3), np.nan, dt)
    x = wide[:, 1:1 + cols]
    x[...] = (3 * rng.standard_normal((rows, cols))).astype(dt)
    t = rng.integers(0, cols, rows).astype('int64')
    t[0], t[-1] = cols - 1, 0
    if rows > 2:
        t[1], t[2] = cols, -1  # name no class
        x[2] += 5
    x64 = x.astype(np.float64)
    top = x64.max(1)
    lse = top + np.log(np.exp(x64 - top[:, None]).sum(1))
    named = (t >= 0) & (t < cols)
    expected = (lse - x64[np.arange(rows), np.where(named, t, 0)])[named].mean()
    X, t_dev = chx.array(wide)[:, 1:1 + cols], chx.array(t)
    got = float(chx.softmax_cross_entropy(X, t_dev).get())
    # float16: a score of about 10 keeps 10 bits, the sum and the number of labels (rounded as the chain rounds them) 10 each
    assert abs(got - expected) <= {'float16': 4e-3, 'float32': 2e-6, 'float64': 1e-13}[dt] * expected, (got, expected)
    for at, value in ((cols // 2, -np.inf), (cols - 2, np.nan), (1, np.inf)):
        y = wide.copy()
        y[-1, 1 + at] = value
        assert np.isnan(float(chx.softmax_cross_entropy(chx.array(y)[:, 1:1 + cols], t_dev).get())), value
    y = wide.copy()
    y[0, 1:1 + cols] = -np.inf
    assert np.isnan(float(chx.softmax_cross_entropy(chx.array(y)[:, 1:1 + cols], t_dev).get()))


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


@pytest.mark.parametrize('m,k,n,dt', [(*mkn, dt) for mkn in [(1, 784, 10), (33, 65, 97), (3, 8, 5)] for dt in ('float16', 'float32', 'float64', 'int32')] +
                         [(*mkn, dt) for mkn in [(100, 1000, 1000), (130, 2048, 1000), (300, 4096, 64), (2100, 650, 2085)]
                          for dt in ('float16', 'float32')])
def test_linear_bias_in_the_product(m, k, n, dt):
    import chainer_amd as chx
    rng = np.random.default_rng(m + k + n)
    draw = (lambda *s: rng.integers(-3, 4, s).astype(dt)) if dt == 'int32' else (lambda *s: (rng.standard_normal(s) / np.sqrt(s[-1])).astype(dt))
    x, w, b = draw(m, k), draw(n, k), draw(2 * n)
    X, W, B = chx.array(x), chx.array(w), chx.array(b)
    got = chx.linear(X, W, B[::2])  # strided bias
    ref = chx.add(chx.dot(X, W.T), B[::2])
    assert_close(got.get(), ref.get(), 0 if dt == 'int32' else None, 'linear')
