"""A step of L.LSTM in one launch: against the composition in float64, at the edges of tiles, chunks, row blocks and accumulator types."""
import numpy as np
import pytest

from helpers import assert_close

pytestmark = pytest.mark.gpu


def sigmoid(v):
    return 1 / (1 + np.exp(-v))


def reference(c, x, wx, b, h, wh):
    c, x, wx, h, wh = [a.astype('float64') for a in (c, x, wx, h, wh)]
    g = (x @ wx.T + (0 if b is None else b.astype('float64')) + h @ wh.T).reshape(c.shape + (4,))
    new_c = np.tanh(g[..., 0]) * sigmoid(g[..., 1]) + sigmoid(g[..., 2]) * c
    return sigmoid(g[..., 3]) * np.tanh(new_c), new_c


def arrays(rng, dt, rows, n_in, units):
    def arr(*shape, k=1.0):
        return (rng.standard_normal(shape) * k).astype(dt)
    return arr(rows, units), arr(rows, n_in), arr(4 * units, n_in, k=n_in ** -0.5), arr(4 * units), arr(rows, units), arr(4 * units, units, k=units ** -0.5)


@pytest.mark.parametrize('dt', ['float32', 'float16'])
@pytest.mark.parametrize('rows,n_in,units', [
    (1, 8, 8), (3, 9, 11), (16, 63, 64), (17, 64, 63), (33, 65, 67), (5, 257, 65),           # shortest reductions; double below 64 terms
    (1, 650, 650), (16, 97, 1025), (16, 130, 650), (17, 130, 650), (20, 31, 1023),           # one and two row blocks, widths 1 and 2
    (128, 333, 501), (128, 650, 649), (100, 1000, 16), (129, 64, 700), (300, 72, 300),       # widths 2, 3 and 4
    (1024, 70, 511), (4, 3, 20), (4, 20, 3), (0, 8, 8)])                                     # several tiles to a compute unit; composed
def test_matches_reference(dt, rows, n_in, units):
    import chainer_amd as chx
    c, x, wx, b, h, wh = arrays(np.random.default_rng(rows + n_in + units), dt, rows, n_in, units)
    # the gates' sums: up to 2000 products of about 1/sqrt(terms), each rounded to 2^-24 of partial sums of a few units; float16 rounds c and h to 2^-11, and a
    # composed call its gates as well
    tol = 4e-6 if dt == 'float32' else 6e-3
    for bias in (b, None):
        got = chx.lstm_step(chx.array(c), chx.array(x), chx.array(wx), None if bias is None else chx.array(bias), chx.array(h), chx.array(wh))
        for g, r, what in zip(got, reference(c, x, wx, bias, h, wh), 'hc'):
            assert g.dtype == np.dtype(dt) and g.shape == (rows, units)
            assert np.allclose(g.get().astype('float64'), r, rtol=tol, atol=tol), what


@pytest.mark.parametrize('dt', ['float32', 'float16'])
def test_views_special_values_and_what_is_composed(dt):
    import chainer_amd as chx
    rng = np.random.default_rng(5)
    c, x, wx, b, h, wh = arrays(rng, dt, 40, 75, 90)
    x[3, 5], h[7, 2], c[9, 1] = np.nan, np.inf, -np.inf
    X, H, WX, WH, C, B = [chx.array(a) for a in (x, h, wx, wh, c, b)]

    def composed(*a):
        return chx.lstm(a[0], chx.add(chx.linear(a[1], a[2], a[3]), chx.linear(a[4], a[5])))
    wide = chx.array(np.concatenate([x, x], 1))
    calls = [(C, X, WX, B, H, WH), (C, wide[:, 75:], WX, B, H, WH), (C[::-1], X[::-1], WX, B[::-1], H[::-1], WH),
             (C[1:, 3:], X[1:], WX[12:], B[12:], H[1:, 3:], WH[12:, 3:]), (C, X[:, ::-1], WX, B, H, WH), (C, X, WX, chx.zeros((1,), dt), H, WH)]
    for a in calls:
        for g, r in zip(chx.lstm_step(*a), composed(*a)):
            assert_close(g.get(), r.get(), 2e-6 if dt == 'float32' else 4e-3, 'views')
    with pytest.raises(chx.DimensionError):
        chx.lstm_step(C, X, WX[4:], B[4:], H, WH[4:])
    with pytest.raises(chx.DtypeError):
        chx.lstm_step(C, X.astype('float64'), WX, B, H, WH)


@pytest.mark.parametrize('dt,rows,n_in,units,taken', [
    ('float32', 128, 650, 650, True), ('float32', 768, 650, 650, True), ('float32', 1024, 650, 650, False),  # rounds of tiles x terms: 1300, 5200; too many tiles
    ('float32', 20, 5000, 300, True), ('float32', 20, 5001, 300, False),                                    # 5300 terms in one round
    ('float16', 20, 7500, 300, True), ('float16', 20, 7501, 300, False),                                    # 7800
    ('float32', 32, 910, 50, True), ('float32', 32, 911, 50, False), ('float16', 32, 911, 50, True),        # 960, in double
    ('float32', 4096, 50, 50, True), ('float32', 8192, 63, 63, False), ('float32', 128, 50, 2048, False),   # 700, 2016, 16784
    ('float32', 4, 3, 20, False), ('float16', 4, 20, 7, False)])                                            # rows shorter than 16 bytes
def test_what_is_taken(dt, rows, n_in, units, taken):
    import chainer_amd as chx
    from chainer_amd import _host
    c, x, wx, b, h, wh = [chx.zeros(s, dt) for s in ((rows, units), (rows, n_in), (4 * units, n_in), (4 * units,), (rows, units), (4 * units, units))]
    assert (_host.lstm_step_direct(c, x, wx, b, h, wh) is not None) == taken


@pytest.mark.parametrize('units', [64, 97, 127, 300])
@pytest.mark.parametrize('rows', [16, 1024])
def test_error_is_not_above_the_separate_calls(rows, units):
    import chainer_amd as chx
    wrong, composed = 0.0, 0.0
    for seed in range(1024 // rows):
        c, x, wx, b, h, wh = arrays(np.random.default_rng(seed), 'float32', rows, units, units)
        C, X, WX, B, H, WH = [chx.array(a) for a in (c, x, wx, b, h, wh)]
        ref = reference(c, x, wx, b, h, wh)
        for g, s, r in zip(chx.lstm_step(C, X, WX, B, H, WH), chx.lstm(C, chx.add(chx.linear(X, WX, B), chx.linear(H, WH))), ref):
            wrong += np.sum((g.get() - r) ** 2)
            composed += np.sum((s.get() - r) ** 2)
    assert wrong <= composed * 1.01  # sums over 65536 elements and more: 0.4 % of chance in either
