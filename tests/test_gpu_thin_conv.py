"""Convolutions of at most 32 terms (thin_conv.hip): one term to 32, remainders of pixel blocks and of 64 filters, strides, padding, cover_all,
rectangular filters and a bias, against the oracle."""
import numpy as np
import pytest

import chainer_amd as chx
from oracle import native as O
from helpers import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt,tol', [('float32', 32 * 2.0 ** -23), ('float16', 2.0 ** -10)])  # 32 terms, each rounded twice at most; an ulp
@pytest.mark.parametrize('n,c,h,w,k,kh,kw,stride,pad,cover_all', [
    (3, 3, 32, 32, 64, 3, 3, 1, 1, False), (2, 1, 28, 28, 20, 5, 5, 1, 0, False), (1, 1, 5, 5, 16, 1, 1, 1, 0, False), (2, 3, 9, 11, 130, 3, 3, 2, 1, True),
    (5, 2, 7, 13, 65, 4, 4, 3, 2, False), (2, 4, 6, 6, 33, 2, 4, 1, (3, 0), False), (1, 16, 3, 50, 70, 2, 1, (1, 2), 0, True), (7, 3, 1, 1, 96, 3, 3, 1, 1, False),
])
def test_against_oracle(dt, tol, n, c, h, w, k, kh, kw, stride, pad, cover_all):
    rng = np.random.default_rng(c * h + w)
    x, f = rng.standard_normal((n, c, h, w)).astype(dt), rng.standard_normal((k, c, kh, kw)).astype(dt)
    bias = rng.standard_normal(k).astype(dt)
    for b in (None, bias):
        got = chx.conv(chx.array(x), chx.array(f), None if b is None else chx.array(b), stride, pad, cover_all).get()
        assert_close(got, O.conv(x, f, b, stride, pad, cover_all), tol, 'conv')
    # whole numbers: exact in any order
    xi, fi = rng.integers(-3, 4, x.shape).astype(dt), rng.integers(-3, 4, f.shape).astype(dt)
    np.testing.assert_array_equal(chx.conv(chx.array(xi), chx.array(fi), None, stride, pad, cover_all).get(), O.conv(xi, fi, None, stride, pad, cover_all))


def test_special_values_stay_where_they_are():
    x = np.ones((2, 3, 6, 7), np.float32)
    x[0, 1, 2, 0], x[1, 2, 5, 6] = np.inf, np.nan
    f = np.ones((24, 3, 3, 3), np.float32)
    f[5, 0, 1, 1] = -np.inf
    np.testing.assert_array_equal(chx.conv(chx.array(x), chx.array(f), None, 1, 1).get(), O.conv(x, f, None, 1, 1))


@pytest.mark.parametrize('dt', ['float32', 'float16'])
def test_route(dt):
    x = chx.zeros((4, 3, 12, 12), dt)
    assert chx.conv_route(x, chx.zeros((64, 3, 3, 3), dt), None, 1, 1) == 5
    assert chx.conv_route(x, chx.zeros((64, 3, 4, 4), dt), None, 1, 1) == 0
    assert chx.conv_route(x, chx.zeros((8, 3, 3, 3), dt), None, 1, 1) == 0
