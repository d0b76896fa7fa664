"""float32 3x3 convolutions that read NCHW in place (direct_conv.hip): planes that no tile divides, remainders of filters and of pixels, one chunk of channels to
several rounds of them, each split of the channels, a bias, and values that are not finite, against the oracle and in whole numbers."""
import numpy as np
import pytest

import chainer_amd as chx
from oracle import native as O
from helpers import assert_close

pytestmark = pytest.mark.gpu

SHAPES = [(1, 8, 1, 1, 1), (1, 64, 5, 7, 33), (3, 72, 9, 4, 32), (2, 16, 1, 70, 40), (5, 24, 33, 3, 65), (1, 200, 14, 14, 31),  # channels over 8 groups of waves
          (23, 40, 17, 19, 34), (9, 128, 31, 33, 96), (2, 136, 40, 41, 250),                                                    # 4
          (70, 8, 31, 30, 64), (36, 24, 29, 31, 65)]                                                                           # 2


@pytest.mark.parametrize('n,c,h,w,k', SHAPES)
def test_whole_numbers(n, c, h, w, k):
    rng = np.random.default_rng(c * h + w)
    x, f = rng.integers(-3, 4, (n, c, h, w)).astype(np.float32), rng.integers(-3, 4, (k, c, 3, 3)).astype(np.float32)
    b = rng.integers(-3, 4, k).astype(np.float32)
    assert chx.conv_route(chx.array(x), chx.array(f), None, 1, 1) == 6
    padded = np.pad(x, ((0, 0), (0, 0), (1, 1), (1, 1)))
    ref = np.zeros((n, k, h, w), np.float32)
    for r in range(3):
        for s in range(3):
            ref += np.tensordot(f[:, :, r, s], padded[:, :, r:r + h, s:s + w], (1, 1)).transpose(1, 0, 2, 3)
    np.testing.assert_array_equal(chx.conv(chx.array(x), chx.array(f), None, 1, 1).get(), ref)
    np.testing.assert_array_equal(chx.conv(chx.array(x), chx.array(f), chx.array(b), 1, 1, True).get(), ref + b[:, None, None])


@pytest.mark.parametrize('n,c,h,w,k', [(1, 64, 5, 7, 33), (7, 24, 33, 20, 65)])
def test_against_oracle(n, c, h, w, k):
    rng = np.random.default_rng(n)
    x, f = rng.standard_normal((n, c, h, w), dtype=np.float32), rng.standard_normal((k, c, 3, 3), dtype=np.float32)
    assert_close(chx.conv(chx.array(x), chx.array(f), None, 1, 1).get(), O.conv(x, f, None, 1, 1), 1e-5, 'conv')


def test_special_values_stay_where_they_are():
    x = np.ones((2, 8, 6, 7), np.float32)
    x[0, 1, 2, 0], x[1, 2, 5, 6], x[1, 7, 0, 3] = np.inf, np.nan, -np.inf
    f = np.ones((24, 8, 3, 3), np.float32)
    f[5, 0, 1, 1] = -np.inf
    np.testing.assert_array_equal(chx.conv(chx.array(x), chx.array(f), None, 1, 1).get(), O.conv(x, f, None, 1, 1))


def test_limits_of_the_route():
    def route(n, c, h, k, stride=1, pad=1, size=3):
        return chx.conv_route(chx.zeros((n, c, h, h), np.float32), chx.zeros((k, c, size, size), np.float32), None, stride, pad)
    assert route(6 * 256, 8, 8, 32 * 2) == 6 and route(6 * 256 + 1, 8, 8, 32 * 2) == 0  # 24 tiles of 32 x 32 to a compute unit, 256 of these
    assert route(2 * 256, 8, 8, 32 * 3) == 6 and route(2 * 256 + 1, 8, 8, 32 * 3) == 0    # 12 of them beyond 64 filters
    assert route(2, 12, 8, 64) == 0 and route(2, 8, 8, 64, stride=2) == 0 and route(2, 8, 8, 64, pad=0) == 0 and route(2, 8, 8, 64, size=5) == 0
    x = chx.zeros((2, 8, 9, 8), np.float32)
    assert chx.conv_route(x[:, :, 1:], chx.zeros((64, 8, 3, 3), np.float32), None, 1, 1) == 0


def test_filters_that_are_a_view_are_copied():
    rng = np.random.default_rng(5)
    x, f = rng.standard_normal((2, 16, 9, 8), dtype=np.float32), rng.standard_normal((16, 24, 3, 3), dtype=np.float32)
    flipped = chx.array(f)[:, :, ::-1, ::-1].transpose((1, 0, 2, 3))
    assert chx.conv_route(chx.array(x), flipped, None, 1, 1) == 6
    dense = chx.conv(chx.array(x), flipped.copy(), None, 1, 1).get()
    np.testing.assert_array_equal(chx.conv(chx.array(x), flipped, None, 1, 1).get(), dense)
    np.testing.assert_array_equal(chx.conv_transpose(chx.array(x), chx.array(f), None, 1, 1).get(), dense)
