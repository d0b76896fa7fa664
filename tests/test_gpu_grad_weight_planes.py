"""Weight gradients of float16 and float32 filters larger than 1x1 from zero-padded planes: rows that end with the next one's padding, odd and even widths,
windows that begin in either copy, padding wider than the filter, planes of each group of threads; whole numbers, exact in any order, against the oracle."""
import numpy as np
import pytest

import chainer_amd as chx
from oracle import native as O

pytestmark = pytest.mark.gpu

_CASES = [  # images, channels, height, width, filters, kernel, pad
    (3, 40, 7, 7, 36, (3, 3), (1, 1)), (2, 33, 14, 14, 20, (3, 3), (1, 1)), (2, 17, 28, 29, 8, (3, 3), (1, 1)), (1, 5, 56, 56, 9, (3, 3), (1, 1)),
    (2, 6, 12, 11, 8, (3, 3), (0, 0)), (2, 6, 12, 12, 8, (5, 5), (2, 2)), (2, 6, 9, 8, 8, (4, 7), (0, 3)), (2, 6, 9, 8, 8, (2, 6), (1, 0)),
    (2, 6, 9, 9, 8, (3, 2), (1, 3)), (2, 6, 9, 10, 8, (3, 1), (1, 0)), (2, 6, 9, 10, 8, (3, 1), (1, 2)), (3, 6, 4, 4, 8, (3, 3), (1, 1)), (300, 2, 7, 7, 3, (3, 3), (1, 1)),
]


@pytest.mark.parametrize('dtype', ['float16', 'float32'])
@pytest.mark.parametrize('n,c,h,w,k,size,pad', _CASES)
def test_against_oracle(n, c, h, w, k, size, pad, dtype):
    rng = np.random.default_rng(c + h)
    shape = (k, c) + size
    x = rng.integers(-1, 2, (n, c, h, w)).astype(dtype)
    gy = rng.integers(-1, 2, (n, k, h + 2 * pad[0] - size[0] + 1, w + 2 * pad[1] - size[1] + 1)).astype(dtype)
    gw = chx.conv_grad_weight(dtype, shape, chx.array(x), chx.array(gy), 1, pad, False).get()
    np.testing.assert_array_equal(gw, O.conv_grad_weight(shape, x, gy, 1, pad, False))
    # an Inf in the last image's first channel and a NaN in the last pixel of another reach the taps that the oracle gives them to, no neighbours
    x[n - 1, 0, 0, 0], x[0, c - 1, h - 1, w - 1] = np.inf, np.nan
    gw = chx.conv_grad_weight(dtype, shape, chx.array(x), chx.array(gy), 1, pad, False).get()
    np.testing.assert_array_equal(gw, O.conv_grad_weight(shape, x, gy, 1, pad, False))


@pytest.mark.parametrize('dtype', ['float16', 'float32'])
@pytest.mark.parametrize('n,c,h,w,k,size,pad', [
    (1, 2, 70, 131, 3, (3, 3), (1, 1)), (2, 1, 129, 64, 5, (3, 3), (0, 1)),   # several workgroups to a plane
    (2, 3, 40, 41, 90, (3, 3), (1, 1)), (2, 3, 40, 40, 90, (2, 3), (1, 0)),   # rows of gy of an odd and of an even number
    (3, 5, 90, 3, 4, (3, 3), (1, 0)), (3, 5, 90, 3, 4, (3, 2), (1, 0)),       # of one and of two
    (65, 3, 7, 7, 4, (3, 3), (1, 1)), (130, 40, 7, 7, 30, (3, 3), (1, 1))])   # more flags of a channel than lanes; two pieces to a thread
def test_parts_of_planes_and_rows_of_gy(n, c, h, w, k, size, pad, dtype):
    test_against_oracle(n, c, h, w, k, size, pad, dtype)
    # the last part of the last plane flags its channel
    rng = np.random.default_rng(w)
    shape = (k, c) + size
    x = rng.integers(-1, 2, (n, c, h, w)).astype(dtype)
    gy = rng.integers(-1, 2, (n, k, h + 2 * pad[0] - size[0] + 1, w + 2 * pad[1] - size[1] + 1)).astype(dtype)
    x[n - 1, c - 1, h - 1, w - 1] = np.inf
    gw = chx.conv_grad_weight(dtype, shape, chx.array(x), chx.array(gy), 1, pad, False).get()
    np.testing.assert_array_equal(gw, O.conv_grad_weight(shape, x, gy, 1, pad, False))
