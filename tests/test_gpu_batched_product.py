"""Weight gradients of float16 convolutions (batched_product.hip): remainders of 128-wide tiles and of 32-pixel chunks, one and many slices, planes read in
place, shifted and staged, against the oracle."""
import numpy as np
import pytest

import chainer_amd as chx
from oracle import native as O
from helpers import assert_close

pytestmark = pytest.mark.gpu

_CASES = [  # images, channels, height, width, filters, kernel, stride, pad
    (1, 1, 4, 8, 1, 1, 1, 0), (2, 129, 6, 6, 127, 1, 1, 0), (3, 40, 2, 17, 300, 1, 1, 0), (9, 64, 14, 14, 256, 1, 1, 0), (40, 33, 7, 10, 65, 1, 1, 0),
    (4, 130, 7, 7, 128, 1, 1, 0), (5, 64, 7, 7, 40, 1, 1, 0),  # odd planes: an even and an odd number of staged pixels
    (2, 3, 9, 11, 130, 3, 1, 1), (3, 64, 14, 14, 64, 3, 1, 1), (2, 20, 5, 5, 129, 3, 1, 0), (2, 8, 12, 10, 16, (1, 5), 1, (0, 2)),
    (2, 64, 14, 14, 130, 1, 2, 0), (2, 3, 30, 30, 64, 7, 2, 3), (1, 24, 13, 9, 24, 3, 2, 1),
]


@pytest.mark.parametrize('n,c,h,w,k,size,stride,pad', _CASES)
def test_against_oracle(n, c, h, w, k, size, stride, pad):
    kh, kw = size if isinstance(size, tuple) else (size, size)
    ph, pw = pad if isinstance(pad, tuple) else (pad, pad)
    rng = np.random.default_rng(c + h)
    oh, ow = (h + 2 * ph - kh) // stride + 1, (w + 2 * pw - kw) // stride + 1
    shape = (k, c, kh, kw)
    # whole numbers whose sums float16 holds: exact in any order
    x, gy = rng.integers(-1, 2, (n, c, h, w)).astype(np.float16), rng.integers(-1, 2, (n, k, oh, ow)).astype(np.float16)
    gw = chx.conv_grad_weight('float16', shape, chx.array(x), chx.array(gy), stride, (ph, pw), False).get()
    np.testing.assert_array_equal(gw, O.conv_grad_weight(shape, x, gy, stride, (ph, pw), False))
    # float sums of n * oh * ow products, rounded once: half an ulp of float16 and the order of the sums
    x, gy = rng.standard_normal(x.shape).astype(np.float16), rng.standard_normal(gy.shape).astype(np.float16)
    gw = chx.conv_grad_weight('float16', shape, chx.array(x), chx.array(gy), stride, (ph, pw), False).get()
    assert_close(gw, O.conv_grad_weight(shape, x, gy, stride, (ph, pw), False), 2e-3, 'gradient')


@pytest.mark.parametrize('n,h,w,size,pad', [(3, 6, 7, 1, 0), (3, 7, 7, 1, 0), (3, 6, 7, 3, 1)])
def test_special_values_stay_where_they_are(n, h, w, size, pad):
    """An Inf or NaN reaches its own channel's or filter's gradients, not those of the rows beside it."""
    rng = np.random.default_rng(h)
    x, gy = rng.integers(1, 3, (n, 40, h, w)).astype(np.float16), rng.integers(1, 3, (n, 36, h, w)).astype(np.float16)
    x[1, 5, 0, 0], x[0, 7, h - 1, w - 1], gy[2, 3, 0, 0], gy[0, 35, 0, 0] = np.inf, np.nan, np.inf, np.nan
    shape = (36, 40, size, size)
    gw = chx.conv_grad_weight('float16', shape, chx.array(x), chx.array(gy), 1, pad, False).get()
    np.testing.assert_array_equal(gw, O.conv_grad_weight(shape, x, gy, 1, pad, False))
