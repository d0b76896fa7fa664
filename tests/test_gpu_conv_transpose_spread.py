"""Transposed 1x1 convolutions at stride 2, whose pixels are spread over a plane of zeros: rows of each vector width, odd rows and columns, strides that differ, an
output that is larger than the pixels reach; against the oracle in whole numbers, which float16 sums exactly."""
import numpy as np
import pytest

import chainer_amd as chx
from oracle import native as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['float16', 'float32', 'float64'])
@pytest.mark.parametrize('h,w,stride,out', [(4, 4, 2, (8, 8)), (4, 4, 2, (7, 7)), (3, 6, 2, (6, 12)), (3, 7, 2, (5, 14)), (5, 1, 2, (10, 2)), (3, 4, (3, 2), (8, 8)),
                                            (3, 4, (1, 2), (3, 8)), (28, 28, 2, (56, 56)), (4, 4, (2, 3), (8, 12)), (3, 5, 2, (6, 8))])
def test_against_oracle(h, w, stride, out, dtype):
    rng = np.random.default_rng(h * w)
    x, f = rng.integers(-2, 3, (3, 24, h, w)).astype(dtype), rng.integers(-2, 3, (24, 17, 1, 1)).astype(dtype)
    b = rng.integers(-2, 3, 17).astype(dtype)
    X, F = chx.array(x), chx.array(f)
    try:
        ref = O.conv_transpose(x, f, b, stride, 0, out)
    except Exception:
        with pytest.raises(Exception):
            chx.conv_transpose(X, F, chx.array(b), stride, 0, out)
        return
    np.testing.assert_array_equal(chx.conv_transpose(X, F, chx.array(b), stride, 0, out).get(), ref)
    np.testing.assert_array_equal(chx.conv_transpose(X, F, None, stride, 0, out).get(), O.conv_transpose(x, f, None, stride, 0, out))
