"""float16 convolutions of few output pixels (small_conv.hip): odd and tiny planes, remainders of pixel and channel tiles, strides, several images and
the fused tail, against the oracle."""
import numpy as np
import pytest

import chainer_amd as chx
from oracle import native as O
from helpers import assert_close

pytestmark = pytest.mark.gpu

_CASES = [  # images, channels, height, width, filters, kernel, stride
    (1, 32, 7, 7, 64, 1, 1), (2, 96, 5, 3, 33, 1, 1), (1, 544, 14, 14, 40, 1, 1), (3, 64, 1, 1, 70, 1, 1), (1, 64, 9, 12, 100, 1, 2),
    (2, 32, 13, 8, 31, 1, 3), (1, 1024, 2, 2, 256, 1, 1), (1, 64, 30, 31, 128, 1, 1),
    (1, 16, 7, 7, 32, 3, 1), (2, 48, 14, 14, 33, 3, 1), (1, 144, 9, 5, 65, 3, 1), (3, 32, 2, 2, 40, 3, 1), (1, 64, 56, 56, 64, 3, 1),
    (1, 32, 3, 62, 20, 3, 1), (1, 16, 40, 6, 16, 3, 1), (2, 512, 7, 7, 64, 3, 1), (1, 256, 1, 34, 8, 3, 1),
    (1, 256, 1, 33, 8, 3, 1),  # (beyond what the NCHW kernels plan for: the general kernel)
]


@pytest.mark.parametrize('n,c,h,w,k,size,stride', _CASES)
def test_against_oracle(n, c, h, w, k, size, stride):
    rng = np.random.default_rng(c + h)
    x = rng.standard_normal((n, c, h, w)).astype(np.float16)
    f = (rng.standard_normal((k, c, size, size)) / np.sqrt(c * size * size)).astype(np.float16)
    b = rng.standard_normal(k).astype(np.float16)
    pad = size // 2
    X, F, B = chx.array(x), chx.array(f), chx.array(b)
    assert_close(chx.conv(X, F, B, stride, pad).get(), O.conv(x, f, b, stride, pad), 2e-3, 'conv')
    # whole numbers: exact in any order
    xi, fi = rng.integers(-2, 3, x.shape).astype(np.float16), rng.integers(-1, 2, f.shape).astype(np.float16)
    np.testing.assert_array_equal(chx.conv(chx.array(xi), chx.array(fi), None, stride, pad).get(), O.conv(xi, fi, None, stride, pad))
    bn = [rng.uniform(0.5, 1.5, k).astype(np.float16) for _ in range(4)]
    y = O.conv(x, f, None, stride, pad)
    r = rng.standard_normal(y.shape).astype(np.float16)
    got = chx.conv_bn_act(X, F, None, stride, pad, False, [chx.array(a) for a in bn], 2e-5, chx.array(r), True).get()
    gamma, beta, mean, var = (a.astype(np.float32)[None, :, None, None] for a in bn)
    expected = np.maximum((y.astype(np.float32) - mean) / np.sqrt(var + 2e-5) * gamma + beta + r.astype(np.float32), 0)
    assert_close(got, expected.astype(np.float16), 4e-3, 'fused')


@pytest.mark.parametrize('n,c,h,w,k,size,stride', [(1, 64, 7, 7, 64, 3, 1), (1, 64, 7, 7, 40, 1, 1), (1, 64, 14, 14, 40, 1, 1)])
def test_special_values_stay_where_they_are(n, c, h, w, k, size, stride):
    x = np.ones((n, c, h, w), np.float16)
    x[0, 5, 3, 0], x[0, 6, 0, w - 1] = np.inf, np.nan
    f = np.ones((k, c, size, size), np.float16)
    pad = size // 2
    np.testing.assert_array_equal(chx.conv(chx.array(x), chx.array(f), None, stride, pad).get(), O.conv(x, f, None, stride, pad))


def test_route():
    """conv_route names these kernels, and the large tiles where those take over."""
    def route(n, c, h, w, k, size, stride):
        return chx.conv_route(chx.zeros((n, c, h, w), np.float16), chx.zeros((k, c, size, size), np.float16), None, stride, size // 2)

    assert [route(*case) for case in _CASES] == [4] * (len(_CASES) - 1) + [0]
    assert route(32, 64, 56, 56, 64, 3, 1) == route(32, 512, 28, 28, 256, 1, 2) == 1


@pytest.mark.parametrize('size', [1, 3])
def test_filters_that_are_a_view(size):
    rng = np.random.default_rng(size)
    x, f = (rng.standard_normal(s).astype(np.float16) for s in ((2, 64, 7, 7), (64, 40, size, size)))
    view = chx.array(f).transpose((1, 0, 2, 3))[:, :, ::-1, ::-1]
    X, pad = chx.array(x), size // 2
    np.testing.assert_array_equal(chx.conv(X, view, None, 1, pad).get(), chx.conv(X, view.copy(), None, 1, pad).get())
    assert_close(chx.conv(X, view, None, 1, pad).get(), O.conv(x, f.transpose((1, 0, 2, 3))[:, :, ::-1, ::-1], None, 1, pad), 2e-3, 'conv')


@pytest.mark.parametrize('n,c,h,w,k,stride', [(2, 32, 8, 8, 16, 2), (1, 64, 8, 9, 40, 3), (1, 32, 7, 8, 33, 2), (1, 32, 8, 7, 33, 2), (64, 64, 56, 56, 128, 2)])
def test_cover_all_reaches_beyond_the_plane(n, c, h, w, k, stride):
    """Outputs whose only pixel lies behind the last row or column are the bias (the last case has the size of NchwConvKernel's)."""
    rng = np.random.default_rng(h)
    x, f = rng.integers(-2, 3, (n, c, h, w)).astype(np.float16), rng.integers(-1, 2, (k, c, 1, 1)).astype(np.float16)
    b = rng.integers(-3, 4, k).astype(np.float16)
    X, F, B = chx.array(x), chx.array(f), chx.array(b)
    expected = O.conv(x, f, b, stride, 0, True)
    assert (expected[:, :, -1, -1] == b).all()
    np.testing.assert_array_equal(chx.conv(X, F, B, stride, 0, True).get(), expected)
    bn = [np.ones(k, np.float16) for _ in range(4)]
    got = chx.conv_bn_act(X, F, B, stride, 0, True, [chx.array(a) for a in bn], 0.0, None, True).get()
    np.testing.assert_array_equal(got, np.maximum(expected, 0))
