"""float16 3x3 convolutions of a few hundred 64 x 64 tiles (mid_conv.hip): planes of odd and even sizes that tiles divide nowhere, remainders of filters and of the
chunks that waves share, both numbers of waves, filters of every stride the packing tells apart, the fused tail, and the limits of the choice."""
import numpy as np
import pytest
import torch

import chainer_amd as chx
from oracle import native as O
from helpers import assert_close

pytestmark = pytest.mark.gpu

CASES = [  # images, channels, height, width, filters
    (45, 64, 7, 7, 330), (61, 144, 5, 5, 200), (300, 16, 3, 3, 320), (65, 32, 2, 4, 520), (70, 48, 2, 10, 520), (7, 128, 14, 14, 260), (5, 16, 31, 17, 257),
    (4, 64, 56, 56, 64), (3, 32, 21, 62, 200), (11, 272, 13, 11, 129), (100, 512, 7, 7, 66),
    (30, 512, 7, 7, 520),  # two tiles to a compute unit
]


def reference(x, f):
    return torch.nn.functional.conv2d(torch.from_numpy(x.astype(np.float32)), torch.from_numpy(f.astype(np.float32)), padding=1).numpy().astype(np.float16)


@pytest.mark.parametrize('n,c,h,w,k', CASES)
def test_whole_numbers(n, c, h, w, k):
    rng = np.random.default_rng(c + h)
    x, f = rng.integers(-2, 3, (n, c, h, w)).astype(np.float16), rng.integers(-1, 2, (k, c, 3, 3)).astype(np.float16)
    b = rng.integers(-3, 4, k).astype(np.float16)
    X, ref = chx.array(x), reference(x, f)  # (sums below 2048: exact in float16 and in any order)
    assert chx.conv_route(X, chx.array(f), None, 1, 1) == 7
    flipped = chx.array(np.ascontiguousarray(f[:, :, ::-1, ::-1]))[:, :, ::-1, ::-1]
    swapped = chx.array(np.ascontiguousarray(f.transpose(1, 0, 2, 3)[:, :, ::-1, ::-1])).transpose(1, 0, 2, 3)[:, :, ::-1, ::-1]
    columns = chx.array(np.ascontiguousarray(f.transpose(0, 1, 3, 2))).transpose(0, 1, 3, 2)
    for F in (chx.array(f), flipped, swapped, columns):
        np.testing.assert_array_equal(chx.conv(X, F, None, 1, 1).get(), ref)
    np.testing.assert_array_equal(chx.conv(X, chx.array(f), chx.array(b), 1, 1).get(), (ref.astype(np.float32) + b[:, None, None]).astype(np.float16))


@pytest.mark.parametrize('n,c,h,w,k', [(45, 64, 7, 7, 330), (7, 128, 14, 14, 260), (30, 512, 7, 7, 520)])
def test_fused_tail(n, c, h, w, k):
    rng = np.random.default_rng(n)
    x, f = rng.standard_normal((n, c, h, w)).astype(np.float16), (rng.standard_normal((k, c, 3, 3)) / np.sqrt(9 * c)).astype(np.float16)
    bn = [rng.uniform(0.5, 1.5, k).astype(np.float16) for _ in range(4)]
    y = reference(x, f)
    assert_close(chx.conv(chx.array(x), chx.array(f), None, 1, 1).get(), y, 2e-3, 'conv')
    gamma, beta, mean, var = (a.astype(np.float32)[None, :, None, None] for a in bn)
    expected = (y.astype(np.float32) - mean) / np.sqrt(var + 2e-5) * gamma + beta
    for residual in (None, rng.standard_normal(y.shape).astype(np.float16)):
        got = chx.conv_bn_act(chx.array(x), chx.array(f), None, 1, 1, False, [chx.array(a) for a in bn], 2e-5, None if residual is None else chx.array(residual), True).get()
        total = expected if residual is None else expected + residual.astype(np.float32)
        assert_close(got, np.maximum(total, 0).astype(np.float16), 4e-3, 'fused')


def test_special_values_stay_where_they_are():
    x = np.ones((45, 16, 7, 7), np.float16)
    x[0, 5, 3, 0], x[1, 6, 0, 6], x[44, 15, 6, 6], x[2, 0, 0, 0] = np.inf, np.nan, -np.inf, np.nan
    f = np.ones((330, 16, 3, 3), np.float16)
    np.testing.assert_array_equal(chx.conv(chx.array(x), chx.array(f), None, 1, 1).get(), O.conv(x, f, None, 1, 1))


def test_limits_of_the_choice():
    def route(n, c, h, k):
        return chx.conv_route(chx.zeros((n, c, h, h), np.float16), chx.zeros((k, c, 3, 3), np.float16), None, 1, 1)
    assert route(256, 64, 8, 128) == 7 and route(257, 64, 8, 128) == 1    # 512 tiles
    assert route(384, 272, 8, 128) == 7 and route(385, 272, 8, 128) == 1  # 768
    assert route(16, 512, 7, 256) == 4 and route(17, 512, 7, 256) == 7    # 256 tiles of 32 x 32
    assert route(51, 64, 8, 128) == 4 and route(52, 64, 8, 128) == 7      # 409
