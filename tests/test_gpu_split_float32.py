"""float32 products and convolutions on the bfloat16 matrix pipes (igemm_split.hip): edges of tiles and steps, rows of 8- and 16-byte pieces, split
reductions, both orientations of the result, and operands whose tile is computed again on the float pipe."""
import numpy as np
import pytest

import chainer_amd as chx
from chainer_amd import _lib
from chainer_amd._array import current_stream

pytestmark = pytest.mark.gpu

# A sum of K float products in any order, each and each partial sum rounded once, is within K 2^-24 of the sum of magnitudes (to first order); what the
# split leaves out of a product is at most 2^-34 of it.
_EPS = 2.0 ** -24


def _check(got, x, w):
    x, w = x.astype(np.float64), w.astype(np.float64)
    bound = (x.shape[1] + 4) * _EPS * (np.abs(x) @ np.abs(w.T)) + 1e-300
    np.testing.assert_array_less(np.abs(got.astype(np.float64) - x @ w.T), bound)


@pytest.mark.parametrize('m,k,n', [(2048, 64, 1024), (2049, 650, 1153), (1793, 66, 1025), (4000, 17 * 2, 700), (4097, 2, 640), (1500, 4098, 1300), (300, 4096, 300),
                                   (20001, 66, 40), (20001, 64, 33), (100, 42, 90), (100, 36, 130)])
def test_products(m, k, n):
    rng = np.random.default_rng(k)
    # magnitudes over thirty powers of two: every part of an operand matters
    x = rng.standard_normal((m, k), dtype=np.float32) * np.exp2(rng.integers(-15, 16, (m, k))).astype(np.float32)
    w = rng.standard_normal((n, k), dtype=np.float32)
    _check(chx.linear(chx.array(x), chx.array(w)).get(), x, w)
    xt = chx.array(np.ascontiguousarray(x.T)).T  # laid out anew
    _check(chx.linear(xt, chx.array(w)).get(), x, w)


def test_reduction_of_transposed_operands_is_split():
    rng = np.random.default_rng(1)
    x, g = rng.standard_normal((6001, 1000), dtype=np.float32), rng.standard_normal((6001, 700), dtype=np.float32)
    _check(chx.dot(chx.array(x).T, chx.array(g)).get(), x.T, g.T)


@pytest.mark.parametrize('shape,filters,kernel,stride,pad', [
    ((16, 16, 33, 31), 64, 3, 1, 1), ((16, 32, 17, 17), 130, 3, 2, 1), ((8, 48, 20, 20), 96, 5, 1, 2), ((64, 20, 28, 28), 72, 1, 1, 0),
    ((3, 64, 40, 40), 256, (1, 3), 1, (0, 1)), ((40, 64, 9, 9), 70, 2, 1, 0),
    ((40, 48, 28, 28), 72, 1, 1, 0), ((30, 16, 25, 23), 130, 3, 1, 1)])
def test_convolutions(shape, filters, kernel, stride, pad):
    rng = np.random.default_rng(filters)
    kh, kw = (kernel, kernel) if isinstance(kernel, int) else kernel
    ph, pw = (pad, pad) if isinstance(pad, int) else pad
    x = rng.standard_normal(shape, dtype=np.float32)
    w = rng.standard_normal((filters, shape[1], kh, kw), dtype=np.float32)
    got = chx.conv(chx.array(x), chx.array(w), None, stride, pad).get()
    padded = np.pad(x, ((0, 0), (0, 0), (ph, ph), (pw, pw)))
    windows = np.lib.stride_tricks.sliding_window_view(padded, (kh, kw), (2, 3))[:, :, ::stride, ::stride]  # [n, c, oh, ow, kh, kw]
    n, _, oh, ow = windows.shape[:4]
    assert got.shape == (n, filters, oh, ow)
    rows = windows.transpose(0, 2, 3, 1, 4, 5).reshape(n * oh * ow, -1)
    _check(got.transpose(0, 2, 3, 1).reshape(n * oh * ow, filters), rows, w.reshape(filters, -1))


@pytest.mark.parametrize('value', [np.inf, -np.inf, np.nan, 3.4e38, -3.39e38, 1e-37, 2.0 ** -149, 2.0 ** -111])
def test_values_that_do_not_split(value):
    """One such value among ordinary ones, and a row of nothing else: finite results are as close as any, the others the same."""
    rng = np.random.default_rng(3)
    m, k, n = 2100, 130, 1100
    x = rng.standard_normal((m, k), dtype=np.float32)
    w = rng.standard_normal((n, k), dtype=np.float32)
    x[5, 7] = value
    x[700] = value
    w[:, 7] *= 0.5
    w[300] = 0
    w[301] = 0
    w[301, 7] = 1
    got = chx.linear(chx.array(x), chx.array(w)).get().astype(np.float64)
    with np.errstate(all='ignore'):
        exact = x.astype(np.float64) @ w.T.astype(np.float64)
        magnitude = np.abs(x).astype(np.float64) @ np.abs(w.T).astype(np.float64)
        bound = (k + 4) * _EPS * magnitude + 2 * k * 2.0 ** -150  # each product and sum also rounds to a multiple of 2^-149
    special = ~np.isfinite(exact)
    np.testing.assert_array_equal(np.isnan(got)[special], np.isnan(exact)[special])
    np.testing.assert_array_equal(got[special & ~np.isnan(exact)], exact[special & ~np.isnan(exact)])
    inside = magnitude < 3.4e38  # no sum of any of the products overflows
    np.testing.assert_array_less(np.abs(got - exact)[inside], bound[inside])
    overflows = np.isfinite(exact) & (np.abs(exact) > 3.5e38)
    assert not np.isfinite(got[overflows]).any()


def test_sums_that_overflow_in_part():
    """A product whose upper parts alone are beyond the largest float, but whose value is not."""
    x, w = np.zeros((2048, 64), np.float32), np.zeros((1024, 64), np.float32)
    x[:, 3], w[:, 3] = np.float32(2 - 2 ** -9) * np.float32(2) ** 100, np.float32(2) ** 27  # bfloat16(x) rounds up to a power of two
    got = chx.linear(chx.array(x), chx.array(w)).get()
    np.testing.assert_array_equal(got, np.full_like(got, x[0, 3] * w[0, 3]))
    assert np.isfinite(got).all()


@pytest.mark.parametrize('scale', [0, -60, -99, -102])
@pytest.mark.parametrize('terms,float_pipe', [(1, 2.53e-8), (2, 3.16e-8), (5, 4.39e-8)])
def test_sums_of_few_terms_among_zeros(terms, float_pipe, scale):
    """One term is rounded once: to half a unit, 2^-24 of it, and what the small parts' own roundings, units of 2^-7 of it at most, do to that.  With more,
    the sum of the upper parts' products and the last addition round too.  Scaled down, the third parts of x are bfloat16's subnormal numbers."""
    rng = np.random.default_rng(terms)
    m, k, n = 2048, 64, 1024
    x = np.zeros((m, k), np.float32)
    for j in range(terms):
        x[np.arange(m), (np.arange(m) * 7 + 11 * j) % k] = (rng.uniform(1, 2, m) * rng.choice([-1, 1], m)).astype(np.float32)
    x *= np.float32(2.0 ** scale)
    w = rng.uniform(1, 2, (n, k)).astype(np.float32)
    got = chx.linear(chx.array(x), chx.array(w)).get().astype(np.float64)
    exact, magnitude = x.astype(np.float64) @ w.T.astype(np.float64), np.abs(x).astype(np.float64) @ np.abs(w.T).astype(np.float64)
    roundings = 1 + 2.0 ** -6 if terms == 1 else 2 * terms + 1  # (the matrix pipe's additions are off by a unit, two halves, at most)
    assert (np.abs(got - exact) / magnitude).max() <= roundings * _EPS
    # no farther off in the 2-norm than v_mfma_f32_32x32x2_f32, which rounds to nearest after every term
    assert np.linalg.norm(got - exact) <= 1.01 * float_pipe * np.linalg.norm(exact)


def _tiny(rng, shape):
    """Values below 2^-120: their third parts, and of most the second, are beyond bfloat16's least number, 2^-133."""
    return (rng.uniform(0.5, 1, shape) * rng.choice([-1, 1], shape) * 2.0 ** -120).astype(np.float32)


def test_tiny_values_beside_ordinary_ones():
    """Bits below 2^-133 are lost in the split, which counts only in sums that are as small."""
    rng = np.random.default_rng(7)
    m, k, n = 2100, 200, 1100
    x, w = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((n, k), dtype=np.float32)
    tiny = _tiny(rng, (m, k))
    x[::3, 5] = tiny[::3, 5]      # among others
    x[7::128] = tiny[7::128]      # rows of nothing else
    x[9::128] = 0
    x[9::128, 3] = tiny[9::128, 3]
    x[11::128] = 0
    w[4::200] = _tiny(rng, w[4::200].shape)
    w[6::200] = 0
    got = chx.linear(chx.array(x), chx.array(w)).get().astype(np.float64)
    exact, magnitude = x.astype(np.float64) @ w.T.astype(np.float64), np.abs(x).astype(np.float64) @ np.abs(w.T).astype(np.float64)
    # as in a sum of ordinary products; each product and sum also rounds to a multiple of 2^-149
    np.testing.assert_array_less(np.abs(got - exact), (k + 4) * _EPS * magnitude + 2 * k * 2.0 ** -150)
    assert (got[11::128] == 0).all() and (got[:, 6::200] == 0).all()


@pytest.mark.parametrize('filters', [40, 130])  # tiles of 256 x 64 and 128 x 128, pixels first
def test_tiny_pixels_and_filters(filters):
    rng = np.random.default_rng(filters)
    n, c, h, w = 30, 48, 27, 29
    x = rng.standard_normal((n, h, w, c), dtype=np.float32).reshape(-1, c)
    f = rng.standard_normal((filters, c), dtype=np.float32)
    x[5::97] = _tiny(rng, x[5::97].shape)
    f[3::31] = _tiny(rng, f[3::31].shape)
    got = chx.conv(chx.array(np.ascontiguousarray(x.reshape(n, h, w, c).transpose(0, 3, 1, 2))), chx.array(f.reshape(filters, c, 1, 1))).get()
    got = got.transpose(0, 2, 3, 1).reshape(-1, filters).astype(np.float64)
    exact, magnitude = x.astype(np.float64) @ f.T.astype(np.float64), np.abs(x).astype(np.float64) @ np.abs(f.T).astype(np.float64)
    np.testing.assert_array_less(np.abs(got - exact), (c + 4) * _EPS * magnitude + 2 * c * 2.0 ** -150)


@pytest.mark.parametrize('given', [0, 256, 1 << 24])
def test_small_outputs_need_no_workspace(given):
    """Transposed operands of a small output are copied for these kernels where there is room, and multiplied as they lie where there is not."""
    rng = np.random.default_rng(2)
    m, k, n = 1000, 4100, 900
    x, g = rng.standard_normal((k, m), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    X, G, out = chx.array(x).T, chx.array(g), chx.zeros((m, n), np.float32)
    assert _lib.load().hipcx_dot_workspace_size(X.desc(), G.desc(), out.desc()) > given
    room = chx.zeros((max(given, 16),), np.uint8)
    _lib.call('hipcx_dot', X.desc(), G.desc(), out.desc(), room.data_ptr if given else None, given, current_stream())
    _check(out.get(), x.T, g.T)


def test_narrow_outputs_are_not_worth_long_copies():
    a, b, out = chx.zeros((60000, 600), np.float32), chx.zeros((60000, 100), np.float32), chx.zeros((600, 100), np.float32)
    need = lambda x: _lib.load().hipcx_dot_workspace_size(x.desc(), b.desc(), out.desc())
    assert need(a.T) < 4 * 60000 * 100 <= need(a.reshape((600, 60000)))
