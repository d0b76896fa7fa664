"""float16 matrix products over rows that start and end anywhere, and of up to four rows: at the edges of pieces, tiles and the rule for few rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(chx, x, w, X, W, what):
    got = chx.dot(X, W.T).get().astype('float64')
    x64, w64 = x.astype('float64'), w.astype('float64')
    ref = x64 @ w64.T
    # one rounding to 2^-11 of the result, float sums of exact products in chains of at most all the terms, float16's smallest step
    bound = 2.0 ** -11 * np.abs(ref) + (x.shape[1] + 40) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T) + 2.0 ** -24
    assert (np.abs(got - ref) <= bound).all(), (what, np.max(np.abs(got - ref) / bound))


@pytest.mark.parametrize('m,k,n', [(5, 1, 7), (6, 7, 9), (1, 9, 40), (3, 15, 33), (64, 33, 500), (33, 65, 47), (20, 651, 2600), (37, 801, 1000), (128, 333, 5000),
                                   (500, 501, 500), (150, 1023, 2049), (1000, 785, 1000), (300, 4001, 300), (129, 771, 9985), (2, 1001, 1000),
                                   (2, 1000, 2560), (2, 1000, 2561), (3, 3072, 1000), (3, 3070, 1000), (4, 332, 3333), (1, 64, 10000)])
def test_products(m, k, n):
    import chainer_amd as chx
    rng = np.random.default_rng(m + k + n)
    x, w = [rng.standard_normal(s).astype('float16') for s in ((m, k + 1), (n, k + 1))]
    X, W = chx.array(x), chx.array(w)
    x[0, -1] = w[0, -1] = x[-1, 0] = w[-1, 0] = np.nan  # what lies beside the operands
    X, W = chx.array(x), chx.array(w)
    ok = np.s_[1:-1] if m > 2 else np.s_[:0]
    x2, w2 = np.ascontiguousarray(np.nan_to_num(x[:, :k])), np.ascontiguousarray(np.nan_to_num(w[:, :k]))
    check(chx, x2, w2, chx.array(x2), chx.array(w2), 'dense')
    check(chx, x[ok, :k], w[1:-1, :k], X[ok, :k], W[1:-1, :k], 'rows of a wider array')
    check(chx, x[ok, 1:], w[1:-1, 1:], X[ok, 1:], W[1:-1, 1:], 'rows that start at odd elements')
    check(chx, x[ok, 1:], w[1:-1, :k], X[ok, 1:], W[1:-1, :k], 'one of each')


@pytest.mark.parametrize('m,k,n', [(1, 8, 40), (1, 9, 40), (2, 15, 33), (2, 1001, 1000), (2, 1000, 2560), (2, 1000, 2561), (1, 64, 10000), (1, 771, 2559), (3, 3071, 1000)])
def test_few_rows_between_what_is_not_a_number(m, k, n):
    import chainer_amd as chx
    rng = np.random.default_rng(m + k + n)
    for first_x, first_w in ((0, 0), (1, 1), (1, 0), (0, 1)):  # even and odd elements
        x, w = [np.full((rows + 2, k + 2), np.nan, 'float16') for rows in (m, n)]
        of_x, of_w = np.s_[1:-1, first_x:first_x + k], np.s_[1:-1, first_w:first_w + k]
        x[of_x], w[of_w] = [rng.standard_normal((rows, k)).astype('float16') for rows in (m, n)]
        X, W = chx.array(x)[of_x], chx.array(w)[of_w]
        assert X.shape == (m, k) and W.shape == (n, k)
        check(chx, x[of_x], w[of_w], X, W, 'starts %d and %d' % (first_x, first_w))


@pytest.mark.parametrize('m,k,n', [(1, 1000, 5600), (1, 1000, 5601), (1, 457, 2560), (1, 457, 2561), (2, 1030, 2575), (2, 1030, 2576), (3, 2048, 1280), (4, 2048, 1281),
                                   (4, 2047, 700), (3, 2047, 1281), (4, 3072, 2001)])
def test_limits_of_the_rule_for_few_rows(m, k, n):
    import chainer_amd as chx
    rng = np.random.default_rng(m + k + n)
    x, w = [rng.standard_normal((rows, k)).astype('float16') for rows in (m, n)]
    check(chx, x, w, chx.array(x), chx.array(w), 'dense')


@pytest.mark.parametrize('k,n', [(2048, 1000), (1000, 2560), (1000, 5600), (2048, 1), (1001, 1), (7, 1)])
def test_stride_of_a_single_row_or_column_says_nothing(k, n):
    import chainer_amd as chx
    rng = np.random.default_rng(k + n)
    x, w = rng.standard_normal((1, k)).astype('float16'), rng.standard_normal((n, k)).astype('float16')
    X, W = chx.array(np.pad(x, ((0, 0), (0, 1 + k % 2))))[:, :k], chx.array(np.pad(w, ((0, 0), (0, 2 - k % 2))))[:, :k]  # rows of even pitch
    rows = [chx.array(x.reshape(1, k, 1, 1)).reshape((1, k)), chx.array(x), X]
    assert len({r.strides for r in rows}) > 1
    columns = [W] if n > 1 else [W, chx.array(w), chx.array(w.reshape(1, k, 1, 1)).reshape((1, k))]
    expect = chx.dot(X, W.T).get()
    check(chx, x, w, X, W, 'even pitch')
    for r in rows:
        for c in columns:  # the same kernel: the same bits
            np.testing.assert_array_equal(chx.dot(r, c.T).get(), expect)
