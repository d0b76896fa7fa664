"""Matrix products in tiles of 64 rows and 32 to 80 columns, at the edges of tiles, chunks of the reduction and quarters of them, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(chx, x, w, b, dt, what, view=None):
    X = chx.array(x) if view is None else view
    got = chx.linear(X, chx.array(w), None if b is None else chx.array(b)).get().astype('float64')
    x64, w64 = x.astype('float64'), w.astype('float64')
    ref = x64 @ w64.T + (0 if b is None else b.astype('float64'))
    # chains of 16 products, one sum to a chunk of 64 (128) terms, four quarters, bias; float16 results are rounded with and without the bias
    roundings = 16 + x.shape[1] / 64 + 6
    bound = roundings * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T + (0 if b is None else np.abs(b.astype('float64'))))
    if dt == 'float16':
        bound += 2.0 ** -10 * (np.abs(ref) + (0 if b is None else np.abs(b.astype('float64')))) + 2.0 ** -24
    assert (np.abs(got - ref) <= bound).all(), (what, np.max(np.abs(got - ref) / bound))


@pytest.mark.parametrize('dt,m,k,n', [
    ('float32', 63, 300, 7672), ('float32', 128, 319, 4096), ('float32', 512, 321, 1000),      # two blocks of columns
    ('float32', 99, 333, 5651), ('float32', 192, 384, 4095),                                   # three
    ('float32', 994, 385, 807), ('float32', 1000, 448, 993),                                   # four
    ('float32', 128, 650, 10000), ('float32', 127, 303, 9985),                                 # five
    ('float32', 1721, 302, 798), ('float32', 670, 511, 2007),                                  # two rounds
    ('float16', 63, 470, 7672), ('float16', 99, 510, 5651), ('float16', 428, 514, 2065), ('float16', 127, 768, 9985), ('float16', 1903, 642, 452),
    ('float32', 128, 299, 10000), ('float16', 994, 468, 807)])                                 # other tiles
def test_products(dt, m, k, n):
    import chainer_amd as chx
    rng = np.random.default_rng(m + k + n)
    x, w, b = [rng.standard_normal(s).astype(dt) for s in ((m, k), (n, k), (n,))]
    check(chx, x, w, b, dt, 'bias')
    check(chx, x, w, None, dt, 'no bias')


@pytest.mark.parametrize('dt', ['float32', 'float16'])
def test_views_and_special_values(dt):
    import chainer_amd as chx
    rng = np.random.default_rng(2)
    wide, w, b = [rng.standard_normal(s).astype(dt) for s in ((130, 516), (9990, 512), (9990,))]
    check(chx, wide[2:, 2:514], w, b, dt, 'rows of a wider array', chx.array(wide)[2:, 2:514])
    x = wide[:128, :512].copy()
    x[5, 511], w[77, 3] = np.nan, np.inf
    got = chx.linear(chx.array(x), chx.array(w), chx.array(b)).get()
    bad = np.zeros(got.shape, bool)
    bad[5], bad[:, 77] = True, True
    assert np.isnan(got[5]).all() and (~np.isfinite(got[:, 77])).all() and np.isfinite(got[~bad]).all()


@pytest.mark.parametrize('m,k,n', [(128, 650, 10000), (512, 1000, 1000), (670, 3324, 2007), (994, 385, 807)])
def test_error_of_chains_of_sixteen(m, k, n):
    """Only these tiles sum float32 in chains of 16 products: 1.0e-7 to 1.6e-7 of the norm, where one chain to a wave has 2.7e-7 and 7.3e-7 at 650 and 3324 terms."""
    import chainer_amd as chx
    rng = np.random.default_rng(k)
    x, w = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((n, k), dtype=np.float32)
    ref = x.astype('float64') @ w.astype('float64').T
    assert np.linalg.norm(chx.linear(chx.array(x), chx.array(w), None).get() - ref) < 1.8e-7 * np.linalg.norm(ref)
