"""Small matrix products over whole 128-byte lines (SmallDotLinesKernel): edges of tiles of every width, lines and 16-byte pieces, one wave to eight, split
reductions, and what lies behind an operand's rows."""
import numpy as np
import pytest

import chainer_amd as chx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt', ['float32', 'float16'])
@pytest.mark.parametrize('m,k,n', [
    (5, 1536, 10), (33, 1538, 65), (64, 4099 * 2, 40),             # few long tiles, one of them split
    (512, 450, 512), (545, 458, 450), (800, 66 * 7, 33 * 32),      # one or two tiles to a compute unit
    (1025, 514, 1000), (1500, 322, 1100), (900, 70 * 8, 1500),     # more
    (100, 802, 1001), (7, 1030, 17), (130, 802, 2390), (300, 450, 1489), (290, 514, 1300),  # 16, 48 and 64 columns
])
def test_rows_in_pieces(dt, m, k, n):
    rng = np.random.default_rng(k)
    pad = 2 if dt == 'float16' else 1  # rows that start at multiples of 4 bytes, with NaN behind them

    def wide(rows):
        a = np.full((rows, k + pad), np.nan, dt)
        a[:, :k] = rng.integers(-2, 3, (rows, k))
        a[:, k // 2:k] *= rng.integers(0, 2, (rows, k - k // 2)).astype(dt)
        return a

    x, w, bias = wide(m), wide(n), rng.integers(-20, 21, n).astype(dt)
    got = chx.linear(chx.array(x)[:, :k], chx.array(w)[:, :k], chx.array(bias)).get()
    expected = x[:, :k].astype(np.float32) @ w[:, :k].T.astype(np.float32)  # whole numbers below 2^24: exact in any order
    np.testing.assert_array_equal(got, (expected.astype(dt).astype(np.float32) + bias.astype(np.float32)).astype(dt))
