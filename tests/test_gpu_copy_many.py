"""Several copies in one launch: concatenation and stacking at the sizes where the batched kernel changes its ways -- segments shorter than
one access, odd lengths, more segments than one launch takes, casts and strided parts in between."""
import numpy as np
import pytest

import chainer_amd as chx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['int8', 'float16', 'float32', 'float64'])
@pytest.mark.parametrize('sizes', [[1], [0, 3, 0], [5, 1, 16, 17, 4095, 4097, 2], list(range(1, 130)), [1 << 20, 7, 5 << 20, 1]])
def test_concatenate(dtype, sizes):
    rng = np.random.RandomState(len(sizes))
    parts = [rng.randint(-50, 50, n).astype(dtype) for n in sizes]
    np.testing.assert_array_equal(chx.to_numpy(chx.concatenate([chx.array(p) for p in parts], 0)), np.concatenate(parts, 0))


def test_mixed_parts():
    rng = np.random.RandomState(0)
    parts = [rng.randint(-50, 50, (3, 7)).astype(t) for t in ('float32', 'int32', 'float32', 'float64', 'float32')]
    arrays = [chx.array(p) for p in parts]
    for axis in (0, 1):
        np.testing.assert_array_equal(chx.to_numpy(chx.concatenate(arrays, axis)), np.concatenate(parts, axis))
    wide = rng.randint(-50, 50, (3, 14)).astype(np.float32)
    got = chx.concatenate([chx.array(wide)[:, ::2], arrays[0], arrays[2]], 0)
    np.testing.assert_array_equal(chx.to_numpy(got), np.concatenate([wide[:, ::2], parts[0], parts[2]], 0))
    for axis in (0, 1, 2):
        same = [arrays[0], arrays[2], arrays[4]]
        np.testing.assert_array_equal(chx.to_numpy(chx.stack(same, axis)), np.stack([parts[0], parts[2], parts[4]], axis))
