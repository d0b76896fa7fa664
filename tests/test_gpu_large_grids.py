"""Problems that need more threads, or more output positions, than one launch counts: 2^32 threads to a grid, 2^31 positions to a
convolution.  Inputs are broadcast; results are looked at where a count would wrap, and at both ends."""
import contextlib

import numpy as np
import pytest

from helpers import assert_close

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def device_memory(nbytes):
    import torch
    import chainer_amd as chx
    if torch.cuda.mem_get_info()[0] < nbytes:
        pytest.skip('needs %d bytes of device memory' % nbytes)
    try:
        yield chx
    finally:
        chx.synchronize()
        chx.free_unused_blocks()


def windows(n, width=50):
    return [lo for lo in (0, (1 << 30) - width // 2, (1 << 31) - width // 2, (1 << 32) - width // 2, n - width) if 0 <= lo <= n - width]


def test_diagflat():
    n = (1 << 16) + 3
    with device_memory(n * n) as chx:
        v = np.arange(n).astype('int8')
        out = chx.diagflat(chx.array(v))
        for row in (0, 1, 1 << 15, (1 << 16) - 1, n - 1):
            expected = np.zeros(n, 'int8')
            expected[row] = v[row]
            assert np.array_equal(out[row].get(), expected), row
        del out


def test_cumsum():
    lines = (1 << 32) + 100
    with device_memory(5 * lines) as chx:
        out = chx.cumsum(chx.array(np.full((1, 1), 3, 'float16')).broadcast_to((lines, 1)), 1)
        for lo in windows(lines):
            assert np.all(out[lo:lo + 50].get() == 3), lo
        del out


def test_add_at():
    n = (1 << 32) + 100
    with device_memory(6 * n) as chx:
        a = chx.array(np.full((1, 1), 5, 'int8')).broadcast_to((1, n))
        b = chx.array(np.full((2, 1), 4, 'int8')).broadcast_to((2, n))
        out = chx.add_at(a, chx.array(np.array([0, 0])), 0, b)
        for lo in windows(n):
            assert np.all(out[0, lo:lo + 50].get() == 13), lo
        del out


def test_integer_dot():
    n = (1 << 30) + 100
    with device_memory(2 * n) as chx:
        a = chx.array(np.array([[3, 5]], 'int8'))
        b = chx.array(np.array([[2], [7]], 'int8')).broadcast_to((2, n))
        out = chx.dot(a, b)
        for lo in windows(n):
            assert np.all(out[0, lo:lo + 50].get() == 41), lo
        del out


def test_float64_dot():
    m = (1 << 30) + 100
    with device_memory(10 * m) as chx:
        a = chx.array(np.array([[3, 5]], 'float64')).broadcast_to((m, 2))
        out = chx.dot(a, chx.array(np.array([[2], [7]], 'float64')))
        for lo in windows(m):
            assert np.all(out[lo:lo + 50, 0].get() == 41), lo
        del out


@pytest.mark.parametrize('dt,images,height,width', [('float32', 1, (1 << 15) + 2, 1 << 15), ('float16', 33, 1 << 13, 1 << 13)])
def test_convolution(dt, images, height, width):
    """2^30 pixels to a plane; 2^31 and more output positions."""
    with device_memory(30 * images * height * width) as chx:
        rng = np.random.default_rng(31)
        line = rng.standard_normal(width).astype(dt)
        w = rng.standard_normal((1, 1, 3, 3)).astype(dt)
        x = chx.array(line.reshape(1, 1, 1, width)).broadcast_to((images, 1, height, width))
        out = chx.conv(x, chx.array(w), None, 1, 1)
        padded = np.concatenate([[0], line.astype('f8'), [0]])
        for n in sorted({0, images // 2, images - 1}):
            for h in (0, 1, height // 2, height - 2, height - 1):
                expected = np.zeros(width)
                for r in range(3):
                    if 0 <= h + r - 1 < height:
                        for s in range(3):
                            expected += w[0, 0, r, s].astype('f8') * padded[s:s + width]
                assert_close(out[n, 0, h].get(), expected.astype(dt), 1e-5 if dt == 'float32' else 4e-3, 'image %d row %d' % (n, h))
        del out
