"""Batch normalisation with a channel in the registers of one workgroup (BnChannelKernel, BnChannelGradKernel) against float64: remainders of its
vectors of every width, one channel to many, the largest channels that fit and the smallest that do not."""
import numpy as np
import pytest

import chainer_amd as chx
from helpers import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dt', ['float32', 'float16'])
@pytest.mark.parametrize('shape', [
    (1, 3, 1, 1), (2, 5, 3, 3), (21, 7, 7, 7), (3, 260, 25, 27), (42, 257, 7, 7), (5, 3, 14, 14), (33, 9, 14, 14),
    (1, 2, 64, 128), (2, 2, 64, 128), (4, 2, 64, 128), (4, 3, 130, 126), (25, 256, 32, 128), (25, 2, 32, 128), (13, 1, 64, 128), (14, 2, 64, 128),
    (7, 2, 64, 126), (2, 257, 62, 66)])
def test_forward_and_gradient(dt, shape):
    rng = np.random.default_rng(shape[0] * shape[1])
    c = shape[1]
    x = (rng.standard_normal(shape) * 2 + 1).astype(dt)
    g = rng.standard_normal(shape).astype(dt)
    gamma, beta, rm, rv = (rng.uniform(0.5, 1.5, c).astype(np.float32) for _ in range(4))
    RM, RV = chx.array(rm), chx.array(rv)
    y, state = chx.batch_norm(chx.array(x), chx.array(gamma), chx.array(beta), RM, RV, 2e-5, 0.9)
    x64, g64 = x.astype(np.float64), g.astype(np.float64)
    wide = lambda a: np.asarray(a, np.float64).reshape(1, c, 1, 1)
    n = x.size // c
    mean, var = x64.mean((0, 2, 3)), x64.var((0, 2, 3))
    inv = 1 / np.sqrt(var + 2e-5)
    x_hat = (x64 - wide(mean)) * wide(inv)
    tol = 2e-3 if dt == 'float16' else 1e-5 * max(1, 20 * (n == 1))  # one rounding to float16; float32 sums
    assert_close(y.get(), (x_hat * wide(gamma) + wide(beta)).astype(dt), tol, 'out')
    assert_close(RM.get(), (rm * 0.9 + 0.1 * mean).astype(np.float32), 1e-5, 'running mean')
    assert_close(RV.get(), (rv * 0.9 + 0.1 * var * (n / max(n - 1, 1))).astype(np.float32), 1e-5, 'running variance')
    gx, ggamma, gbeta = chx.batch_norm_grad(chx.array(x), chx.array(gamma), chx.array(g), state)
    sg, sgx = g64.sum((0, 2, 3)), (g64 * x_hat).sum((0, 2, 3))
    scale = np.sqrt(n)  # what the sums of n random terms come to
    assert np.abs(gbeta.get() - sg).max() <= 2e-6 * scale * 10 and np.abs(ggamma.get() - sgx).max() <= 2e-6 * scale * 10
    expected = wide(gamma * inv) * (g64 - (x_hat * wide(sgx) + wide(sg)) / n)
    assert_close(gx.get(), expected.astype(dt), 2e-3 if dt == 'float16' else (1e-5 if n > 1 else 1), 'gx')
