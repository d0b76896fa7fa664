"""Batch norm with Relu behind it and its gradient, the sum of two gradients before Relu's, and updates of many parameters: each against the routines that it stands
for, bit for bit, in the layouts of the kernels that take a channel in registers, of those that do not, and of none."""
import numpy as np
import pytest

import chainer_amd as chx

pytestmark = pytest.mark.gpu

SHAPES = [(1, 3, 1, 1), (21, 7, 7, 7), (42, 257, 7, 7), (5, 3, 14, 14), (4, 2, 64, 128), (25, 256, 32, 128), (25, 2, 32, 128), (14, 2, 64, 129), (7, 2, 63, 127)]


def same(a, b):
    np.testing.assert_array_equal(a.get().view('u%d' % a.dtype.itemsize), b.get().view('u%d' % b.dtype.itemsize))


@pytest.mark.parametrize('dt,pt', [('float32', 'float32'), ('float16', 'float32'), ('float16', 'float16'), ('float64', 'float64')])
@pytest.mark.parametrize('shape', SHAPES)
def test_batch_norm_relu(dt, pt, shape):
    rng = np.random.default_rng(shape[0] * shape[1])
    c = shape[1]
    x, r, g = (chx.array(rng.integers(-2, 3, shape).astype(dt)) for _ in range(3))  # whole numbers: results of exactly zero among them
    gamma, beta = chx.array(rng.choice([-1., 0., 1., .5], c).astype(pt)), chx.array(rng.choice([-1., 0., 1.], c).astype(pt))
    for residual in (None, r):
        stats = [chx.array(rng.uniform(0.5, 1.5, c).astype(pt)) for _ in range(2)]
        ref_stats = [chx.array(s.get()) for s in stats]
        b, ref_state = chx.batch_norm(x, gamma, beta, *ref_stats)
        y, total, state = chx.batch_norm_relu(x, gamma, beta, *stats, residual=residual)
        if residual is None:
            assert total is None
        else:
            same(total, chx.add(b, residual))
        same(y, chx.relu(b if total is None else total))
        for got, ref in zip(stats + list(state[:2]), ref_stats + list(ref_state[:2])):
            same(got, ref)
    for got, ref in zip(chx.batch_norm_relu_grad(x, gamma, beta, g, state), chx.batch_norm_grad(x, gamma, chx.if_less_else(b, 0, 0, g), state)):
        same(got, ref)


@pytest.mark.parametrize('dt', ['float16', 'float32'])
def test_batch_norm_relu_special_values(dt):
    x = np.zeros((2, 4, 8, 8), dt)
    x[0, 0, 0, 0], x[1, 1, 2, 3], x[:, 2] = np.nan, np.inf, -0.0
    args = [chx.array(a) for a in (x, np.ones(4, np.float32), np.array([0, 0, -0.0, 1], np.float32))]
    g, stats = chx.array(np.full(x.shape, 2, dt)), [chx.array(np.ones(4, np.float32)) for _ in range(4)]
    b, ref_state = chx.batch_norm(*args, *stats[:2])
    y, _, state = chx.batch_norm_relu(*args, *stats[2:])
    np.testing.assert_array_equal(y.get(), chx.relu(b).get())
    for got, ref in zip(chx.batch_norm_relu_grad(*args, g, state), chx.batch_norm_grad(args[0], args[1], chx.if_less_else(b, 0, 0, g), ref_state)):
        np.testing.assert_array_equal(got.get(), ref.get())


def test_batch_norm_relu_of_other_layouts():
    rng = np.random.default_rng(3)
    x, r, g = (chx.array(rng.standard_normal((5, 4, 6, 7), dtype=np.float32)).transpose(0, 2, 3, 1) for _ in range(3))
    p = [chx.array(rng.uniform(0.5, 1.5, 6).astype(np.float32)) for _ in range(6)]
    b, ref_state = chx.batch_norm(x, *p[:4])
    y, total, state = chx.batch_norm_relu(x, p[0], p[1], p[4], p[5], residual=r)
    same(total, chx.add(b, r))
    same(y, chx.relu(total))
    for got, ref in zip(chx.batch_norm_relu_grad(x, p[0], p[1], g, state), chx.batch_norm_grad(x, p[0], chx.if_less_else(b, 0, 0, g), state)):
        same(got, ref)


@pytest.mark.parametrize('dt', ['float16', 'float32', 'float64'])
def test_add_relu_grad(dt):
    rng = np.random.default_rng(1)
    x, a, b = (rng.standard_normal((3, 5, 11)).astype(dt) for _ in range(3))
    x[0, 0, :4] = [np.nan, 0, -0.0, np.inf]
    a[0, 1, 0] = np.nan
    for order in (None, (2, 0, 1)):
        X, A, B = (chx.array(v) if order is None else chx.array(v).transpose(*order) for v in (x, a, b))
        same(chx.add_relu_grad(X, A, B), chx.if_less_else(X, 0, 0, chx.add(A, B)))
    same(chx.add_relu_grad(chx.array(x), chx.array(a[:, :1]), chx.array(b)), chx.if_less_else(chx.array(x), 0, 0, chx.add(chx.array(a[:, :1]), chx.array(b))))


@pytest.mark.parametrize('sizes', [[1], [0, 7, 8, 9], [255 * 8 + 3, 256 * 8, 4096 * 8 + 1], list(range(1, 240)), [5 << 20, 3, (6 << 20) + 5]])
def test_sgd_update(sizes):
    rng = np.random.default_rng(len(sizes))
    for dts in (['float16'], ['float32'], ['float16', 'float32', 'float64']):
        ps, gs = [], []
        for i, n in enumerate(sizes):
            dt = dts[i % len(dts)]
            wide = chx.array(rng.standard_normal(n + 3).astype(dt))
            ps.append(wide[i % 3:i % 3 + n])  # starts at any element
            gs.append(chx.array(rng.standard_normal((1, n)).astype(dt)))
        for lr in (0.01, 2):
            for p, g, got in zip(ps, gs, chx.sgd_update(ps, gs, lr)):
                same(got, chx.subtract(p, chx.multiply(g.reshape(p.shape), lr)))
    # other layouts and types that promote
    p, g = chx.array(rng.standard_normal((40, 30)).astype('float16')).T, chx.array(rng.standard_normal((30, 40)).astype('float16'))
    same(chx.sgd_update([p], [g], 0.5)[0], chx.subtract(p, chx.multiply(g, 0.5)))
    same(chx.sgd_update([p], [g.astype('float32')], 0.5)[0], chx.subtract(p, chx.multiply(g.astype('float32'), 0.5)))
    with pytest.raises(chx.DimensionError):
        chx.sgd_update([p], [g, g], 0.5)


@pytest.mark.parametrize('dt,pt', [('float32', 'float32'), ('float16', 'float32'), ('float16', 'float16'), ('float64', 'float64')])
@pytest.mark.parametrize('shape', SHAPES)
def test_batch_norm_relu_is_one_call(dt, pt, shape):
    """Arrays of the tests above run on the dedicated kernels, not on the routines that they are compared with."""
    from chainer_amd import _host
    c = shape[1]
    x, r, g, (gamma, beta, mean, var) = chx.zeros(shape, dt), chx.zeros(shape, dt), chx.zeros(shape, dt), [chx.ones((c,), pt) for _ in range(4)]
    for residual in (None, r):
        y, total, state = _host.batch_norm_direct(x, gamma, beta, mean, var, 2e-5, 0.9, None, True, residual)
        assert y.shape == shape and (total is None) == (residual is None)
    assert len(_host.batch_norm_grad_direct(x, gamma, g, *state, None, beta)) == 3


def test_which_calls_are_composed():
    from chainer_amd import _host
    x, p = chx.zeros((5, 6, 7, 4), 'float32'), [chx.ones((6,), 'float32') for _ in range(4)]
    y = chx.zeros((5, 7, 4, 6), 'float32').transpose(0, 3, 1, 2)
    state = _host.batch_norm_direct(x, *p, 2e-5, 0.9, None, True, None)[2]
    assert _host.batch_norm_direct(y, *p, 2e-5, 0.9, None, True, None) is None and _host.batch_norm_direct(x, *p, 2e-5, 0.9, None, True, y) is None
    assert _host.batch_norm_grad_direct(x, p[0], y, *state, None, p[1]) is None and _host.batch_norm_grad_direct(x, p[0], x, *state, None, p[1].astype('float64')) is None
    assert _host.add_relu_grad_direct(x, x, x) is not None and _host.add_relu_grad_direct(y, x[:, :, :, ::-1], x) is not None
    assert _host.add_relu_grad_direct(x, x[:, :1], x) is None and _host.add_relu_grad_direct(x, x.astype('float16'), x) is None
    assert len(_host.sgd_update_direct([x, y], [x, x.reshape((-1,))], 0.5)) == 2 and _host.sgd_update_direct([], [], 0.5) == []
    assert _host.sgd_update_direct([x], [x.astype('float16')], 0.5) is None and _host.sgd_update_direct([x], [x], x[0, 0, 0, 0]) is None
