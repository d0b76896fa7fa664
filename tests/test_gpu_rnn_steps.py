"""Recurrent networks whose steps advance several layer-directions in one launch (rnn.hip), against a float64 composition with automatic
differentiation: rows and units at the edges of tiles, lines and 16-byte pieces, networks that run as a wavefront and others, batches that shrink and grow."""
import numpy as np
import pytest
import torch

from oracle import native as O
from helpers import assert_close
from test_oracle_pins import _rnn_problem

pytestmark = pytest.mark.gpu

_GATES = {'lstm': 4, 'gru': 3, 'rnn': 1}


def _layer(kind, w, b, xs, h, c, reverse):
    """(outputs by step, h, c) of one layer-direction; rows beyond a step's batch keep their state."""
    g, ys = _GATES[kind], [None] * len(xs)
    for t in (reversed(range(len(xs))) if reverse else range(len(xs))):
        n = xs[t].shape[0]
        hn = h[:n]
        sx = [xs[t] @ w[i].T + b[i] for i in range(g)]
        sh = [hn @ w[g + i].T + b[g + i] for i in range(g)]
        if kind == 'lstm':
            i, f, a, o = torch.sigmoid(sx[0] + sh[0]), torch.sigmoid(sx[1] + sh[1]), torch.tanh(sx[2] + sh[2]), torch.sigmoid(sx[3] + sh[3])
            cn = a * i + f * c[:n]
            new = o * torch.tanh(cn)
            c = torch.cat([cn, c[n:]])
        elif kind == 'gru':
            r, z = torch.sigmoid(sx[0] + sh[0]), torch.sigmoid(sx[1] + sh[1])
            a = torch.tanh(sx[2] + r * sh[2])
            new = (1 - z) * a + z * hn
        else:
            new = torch.tanh(sx[0] + sh[0])
        h = torch.cat([new, h[n:]])
        ys[t] = new
    return ys, h, c


@pytest.mark.parametrize('kind,layers,bidirectional,in_size,units,batches', [
    ('lstm', 1, False, 1, 1, (1, 1)),
    ('lstm', 2, False, 3, 5, (3, 3, 2, 1)),
    ('lstm', 4, False, 33, 31, (33, 32, 31, 1, 1)),
    ('lstm', 3, False, 70, 66, (40, 7, 40, 33, 2)),       # rows that come back
    ('lstm', 5, False, 20, 40, (6, 6, 4)),                # more layers than a launch advances
    ('lstm', 2, True, 30, 300, (40, 40, 35)),             # more workgroups than the input's products run in the steps of
    ('gru', 3, False, 5, 4, (5, 4)),
    ('gru', 2, False, 65, 130, (64, 33, 1)),
    ('gru', 2, True, 2, 36, (9, 3, 9, 1)),
    ('gru', 5, False, 16, 24, (4, 4, 1)),
    ('rnn', 3, False, 40, 65, (65, 64, 3)),
    ('rnn', 2, True, 7, 33, (2, 2)),
    ('gru', 1, False, 20, 513, (385, 384, 31)),           # steps whose products are library calls
    ('gru', 2, True, 33, 512, (390, 385, 390)),
    ('lstm', 1, False, 65, 520, (930, 929, 17)),
    ('lstm', 2, True, 16, 510, (970, 961)),
    ('rnn', 1, False, 30, 1030, (950, 945)),
])
def test_against_autograd(kind, layers, bidirectional, in_size, units, batches):
    import chainer_amd as chx
    rng = np.random.default_rng(units)
    g, d = _GATES[kind], 2 if bidirectional else 1

    def arr(*shape, scale=1.0):
        return (rng.standard_normal(shape) * scale).astype(np.float32)

    ws, bs = [], []
    for layer in range(layers):
        n_in = in_size if layer == 0 else d * units
        for _ in range(d):
            ws.append([arr(units, n_in, scale=n_in ** -0.5) for _ in range(g)] + [arr(units, units, scale=units ** -0.5) for _ in range(g)])
            bs.append([arr(units, scale=0.3) for _ in range(2 * g)])
    rows = max(batches) + 1  # one row that no step holds
    hx, cx = arr(layers * d, rows, units, scale=0.5), arr(layers * d, rows, units, scale=0.5)
    xs = [arr(n, in_size) for n in batches]
    dys = [arr(n, d * units) for n in batches]
    dhy, dcy = arr(*hx.shape), arr(*hx.shape)

    def leaf(a):
        return torch.tensor(a.astype(np.float64), requires_grad=True)

    tw, tb = [[leaf(m) for m in group] for group in ws], [[leaf(v) for v in group] for group in bs]
    tx, th, tc = [leaf(x) for x in xs], leaf(hx), leaf(cx)
    ys, hs, cs = tx, [], []
    for layer in range(layers):
        outs = []
        for k in range(d):
            i = layer * d + k
            out, h, c = _layer(kind, tw[i], tb[i], ys, th[i], tc[i], k == 1)
            outs.append(out)
            hs.append(h)
            cs.append(c)
        ys = [torch.cat([o[t] for o in outs], 1) for t in range(len(xs))]
    loss = sum((y * torch.tensor(gy.astype(np.float64))).sum() for y, gy in zip(ys, dys)) + (torch.stack(hs) * torch.tensor(dhy.astype(np.float64))).sum()
    if kind == 'lstm':
        loss = loss + (torch.stack(cs) * torch.tensor(dcy.astype(np.float64))).sum()
    loss.backward()

    up = chx.array
    # matrices and inputs that are not dense among them
    W = [[up(m) if n % 3 else up(np.ascontiguousarray(m.T)).T for n, m in enumerate(group)] for group in ws]
    B = [[up(v) for v in group] for group in bs]
    X = [up(np.concatenate([x, x], 1))[:, in_size:] for x in xs]
    lstm = kind == 'lstm'
    for training in (False, True):
        (hy, cy), got, saved = chx.rnn(layers, up(hx), up(cx) if lstm else None, W, B, X, bidirectional, kind, training=training)
        assert_close(hy.get(), torch.stack(hs).detach().numpy().astype(np.float32), 1e-5, 'hy')
        if lstm:
            assert_close(cy.get(), torch.stack(cs).detach().numpy().astype(np.float32), 1e-5, 'cy')
        for t, y in enumerate(got):
            assert_close(y.get(), ys[t].detach().numpy().astype(np.float32), 1e-5, 'y%d' % t)
    (dhx, dcx), dws, dbs, dxs = chx.rnn_backward(saved, up(dhy), up(dcy) if lstm else None, [up(a) for a in dys])
    # float32 sums over steps and rows: a few times the forward tolerance
    assert_close(dhx.get(), th.grad.numpy().astype(np.float32), 5e-5, 'dhx')
    if lstm:
        assert_close(dcx.get(), tc.grad.numpy().astype(np.float32), 5e-5, 'dcx')
    for t, a in enumerate(dxs):
        assert_close(a.get(), tx[t].grad.numpy().astype(np.float32), 5e-5, 'dx%d' % t)
    flat = lambda groups: [a for group in groups for a in (group if isinstance(group, (list, tuple)) else [group])]
    for n, (a, r) in enumerate(zip(flat(dws), flat(tw))):
        assert_close(a.get(), r.grad.numpy().astype(np.float32), 5e-5, 'dw%d' % n)
    for n, (a, r) in enumerate(zip(flat(dbs), flat(tb))):
        assert_close(a.get(), r.grad.numpy().astype(np.float32), 5e-5, 'db%d' % n)


@pytest.mark.parametrize('kind', ['lstm', 'gru', 'rnn'])
def test_infinite_inputs_and_states(kind):
    """They saturate the gates of their own side and reach nothing else (weights of one sign: inf * w sums to inf)."""
    import chainer_amd as chx
    rng = np.random.default_rng(5)
    ws, bs, _, xs, hx, cx = _rnn_problem(rng, kind, 1, False, 17, 33, (4, 4, 2))
    ws = [[np.abs(m) + np.float32(0.01) for m in group] for group in ws]
    xs[0][2, 1] = np.inf
    if kind != 'gru':  # z * h of an infinite state is infinite or NaN by definition
        hx[0, 0, :3] = np.inf
    up = chx.array
    (hy, _), ys, _ = chx.rnn(1, up(hx), up(cx) if kind == 'lstm' else None, [[up(m) for m in g] for g in ws], [[up(v) for v in g] for g in bs],
                             [up(x) for x in xs], False, kind)
    if kind == 'lstm':
        ref = O.n_step_lstm(1, hx, cx, ws, bs, xs)
    else:
        ref = O.n_step_gru(1, hx, ws, bs, xs) if kind == 'gru' else O.n_step_rnn(1, hx, ws, bs, xs, 'tanh')
    assert np.isfinite(ref[0]).all()
    assert_close(hy.get(), ref[0], 1e-5, 'hy')
    for y, r in zip(ys, ref[-1]):
        assert_close(y.get(), r, 1e-5, 'y')


def _arguments(chx, kind, layers, in_size, units, lengths, seed):
    """Arrays and descriptor pointers for direct calls of the C entries: (hx, cx, pointers of ws, bs, xs), and what they point to."""
    from chainer_amd import routines
    ws, bs, _, xs, hx, cx = _rnn_problem(np.random.default_rng(seed), kind, layers, False, in_size, units, lengths)
    W, B, X = [chx.array(m) for g in ws for m in g], [chx.array(v) for g in bs for v in g], [chx.array(x) for x in xs]
    return chx.array(hx), chx.array(cx), [routines._descriptor_pointers(a) for a in (W, B, X)], (W, B, X)


@pytest.mark.parametrize('kind', ['lstm', 'gru', 'rnn'])
@pytest.mark.parametrize('training', [0, 1])
def test_workspace_too_small(kind, training):
    """Refused before anything is written."""
    import ctypes
    import chainer_amd as chx
    from chainer_amd import _lib, routines
    from chainer_amd._array import current_stream
    mode, units = {'gru': 0, 'lstm': 1, 'rnn': 2}[kind], 40
    hx, cx, (pw, pb, px), (W, B, X) = _arguments(chx, kind, 2, 24, units, (4, 4, 3, 1), 3)
    L, T = _lib.load(), len(X)
    reserve = chx.zeros((L.hipcx_n_step_rnn_reserve_size(2, 0, mode, hx.desc(), px, T),), np.uint8) if training else None
    need = L.hipcx_n_step_rnn_workspace_size(2, 0, mode, training, hx.desc(), px, T)
    room = chx.array(np.full(need, 255, np.uint8))
    hy, cy = chx.zeros(hx.shape, np.float32), chx.zeros(hx.shape, np.float32)
    ys = [chx.zeros((x.shape[0], units), np.float32) for x in X]
    for given in (256, 2048):
        with pytest.raises(chx.ChainerxError, match='too small'):
            _lib.call('hipcx_n_step_rnn', 2, 0, mode, 0, hx.desc(), cx.desc() if kind == 'lstm' else None, pw, pb, px, T, hy.desc(),
                      cy.desc() if kind == 'lstm' else None, routines._descriptor_pointers(ys), ctypes.c_void_p(reserve.data_ptr) if training else None,
                      reserve.nbytes if training else 0, ctypes.c_void_p(room.data_ptr), given, current_stream())
    assert (room.get() == 255).all() and not any(y.get().any() for y in ys + [hy, cy])


@pytest.mark.parametrize('kind', ['lstm', 'gru', 'rnn'])
@pytest.mark.parametrize('layers,bidirectional,units,lengths', [(1, False, 33, (4, 4, 2)), (3, False, 40, (5, 3, 3, 1)), (2, True, 34, (4, 2, 2)), (2, True, 300, (3,) * 40)])
@pytest.mark.parametrize('training', [0, 1])
def test_results_that_share_memory(kind, layers, bidirectional, units, lengths, training):
    """One scratch array for every ys[t], ys[t] in place of xs[t], new states in place of the old ones: the states are right, and what is left in shared
    memory is what was written last.  Steps of one batch-major array interleave without sharing any."""
    import ctypes
    import chainer_amd as chx
    from chainer_amd import _lib, routines
    from chainer_amd._array import current_stream
    d, mode, lstm = 2 if bidirectional else 1, {'gru': 0, 'lstm': 1, 'rnn': 2}[kind], kind == 'lstm'
    ws, bs, _, xs, h, c = _rnn_problem(np.random.default_rng(units), kind, layers, bidirectional, d * units, units, lengths)
    W, B, X = [chx.array(m) for g in ws for m in g], [chx.array(v) for g in bs for v in g], [chx.array(x) for x in xs]
    hx, cx = chx.array(h), chx.array(c)
    (hy, cy), ys, _ = chx.rnn(layers, hx, cx if lstm else None, [W[i * len(ws[0]):][:len(ws[0])] for i in range(len(ws))],
                              [B[i * len(bs[0]):][:len(bs[0])] for i in range(len(bs))], X, bidirectional, kind, training=bool(training))
    hy, cy, ys = hy.get(), cy.get() if lstm else None, [y.get() for y in ys]
    L, T, pointers = _lib.load(), len(X), routines._descriptor_pointers
    px = pointers(X)
    need = L.hipcx_n_step_rnn_workspace_size(layers, int(bidirectional), mode, training, hx.desc(), px, T)
    room = chx.zeros((need,), np.uint8)
    reserve = chx.zeros((L.hipcx_n_step_rnn_reserve_size(layers, int(bidirectional), mode, hx.desc(), px, T),), np.uint8) if training else None

    def run(h_in, c_in, x_in, h_out, c_out, y_out):
        _lib.call('hipcx_n_step_rnn', layers, int(bidirectional), mode, 0, h_in.desc(), c_in.desc() if lstm else None, pointers(W), pointers(B), pointers(x_in), T,
                  h_out.desc(), c_out.desc() if lstm else None, pointers(y_out), ctypes.c_void_p(reserve.data_ptr) if training else None,
                  reserve.nbytes if training else 0, ctypes.c_void_p(room.data_ptr), need, current_stream())
        np.testing.assert_array_equal(h_out.get(), hy)
        if lstm:
            np.testing.assert_array_equal(c_out.get(), cy)

    new = lambda: (chx.zeros(hx.shape, np.float32), chx.zeros(hx.shape, np.float32))
    scratch = chx.zeros(ys[0].shape, np.float32)
    run(hx, cx, X, *new(), [scratch[:len(y)] for y in ys])
    last = ys[-1][:, :units]  # the first direction's last step, and the second one's, which ends with step 0
    np.testing.assert_array_equal(scratch.get()[:len(last), :units], last)
    if bidirectional:
        np.testing.assert_array_equal(scratch.get()[:, units:], ys[0][:, units:])
    in_place = [x.copy() for x in X]
    run(hx, cx, in_place, *new(), in_place)
    for y, r in zip(in_place, ys):
        np.testing.assert_array_equal(y.get(), r)
    h2, c2 = hx.copy(), cx.copy()
    run(h2, c2, X, h2, c2, [chx.zeros(y.shape, np.float32) for y in ys])
    h2, c2 = hx.copy(), cx.copy()
    run(h2, c2, X, c2, h2, [chx.zeros(y.shape, np.float32) for y in ys])
    batch_major = chx.zeros((ys[0].shape[0], T, d * units), np.float32)
    interleaved = [batch_major[:len(y), t] for t, y in enumerate(ys)]
    run(hx, cx, X, *new(), interleaved)
    for y, r in zip(interleaved, ys):
        np.testing.assert_array_equal(y.get(), r)
