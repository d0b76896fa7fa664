"""Performance cases of the hip backend: whole calls as a program that uses chainer_amd issues them, eagerly, on resident arrays.

Eight kinds of work, each with the shapes of the package's own workloads (chainer_amd/configs.py, bench.py) and a range around them:

  mlp       MNIST-shaped perceptron, forward + softmax cross entropy
  sweep     element-wise, reduction and log-softmax calls on one matrix
  cifar     3x3 convolution stack with fixed batch norm
  resnet50  ResNet-50 inference in float16, call by call or through the fused convolution entry
  train     one ResNet-50 training step, float16 with float32 batch-norm parameters
  lstm_lm   LSTM language model, one call chain per time step
  rnn       a whole recurrent network per call (RnnKernel), forward alone or with backpropagation through time
  linear    a fully connected layer, forward and backward
"""
import math

import numpy as np
import torch

import chainer_amd as chx
from chainer_amd import configs as cfg


def listed():
    return [
        # one digit at a time: nothing but launches and host work
        {'name': 'mlp_b1', 'kind': 'mlp', 'batch': 1, 'units': 1000, 'dtype': 'float32'},
        # the MNIST example's batch
        {'name': 'mlp_b100', 'kind': 'mlp', 'batch': 100, 'units': 1000, 'dtype': 'float32'},
        # activations of an odd-sized layer: rows that no vector width divides
        {'name': 'sweep_333x1001_f16', 'kind': 'sweep', 'rows': 333, 'cols': 1001, 'dtype': 'float16'},
        # the element-wise / reduction sweep
        {'name': 'sweep_4096x4096', 'kind': 'sweep', 'rows': 4096, 'cols': 4096, 'dtype': 'float32'},
        # evaluation of the CIFAR network
        {'name': 'cifar_b256', 'kind': 'cifar', 'batch': 256, 'dtype': 'float32'},
        # one image, answered as fast as possible
        {'name': 'resnet50_b1', 'kind': 'resnet50', 'batch': 1, 'size': 224, 'fused': False},
        # throughput inference, the headline workload
        {'name': 'resnet50_b128', 'kind': 'resnet50', 'batch': 128, 'size': 224, 'fused': False},
        # a server's partly filled batch through the fused entry
        {'name': 'resnet50_fused_b37', 'kind': 'resnet50', 'batch': 37, 'size': 224, 'fused': True},
        # one GPU's share of ImageNet training
        {'name': 'train_b32', 'kind': 'train', 'batch': 32, 'size': 224},
        # the PTB model, evaluated on a batch of windows
        {'name': 'lstm_lm_b128', 'kind': 'lstm_lm', 'batch': 128, 'seq': 35, 'units': 650, 'vocab': 10000, 'dtype': 'float32'},
        # PTB training at the example's batch through the recurrent-network kernels
        {'name': 'rnn_lstm_train_b20', 'kind': 'rnn', 'mode': 'lstm', 'layers': 2, 'bidirectional': False, 'steps': 35, 'batch': 20,
         'units': 650, 'ragged': False, 'train': True},
        # the PTB model's output layer over all time steps, both directions, 650 being no multiple of a tile
        {'name': 'linear_4480x650x10000_f16', 'kind': 'linear', 'rows': 4480, 'n_in': 650, 'n_out': 10000, 'dtype': 'float16'},
    ]


def _log_int(rng, low, high):
    return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))


def draw(rng):
    kind = rng.choice(['mlp', 'sweep', 'cifar', 'resnet50', 'train', 'lstm_lm', 'rnn', 'linear'])
    if kind == 'mlp':
        return {'kind': kind, 'batch': _log_int(rng, 1, 1000), 'units': _log_int(rng, 50, 1000), 'dtype': rng.choice(['float32', 'float16'])}
    if kind == 'sweep':
        total = _log_int(rng, 1 << 10, 1 << 26)
        rows = _log_int(rng, 1, min(total // 2, 1 << 16))
        return {'kind': kind, 'rows': rows, 'cols': total // rows, 'dtype': rng.choice(['float32', 'float16'])}
    if kind == 'cifar':
        return {'kind': kind, 'batch': _log_int(rng, 1, 256), 'dtype': rng.choice(['float32', 'float16'])}
    if kind == 'resnet50':
        return {'kind': kind, 'batch': _log_int(rng, 1, 127), 'size': 32 * rng.randint(2, 7), 'fused': rng.random() < 0.5}
    if kind == 'train':
        return {'kind': kind, 'batch': _log_int(rng, 2, 31), 'size': 32 * rng.randint(2, 7)}
    if kind == 'lstm_lm':
        return {'kind': kind, 'batch': _log_int(rng, 1, 128), 'seq': _log_int(rng, 1, 34), 'units': _log_int(rng, 50, 650),
                'vocab': _log_int(rng, 100, 10000), 'dtype': rng.choice(['float32', 'float16'])}
    if kind == 'rnn':
        return {'kind': kind, 'mode': rng.choice(['lstm', 'gru', 'rnn']), 'layers': rng.randint(1, 3), 'bidirectional': rng.random() < 0.5,
                'steps': _log_int(rng, 1, 35), 'batch': _log_int(rng, 1, 128), 'units': _log_int(rng, 16, 649),
                'ragged': rng.random() < 0.5, 'train': rng.random() < 0.5}
    rows, n_in = _log_int(rng, 1, 8192), _log_int(rng, 16, 4096)
    return {'kind': kind, 'rows': rows, 'n_in': n_in, 'n_out': _log_int(rng, 10, min(10000, max(10, 40000000000 // (rows * n_in)))),
            'dtype': rng.choice(['float32', 'float16'])}


def _step_sizes(case):
    """Batch rows of every time step; ragged batches shrink as their shorter sequences end."""
    n, b = case['steps'], case['batch']
    return [max(1, b * (n - t) // n) if case['ragged'] else b for t in range(n)]


_GATES = {'lstm': 4, 'gru': 3, 'rnn': 1}


def _rnn_inputs(case, rng):
    d, u, g = (2 if case['bidirectional'] else 1), case['units'], _GATES[case['mode']]

    def arr(*shape, scale=1.0):
        return chx.array((rng.standard_normal(shape, dtype=np.float32) * np.float32(scale)))

    ws, bs = [], []
    for layer in range(case['layers']):
        n_in = u if layer == 0 else d * u
        for _ in range(d):
            ws.append([arr(u, n_in, scale=1 / math.sqrt(n_in)) for _ in range(g)] + [arr(u, u, scale=1 / math.sqrt(u)) for _ in range(g)])
            bs.append([arr(u, scale=0.1) for _ in range(2 * g)])
    state_shape = (case['layers'] * d, case['batch'], u)
    sizes = _step_sizes(case)
    lstm = case['mode'] == 'lstm'
    state = {'ws': ws, 'bs': bs, 'x': arr(sum(sizes), u), 'bounds': [int(s) for s in np.cumsum(sizes)[:-1]],
             'hx': arr(*state_shape, scale=0.5), 'cx': arr(*state_shape, scale=0.5) if lstm else None}
    if case['train']:
        state.update(dy=arr(sum(sizes), d * u, scale=0.1), dhy=arr(*state_shape, scale=0.1), dcy=arr(*state_shape, scale=0.1) if lstm else None)
    return state


def prepare(case, seed):
    kind = case['kind']
    rng = np.random.Generator(np.random.PCG64(seed))
    up = chx.array
    state = {'case': case}
    if kind == 'mlp':
        dt = np.dtype(case['dtype'])
        x, t = cfg.mlp_input(seed, case['batch'], dt)
        state.update(p=cfg.tree_map(up, cfg.mlp_params(seed, dt, n_units=case['units'])), x=up(x), t=up(t))
    elif kind == 'sweep':
        dt = np.dtype(case['dtype'])
        state.update(x=up(rng.standard_normal((case['rows'], case['cols']), dtype=np.float32).astype(dt)),
                     b=up(rng.standard_normal(case['cols'], dtype=np.float32).astype(dt)))
    elif kind == 'cifar':
        dt = np.dtype(case['dtype'])
        state.update(p=cfg.tree_map(up, cfg.cifar_params(seed, dt)), x=up(cfg.cifar_input(seed, case['batch'], dt)))
    elif kind == 'resnet50':
        state.update(p=cfg.tree_map(up, cfg.resnet50_params(seed)), x=up(cfg.resnet50_input(seed, case['batch'], size=case['size'])))
    elif kind == 'train':
        p = cfg.resnet50_params_mixed(seed=seed)
        # the running statistics of all layers lie in one array, as a program that saves or averages them keeps them
        norms = [blk[k] for stage in p['stages'] for blk in stage for k in sorted(blk) if k.startswith('bn')] + [p['bn1']]
        flat = up(np.concatenate([bn[k] for bn in norms for k in ('mean', 'var')]))
        pos = 0
        for bn in norms:
            for k in ('mean', 'var'):
                n = bn[k].size
                bn[k] = flat[pos:pos + n]
                pos += n
        state.update(p=cfg.tree_map(lambda a: a if isinstance(a, chx.ndarray) else up(a), p), statistics=flat, ops=cfg.DeviceTrainOps(chx),
                     x=up(cfg.resnet50_input(seed, case['batch'], size=case['size'])), t=up(rng.integers(0, 1000, case['batch']).astype(np.int32)))
    elif kind == 'lstm_lm':
        p = cfg.lstm_lm_params(seed, np.dtype(case['dtype']), case['vocab'], case['units'])
        state.update(p=cfg.tree_map(up, p), ids=up(cfg.lstm_lm_input(seed, case['batch'], case['seq'], case['vocab'])))
    elif kind == 'rnn':
        state.update(_rnn_inputs(case, rng))
    else:
        dt = np.dtype(case['dtype'])

        def arr(*shape, scale=1.0):
            return up((rng.standard_normal(shape, dtype=np.float32) * np.float32(scale)).astype(dt))

        rows, n_in, n_out = case['rows'], case['n_in'], case['n_out']
        state.update(x=arr(rows, n_in), w=arr(n_out, n_in, scale=1 / math.sqrt(n_in)), b=arr(n_out, scale=0.1), gy=arr(rows, n_out, scale=0.01))
    return state


class _Exported(object):
    """Device memory of an array, described for torch."""

    def __init__(self, a):
        self.array = a  # keeps the memory
        self.__cuda_array_interface__ = {'shape': a.shape, 'typestr': a.dtype.str, 'data': (a.data_ptr, False), 'version': 2}


def _out(a):
    return torch.as_tensor(_Exported(a), device='cuda')


def run(state):
    case = state['case']
    kind = case['kind']
    if kind == 'mlp':
        return [_out(a) for a in cfg.mlp_forward(chx, state['p'], state['x'], state['t'])]
    if kind == 'sweep':
        x, b = state['x'], state['b']
        results = {'add': chx.add(x, b), 'multiply': chx.multiply(x, b), 'exp': chx.exp(x), 'tanh': chx.tanh(x), 'relu': chx.relu(x),
                   'sum0': chx.sum(x, 0), 'sum1': chx.sum(x, 1), 'max1': chx.amax(x, 1), 'argmax1': chx.argmax(x, 1),
                   'log_softmax': chx.log_softmax(x, 1)}
        return {k: _out(a) for k, a in results.items()}
    if kind == 'cifar':
        return _out(cfg.cifar_forward(chx, state['p'], state['x']))
    if kind == 'resnet50':
        forward = cfg.resnet50_forward_fused if case['fused'] else cfg.resnet50_forward
        return _out(forward(chx, state['p'], state['x']))
    if kind == 'train':
        p = cfg.tree_map(lambda a: a, state['p'])  # the step puts new arrays into the tree it is given; every pass starts from the same ones
        loss = cfg.resnet50_train_step(state['ops'], p, state['x'], state['t'])
        blocks = [blk for stage in p['stages'] for blk in stage]
        results = [loss, p['conv1'], p['fc_w'], p['fc_b'], p['bn1']['gamma'], p['bn1']['beta'], blocks[-1]['bn3']['gamma'], blocks[-1]['bn3']['beta']]
        results += [blk[k] for blk in blocks for k in ('conv1', 'conv2', 'conv3', 'conv4') if k in blk]
        return [_out(a) for a in results + [state['statistics']]]
    if kind == 'lstm_lm':
        y, hs, cs = cfg.lstm_lm_forward(chx, state['p'], state['ids'], chx.zeros)
        return [_out(a) for a in [y] + hs + cs]
    if kind == 'rnn':
        xs = chx.split(state['x'], state['bounds'], 0)
        (hy, cy), ys, saved = chx.rnn(case['layers'], state['hx'], state['cx'], state['ws'], state['bs'], xs, case['bidirectional'], case['mode'],
                                      training=case['train'])
        results = [chx.concatenate(ys, 0), hy] + ([cy] if cy is not None else [])
        if case['train']:
            (dhx, dcx), dws, dbs, dxs = chx.rnn_backward(saved, state['dhy'], state['dcy'], chx.split(state['dy'], state['bounds'], 0))
            results += [dhx, chx.concatenate(dxs, 0)] + ([dcx] if dcx is not None else []) + dws[:24] + dbs[:24]
        return [_out(a) for a in results]
    x, w, gy = state['x'], state['w'], state['gy']
    return [_out(a) for a in (chx.linear(x, w, state['b']), chx.dot(gy, w), chx.dot(gy.T, x), chx.sum(gy, 0))]


def _cifar_work(case):
    it, b = np.dtype(case['dtype']).itemsize, case['batch']
    flops, params, c_in, side = 0, 0, 3, 32
    for i, c_out in enumerate(cfg.CIFAR_CHANNELS):
        flops += 2 * 9 * c_in * c_out * side * side
        params += 9 * c_in * c_out + 4 * c_out
        c_in = c_out
        side //= 1 + i % 2
    return {'flops': b * (flops + 20 * c_in), 'bytes': it * (b * (3 * 32 * 32 + 10) + params + 10 * c_in + 10)}


def _resnet_params():
    """(filters and classifier, batch-norm channels)."""
    filters, channels, c_in = 64 * 3 * 49, 64, 64
    for si, n_blocks in enumerate(cfg.RESNET50_BLOCKS):
        mid = 64 * 2 ** si
        for bi in range(n_blocks):
            filters += mid * c_in + 9 * mid * mid + 4 * mid * mid + (4 * mid * c_in if bi == 0 else 0)
            channels += 6 * mid + (4 * mid if bi == 0 else 0)
            c_in = 4 * mid
    return filters + 1001 * c_in - c_in + 1000, channels


def work(case):
    """Every input of the pass read once, every output written once, and its multiply-adds."""
    kind = case['kind']
    it = np.dtype(case.get('dtype', 'float32')).itemsize
    if kind == 'mlp':
        b, u = case['batch'], case['units']
        weights = 784 * u + u * u + 10 * u
        return {'flops': 2 * b * weights, 'bytes': it * (weights + 2 * u + 10 + b * (784 + 10)) + 4 * b}
    if kind == 'sweep':
        n, r, c = case['rows'] * case['cols'], case['rows'], case['cols']
        return {'flops': 14 * n, 'bytes': it * (7 * n + 2 * c + 2 * r) + 8 * r}  # six results are matrices
    if kind == 'cifar':
        return _cifar_work(case)
    if kind in ('resnet50', 'train'):
        b, s = case['batch'], case['size']
        weights, channels = _resnet_params()
        flops = cfg.resnet50_flops(b, s)
        if kind == 'resnet50':
            return {'flops': flops, 'bytes': 2 * (b * (3 * s * s + 1000) + weights + 4 * channels)}
        return {'flops': 3 * flops, 'bytes': 2 * (b * 3 * s * s + 2 * weights) + 4 * (8 * channels + b)}
    if kind == 'lstm_lm':
        b, t, u, v = case['batch'], case['seq'], case['units'], case['vocab']
        # the chain computes the output layer at every step
        return {'flops': 2 * b * t * (16 * u * u + u * v), 'bytes': it * (16 * u * u + 8 * u + u * v + v + min(v, b * t) * u + b * v + 4 * b * u) + 4 * b * t}
    if kind == 'rnn':
        d, u, g = (2 if case['bidirectional'] else 1), case['units'], _GATES[case['mode']]
        rows = sum(_step_sizes(case))
        weights = sum(d * g * u * ((u if layer == 0 else d * u) + u) for layer in range(case['layers']))
        biases = case['layers'] * d * 2 * g * u
        states = (2 if case['mode'] == 'lstm' else 1) * case['layers'] * d * case['batch'] * u
        once = weights + biases + 2 * states + rows * (u + d * u)
        return {'flops': (3 if case['train'] else 1) * 2 * rows * weights, 'bytes': 4 * once * (2 if case['train'] else 1)}
    r, i, o = case['rows'], case['n_in'], case['n_out']
    return {'flops': 6 * r * i * o, 'bytes': it * (2 * (r * i + o * i + o) + 2 * r * o)}


def tolerance(case):
    """float32 sums in another order; float16 results rounded once more or less per call, over the calls that follow each other."""
    kind = case['kind']
    if kind in ('resnet50', 'train'):
        return {'rel': 1e-2}
    if case.get('dtype', 'float32') == 'float32':
        return {'rel': 1e-5}
    return {'rel': 2e-3 if kind in ('sweep', 'linear') else 1e-2}
