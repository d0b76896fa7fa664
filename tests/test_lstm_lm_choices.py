"""Which routines configs.lstm_lm_forward calls for its `fused` and `step` arguments."""
import numpy as np
import pytest

from chainer_amd import configs as cfg


class Recorder(object):
    def __init__(self, has_step):
        self.calls = []
        for name in ('take', 'linear', 'add', 'lstm', 'lstm_fused', 'log_softmax', 'log_softmax_fused') + (('lstm_step',) if has_step else ()):
            setattr(self, name, self._routine(name))

    def _routine(self, name):
        def run(*args):
            self.calls.append(name)
            return (args[0], args[0]) if name.startswith('lstm') else args[0]
        return run


@pytest.mark.parametrize('has_step,arguments,cell,softmax', [
    (True, {}, ['lstm_step'], 'log_softmax'), (True, {'step': True, 'fused': True}, ['lstm_step'], 'log_softmax_fused'),
    (True, {'step': False}, ['linear', 'linear', 'add', 'lstm'], 'log_softmax'),
    (True, {'fused': True}, ['linear', 'linear', 'add', 'lstm_fused'], 'log_softmax_fused'),
    (False, {}, ['linear', 'linear', 'add', 'lstm'], 'log_softmax'), (False, {'fused': True}, ['linear', 'linear', 'add', 'lstm_fused'], 'log_softmax_fused')])
def test_routines(has_step, arguments, cell, softmax):
    F = Recorder(has_step)
    cfg.lstm_lm_forward(F, cfg.lstm_lm_params(vocab=7, units=3), cfg.lstm_lm_input(batch=2, seq=2, vocab=7), np.zeros, **arguments)
    assert F.calls == (['take'] + cell + cell + ['linear']) * 2 + [softmax]
