"""CPU tests: what a convolution and its weight gradient ask of the library before they run answers for empty batches, channels and planes too.  The
questions go to a process of their own: an integer divided by zero ends it."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

ASK = '''
import ctypes, itertools
from chainer_amd import _lib
lib = _lib.load()

def array(shape, dtype):
    a = _lib.CArray(data=4096, dtype=dtype, ndim=len(shape))
    step = {7: 2, 8: 4}[dtype]
    for i in reversed(range(len(shape))):
        a.shape[i], a.strides[i] = shape[i], step
        step *= max(1, shape[i])
    return ctypes.byref(a)

one, answers = (ctypes.c_int64 * 2)(1, 1), set()
for dtype, n, c, k, h, w, size in itertools.product((7, 8), (0, 1, 40), (0, 3, 64), (0, 5), (0, 1, 9), (0, 9), (1, 3)):
    if 0 not in (n, c, k, h, w):
        continue
    pad = (ctypes.c_int64 * 2)(size // 2, size // 2)
    x, filters, y = array((n, c, h, w), dtype), array((k, c, size, size), dtype), array((n, k, h, w), dtype)
    answers.add(%s)
print(sorted(answers))
'''


@pytest.mark.parametrize('question,answers', [
    ('lib.hipcx_conv_grad_weight_workspace_size(x, y, filters, one, pad, 0) >= 0', '[True]'),
    ('lib.hipcx_conv_workspace_size(x, filters, y) >= 0', '[True]'),
    ('lib.hipcx_conv_route(x, filters, None, one, pad, y) if 0 in (n, k, h, w) else 0', '[0]'),
])
def test_empty_arrays(question, answers):
    done = subprocess.run([sys.executable, '-c', ASK % question], cwd=ROOT, capture_output=True, text=True)
    assert done.returncode == 0 and done.stdout.strip() == answers, (done.returncode, done.stdout, done.stderr[-500:])
