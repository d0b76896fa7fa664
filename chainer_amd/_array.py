"""Device array of the ``hip`` backend, seen from Python.

It plays the role of ``chainerx.ndarray`` for the harness and the tests: a (buffer, offset, shape,
byte-strides, dtype) tuple, with views made on the host and every arithmetic operation forwarded
to one C-ABI kernel call.  Device memory comes from the library's own pool (``hipcx_malloc`` /
``hipcx_free``) and crosses the host boundary through its copy entry points
(``hipcx_from_host_memory``, ``hipcx_memcpy_to_host``): the Device interface of the backend.
PyTorch is only asked for the current stream (and captures HIP graphs in the benchmarks).
"""
import ctypes

import numpy

from chainer_amd import _lib

# chainerx::Dtype codes (CX/dtype.h:19-29)
_DTYPE_CODES = {
    numpy.dtype('bool'): 1,
    numpy.dtype('int8'): 2,
    numpy.dtype('int16'): 3,
    numpy.dtype('int32'): 4,
    numpy.dtype('int64'): 5,
    numpy.dtype('uint8'): 6,
    numpy.dtype('float16'): 7,
    numpy.dtype('float32'): 8,
    numpy.dtype('float64'): 9,
}

_torch = None
_host = _lib.host()


def torch():
    global _torch
    if _torch is None:
        import torch as _t
        _torch = _t
    return _torch


def device_available():
    return torch().cuda.is_available()


def _require_device():
    if not torch().cuda.is_available():
        raise _lib.BackendError('no HIP device is visible: the hip backend has no CPU fallback')


def _start_device():
    """Before the first allocation or stream look-up: checks for a device, initialises PyTorch's side of the runtime and takes its
    stream functions, which a build of PyTorch without device support does not have."""
    _require_device()
    torch().cuda.init()
    _host.setup({'raw_stream': torch()._C._cuda_getCurrentRawStream, 'get_device': torch()._C._cuda_getDevice})


def current_stream():
    return ctypes.c_void_p(_host.current_stream())


def synchronize():
    """Device::Synchronize (CX/device.h:71).  Raises the IndexError of an earlier take / add_at (default bounds mode) whose indices
    were out of range."""
    torch().cuda.synchronize()
    _lib.call('hipcx_synchronize', DEVICE_INDEX)


def dtype_code(dtype):
    try:
        return _DTYPE_CODES[numpy.dtype(dtype)]
    except KeyError:
        raise _lib.DtypeError('unsupported dtype: %s' % (dtype,))


def contiguous_strides(shape, itemsize):
    """C-contiguous byte strides; zero-sized axes count as 1 (CX/strides.cc:17-26)."""
    st = []
    acc = itemsize
    for d in reversed(shape):
        st.append(acc)
        acc *= max(1, d)
    return tuple(reversed(st))


DEVICE_INDEX = 0


DeviceBuffer = _host.DeviceBuffer


def alloc_bytes(nbytes):
    return DeviceBuffer(nbytes)


def pool_stats():
    """Counters of the device memory pool (hipcx_pool_stats)."""
    st = _lib.CPoolStats()
    _lib.call('hipcx_pool_stats', DEVICE_INDEX, ctypes.byref(st))
    return {name: int(getattr(st, name)) for name, _ in _lib.CPoolStats._fields_}


def free_unused_blocks():
    """MemoryPool::FreeUnusedBlocks (CX/cuda/memory_pool.cc:172-203)."""
    _lib.call('hipcx_pool_free_unused', DEVICE_INDEX)


_next_arena = [1]


class memory_arena(object):
    """Allocations made inside the ``with`` block come from, and return to, free lists of their own.  A HIP graph is
    captured inside one (after an eager pass in the same arena has filled its free lists, so that the capture itself never
    reaches the driver): the addresses baked into the graph are then not handed to anybody else until ``release()``."""

    def __init__(self):
        self.id = _next_arena[0]
        _next_arena[0] += 1

    def __enter__(self):
        _lib.call('hipcx_pool_set_arena', DEVICE_INDEX, self.id)
        return self

    def __exit__(self, *exc):
        _lib.call('hipcx_pool_set_arena', DEVICE_INDEX, 0)
        return False

    def release(self):
        _lib.call('hipcx_pool_release_arena', DEVICE_INDEX, self.id)


class ndarray(_host.ArrayBase):
    """Strided view of device memory.  Fields, views, copies and descriptors are native (csrc/python/array.cc)."""

    __slots__ = ()

    def record_stream(self, stream=None):
        """See DeviceBuffer.record_stream: call it when the array is used on a stream other than the one it was created on and may
        be dropped before that stream is waited for."""
        self._buf.record_stream(stream)

    def __repr__(self):
        return 'chainer_amd.ndarray(shape=%r, dtype=%s, strides=%r, device=hip:0)' % (self.shape, self.dtype, self.strides)

    def get(self):
        """Device -> host (numpy) copy; synchronises like Array::ToNative (CX/array.cc:399-444)."""
        a = self.as_contiguous()
        n = a.size * a.itemsize
        host = numpy.empty(a.shape, a.dtype)
        if n == 0:
            return host
        _lib.call('hipcx_memcpy_to_host', DEVICE_INDEX, ctypes.c_void_p(host.ctypes.data), ctypes.c_void_p(a._ptr), n, current_stream())
        return host

    def __array__(self, dtype=None, copy=None):
        a = self.get()
        return a if dtype is None else a.astype(dtype)

    def item(self):
        return self.get().item()

    def __float__(self):
        return float(self.item())

    def __int__(self):
        return int(self.item())

    # arithmetic operators are attached by chainer_amd.routines


def _prod(xs):
    n = 1
    for x in xs:
        n *= int(x)
    return n


def _as_shape(shape):
    if isinstance(shape, (int, numpy.integer)):
        return (int(shape),)
    return tuple(int(s) for s in shape)


def _normalize_axis(axis, ndim):
    axis = int(axis)
    if axis < -ndim or axis >= ndim:
        raise _lib.DimensionError('axis %d is out of bounds for array of dimension %d' % (axis, ndim))
    return axis + ndim if axis < 0 else axis


_nocopy_reshape_strides = _host.nocopy_reshape_strides  # strides of a new shape over the same memory, or None if a copy is needed

_host.setup({
    'ndarray': ndarray,
    'dtypes': [None] + [dt for dt, _ in sorted(_DTYPE_CODES.items(), key=lambda item: item[1])],
    'np_dtype': numpy.dtype, 'np_bool': numpy.bool_, 'np_integer': numpy.integer, 'np_floating': numpy.floating,
    'require_device': _start_device,
})


def array(obj, dtype=None):
    """Host -> device upload: chainerx.array(numpy_array, device='hip:0') (Device::FromHostMemory)."""
    if isinstance(obj, ndarray):
        return obj.astype(dtype if dtype is not None else obj.dtype)
    a = numpy.asarray(obj, dtype=dtype)
    dtype_code(a.dtype)
    a = numpy.ascontiguousarray(a)
    _require_device()
    if a.size == 0:
        return ndarray.empty(a.shape, a.dtype)
    out = ctypes.c_void_p()
    _lib.call('hipcx_from_host_memory', DEVICE_INDEX, ctypes.c_void_p(a.ctypes.data), a.nbytes, ctypes.byref(out), current_stream())
    buf = DeviceBuffer.adopt(out.value, a.nbytes)
    return ndarray(buf, 0, a.shape, contiguous_strides(a.shape, a.dtype.itemsize), a.dtype)


def to_numpy(a):
    return a.get()
