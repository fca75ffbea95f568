"""Argument marshalling for one C-ABI call.

Inputs accept numpy arrays, host tensors or device tensors and are forced to
the kernel's dtype (the reference's pybind ``forcecast``).  Outputs are either
device tensors (written in place, asynchronously) or numpy arrays (a device
temporary is written and copied back after the call, which synchronizes the
stream).  Every buffer is checked to hold at least the elements the kernel
will touch before anything is uploaded or launched.
"""

from __future__ import annotations

import numpy as np

from asdsl import _hip

try:
    from torch import Tensor as _Tensor
    from torch import float32 as _f32
    from torch import int8 as _i8
    from torch import int32 as _i32
    from torch import uint8 as _u8

    _TORCH_DTYPE = {np.float32: _f32, np.int8: _i8, np.uint8: _u8, np.int32: _i32, np.uint32: _i32}
except ImportError:  # host arrays only: every buffer takes _Slot's way, whose upload reports it
    class _Tensor:
        pass

    _TORCH_DTYPE = {}


def _numel(a) -> int:
    if isinstance(a, _Tensor):
        return a.numel()
    return int(np.asarray(a).size)


def shape_of(a) -> tuple:
    if isinstance(a, _Tensor):
        return tuple(a.shape)
    return tuple(np.shape(a))


def on_device(*arrays) -> bool:
    for a in arrays:
        if isinstance(a, _Tensor) and a.is_cuda:
            return True
    return False


def new_output(shape, dtype, *like):
    """Output array for a returning wrapper: a device tensor when any input is
    one (the call stays asynchronous on the current stream), else numpy."""
    if on_device(*like):
        return _hip.empty_device(shape, dtype)
    return np.empty(shape, dtype)


class _Slot:
    __slots__ = ("array", "dtype", "n", "name", "is_output")

    def __init__(self, array, dtype, n, name, is_output):
        self.array, self.dtype, self.n, self.name, self.is_output = array, np.dtype(dtype), n, name, is_output


class _Scratch:
    __slots__ = ("n", "dtype")

    def __init__(self, n, dtype):
        self.n, self.dtype = n, dtype


class DeviceCall:
    """One C-ABI call.  input() and output() check a buffer and return what
    run() takes in its place: the address itself for a contiguous device tensor
    of the kernel's dtype (the caller holds the tensor until its call returns),
    a _Slot for anything that has to be uploaded or copied back.  The layer
    GEMVs take 3-10 us on the device, so this path is what bounds a program
    that calls them one by one: with every buffer a _Slot resolved in run() a
    3072 x 3072 GEMV took 12.8 us of host time a call, this way it takes 7.2
    (3.2 of them the launch)."""

    __slots__ = ("fn", "plain")

    def __init__(self, fn: str):
        self.fn = fn
        self.plain = True  # every argument so far is a plain value

    def _check(self, a, dtype, n: int, name: str, is_output: bool) -> _Slot:
        if a is None:
            raise ValueError(f"{self.fn}: {name} is None")
        have = _numel(a)
        if have < n:
            raise ValueError(f"{self.fn}: {name} has {have} elements, needs {n}")
        if is_output:
            if isinstance(a, _Tensor):
                if not a.is_cuda or a.dtype != _TORCH_DTYPE[dtype] or not a.is_contiguous():
                    raise ValueError(f"{self.fn}: {name} must be a contiguous {np.dtype(dtype).name} device tensor")
            elif not isinstance(a, np.ndarray) or a.dtype != np.dtype(dtype) or not a.flags.c_contiguous:
                raise ValueError(f"{self.fn}: {name} must be a C-contiguous {np.dtype(dtype).name} array")
        self.plain = False
        return _Slot(a, dtype, n, name, is_output)

    def input(self, a, dtype, n: int, name: str):
        if isinstance(a, _Tensor) and a.is_cuda and a.dtype is _TORCH_DTYPE[dtype] and a.numel() >= n \
                and a.is_contiguous():
            return a.data_ptr()
        return self._check(a, dtype, n, name, False)

    def output(self, a, dtype, n: int, name: str):
        if isinstance(a, _Tensor) and a.is_cuda and a.dtype is _TORCH_DTYPE[dtype] and a.numel() >= n \
                and a.is_contiguous():
            return a.data_ptr()
        return self._check(a, dtype, n, name, True)

    def scratch(self, n: int, dtype) -> "_Scratch":
        """Device-only temporary of n elements (never copied back)."""
        self.plain = False
        return _Scratch(n, dtype)

    def run(self, entry: str, *args) -> None:
        if self.plain:
            _hip.call(entry, *args, _hip.stream_handle())
            return
        keep, copyback, cargs = [], [], []
        for a in args:
            if isinstance(a, _Scratch):
                t = _hip.empty_device((max(a.n, 1),), a.dtype)
                keep.append(t)
                cargs.append(t.data_ptr())
                continue
            if not isinstance(a, _Slot):
                cargs.append(a)
                continue
            if a.is_output:  # a device tensor that passed the checks is an address already
                t = _hip.empty_device((a.n,), a.dtype)
                keep.append(t)
                copyback.append((a.array, t, a.n))
                cargs.append(t.data_ptr())
            else:
                t = _hip.to_device(a.array, a.dtype)
                keep.append(t)
                cargs.append(t.data_ptr())
        _hip.call(entry, *cargs, _hip.stream_handle())
        for host, dev, n in copyback:
            host.reshape(-1)[:n] = dev.cpu().numpy().view(host.dtype)
