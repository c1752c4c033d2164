"""``KnetArray``: a device array as (pointer, dims), column-major, float32/float64/int32.

Mirrors src/knetarrays/karray.jl:53-56 (``KnetArray{T,N}(ptr::KnetPtr, dims)``) and the storage side of
src/knetarrays/kptr.jl: the pointer comes from ``knet8_malloc`` (a size-class pool over ``hipMalloc``)
and goes back to the pool when the last array sharing it is collected, as the reference's finalizer
does (kptr.jl:105-142).  ``dims`` are Julia dims: the first varies fastest in memory.
"""
import copy
import ctypes

import numpy as np

from .libknet8 import host, libknet8

KnetPtr = host.KnetPtr   # owner of one device allocation; a block of a borrowed address if `keep` is given


class KnetArray(host.ArrayBase):
    """Dense column-major device array.  ``KnetArray(np_array)`` copies to the device, ``Array(k)`` back.

    The native base holds ``kptr, dims, dtype, offset`` and gives ``ptr, length, ndims, suffix, size, stride, similar``."""

    __array_priority__ = 1000

    def __init__(self, data=None, dtype=None, dims=None, _ptr=None, _offset=0):
        if _ptr is not None:
            self._init(_ptr, dims, dtype, int(_offset))
            return
        if data is None:
            self._init(None, dims, dtype if dtype is not None else np.float32)
            return
        a = np.asarray(data, dtype=dtype)
        if a.dtype not in (np.float32, np.float64, np.int32):
            raise TypeError("KnetArray supports Float32, Float64 and Int32 elements, got %s" % a.dtype)
        self._init(None, a.shape, a.dtype)
        flat = np.ascontiguousarray(a.ravel(order="F"))
        lib = libknet8()
        lib.fn["knet8_memcpy"](self.ptr, flat.ctypes.data, flat.nbytes, 1, lib.stream)
        lib.check()

    @property
    def ctype(self):
        return ctypes.c_float if self.dtype == np.float32 else ctypes.c_double

    # -- the copy and pickle protocols: the native base has no state that they could take by themselves ---
    def __copy__(self):
        """The same memory, as ``reshape`` shares it."""
        y = type(self).__new__(type(self))
        y._init(self.kptr, self.dims, self.dtype, self.offset)
        y.__dict__.update(self.__dict__)
        return y

    def __deepcopy__(self, memo):
        """Memory of its own with the same contents, as ``copy()``."""
        y = type(self).__new__(type(self))
        memo[id(self)] = y
        y._init(None, self.dims, self.dtype)
        libknet8().fn["knet8_memcpy"](y.ptr, self.ptr, self.length * self.dtype.itemsize, 3, libknet8().stream)
        y.__dict__.update(copy.deepcopy(self.__dict__, memo))
        return y

    def __reduce_ex__(self, protocol):
        """Through the host: the elements, which are uploaded where it is read."""
        return type(self), (self.to_numpy(),), self.__dict__ or None

    def __repr__(self):
        return "KnetArray{%s,%d}%r" % (self.dtype.name, self.ndims, self.dims)

    def reshape(self, *dims):
        """Shares the pointer (src/knetarrays/reshape.jl:3-11); one dim may be -1 (Julia's ``:``)."""
        if len(dims) == 1 and isinstance(dims[0], (tuple, list)):
            dims = dims[0]
        if -1 in dims:
            dims = list(dims)
            k = dims.index(-1)
            rest = 1
            for i, d in enumerate(dims):
                if i != k:
                    rest *= d
            dims[k] = self.length // rest if rest else 0
        y = self._view(dims)
        if y.length != self.length:
            raise ValueError("DimensionMismatch: new dimensions %r must be consistent with array size %d" % (tuple(dims), self.length))
        return y

    def view1d(self, start, n):
        """Contiguous sub-array of ``n`` elements starting at 0-based linear index ``start`` (shares memory)."""
        if start < 0 or start + n > self.length:
            raise IndexError("BoundsError")
        return self._view((n,), self.offset + start * self.dtype.itemsize)

    @classmethod
    def from_torch(cls, t, dims=None):
        """Wrap a contiguous torch device tensor without copying; ``dims`` are the Julia dims of its memory."""
        dt = {"torch.float32": np.float32, "torch.float64": np.float64, "torch.int32": np.int32}[str(t.dtype)]
        if not t.is_contiguous():
            raise ValueError("tensor must be contiguous")
        dims = tuple(reversed(t.shape)) if dims is None else tuple(dims)
        return cls(dtype=dt, dims=dims, _ptr=KnetPtr(nbytes=t.numel() * t.element_size(), ptr=t.data_ptr(), keep=t))

    # -- host transfer ---------------------------------------------------------------------------------
    def to_numpy(self):
        """``Array(x)``: copy back to the host (blocks until the data has landed)."""
        flat = np.empty(self.length, dtype=self.dtype)
        lib = libknet8()
        if self.length:
            lib.fn["knet8_memcpy"](flat.ctypes.data, self.ptr, flat.nbytes, 2, lib.stream)
            lib.check()
        return flat.reshape(self.dims, order="F")

    def copy(self):
        y = self.similar()
        lib = libknet8()
        lib.fn["knet8_memcpy"](y.ptr, self.ptr, self.length * self.dtype.itemsize, 3, lib.stream)
        return y

    # -- operators: defined in ops20 / binary and attached there --------------------------------------


host.array_type(KnetArray)


def number(x, v):
    """``v`` as an argument of the element type of ``x``: numbers as they are, anything else as ctypes converts or refuses it."""
    return v if isinstance(v, (float, int, np.floating)) else x.ctype(v)


def Array(x):
    return x.to_numpy() if isinstance(x, KnetArray) else np.asarray(x)


def upload(data):
    """Device array of a contiguous host vector for launches that follow on the current stream: the caller does not wait for the copy (``knet8_upload``).
    For arrays that stay inside one operation; ``KnetArray(data)`` is ready on every stream."""
    a = np.ascontiguousarray(data)
    k = KnetArray(dtype=a.dtype, dims=a.shape)
    lib = libknet8()
    if lib.fn["knet8_upload"](k.ptr, a.ctypes.data, a.nbytes, lib.stream) != 0:
        lib.check()
    return k


def synchronize():
    lib = libknet8()
    lib.fn["knet8_synchronize"](lib.stream)
    lib.check()


class Graph:
    """A captured launch sequence (hipGraph).  ``replay()`` launches it on the stream it was captured on; ``outputs`` is what the
    captured function returned (device arrays whose contents every replay overwrites)."""

    def __init__(self, handle, stream, outputs, parked):
        self.handle, self.stream, self.outputs, self._parked = handle, stream, outputs, parked

    def replay(self):
        lib = libknet8()
        if lib.fn["knet8_graph_launch"](self.handle, self.stream) != 0:
            lib.check()
            raise RuntimeError("graph launch failed")

    def __del__(self):
        try:
            lib = libknet8()
            lib.fn["knet8_synchronize"](self.stream)
            lib.fn["knet8_graph_destroy"](self.handle)
            for p in self._parked:
                lib.fn["knet8_free"](p)
        except Exception:
            pass


_CAPTURE_STREAM = None


def capture_stream():
    """The stream ``capture`` records on: created at first use, owned by the package, destroyed at interpreter exit."""
    global _CAPTURE_STREAM
    if _CAPTURE_STREAM is None:
        import atexit
        lib = libknet8()
        _CAPTURE_STREAM = lib.fn["knet8_stream_create"]()

        def _destroy():
            global _CAPTURE_STREAM
            if _CAPTURE_STREAM is not None:
                try:
                    if lib.stream == _CAPTURE_STREAM:
                        lib.stream = None
                    lib.fn["knet8_stream_destroy"](_CAPTURE_STREAM)
                except Exception:
                    pass
                _CAPTURE_STREAM = None
        atexit.register(_destroy)
    return _CAPTURE_STREAM


def capture(fn):
    """Run ``fn()`` once eagerly (so that pool blocks, reduction scratch and GEMM plans exist), then once more under
    stream capture, and return a ``Graph``.  ``fn`` must not synchronise with the host (no ``Array(x)``, no ``dims=:``
    reductions, no host labels): it may only enqueue work."""
    lib = libknet8()
    if lib.stream is None:
        # Capture needs a stream of its own.  Work already queued on the null stream (fills, copies and random draws that built the
        # parameters) must have landed first: a non-blocking stream does not wait for the null stream.  The stream is created once,
        # kept as the package's capture stream and destroyed when the interpreter exits; the caller restores `lib.stream` if it wants
        # the null stream back.
        lib.fn["knet8_synchronize"](None)
        lib.stream = capture_stream()
    # Warm-up under the same parking rule as the capture itself, so that the pool ends up holding one block for every
    # allocation of the sequence (blocks freed while parked are not recycled within the run).
    warm = []
    host.park(warm)
    try:
        fn()
    finally:
        host.park(None)
    lib.fn["knet8_synchronize"](lib.stream)
    for p in warm:
        lib.fn["knet8_free"](p)
    lib.check()
    parked = []
    # While the sequence is being captured, blocks that are released must not go back to the pool: the graph keeps using their addresses, and owns them.
    host.park(parked)
    try:
        if lib.fn["knet8_graph_begin"](lib.stream) != 0:
            lib.check()
        try:
            out = fn()
        finally:
            handle = lib.fn["knet8_graph_end"](lib.stream)
    finally:
        host.park(None)
    if not handle:
        lib.check()
        raise RuntimeError("graph capture failed")
    return Graph(handle, lib.stream, out, parked)
