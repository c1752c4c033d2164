"""The native part of the host mirror, on the CPU: calls are checked against Python functions bound in the place of entry points, arrays over made-up addresses."""
import copy
import ctypes
import gc
import importlib.machinery
import itertools
import pickle
import sys

import numpy as np
import pytest

CTYPES = {"v": None, "i": ctypes.c_int, "u": ctypes.c_ulonglong, "l": ctypes.c_longlong, "f": ctypes.c_float, "d": ctypes.c_double, "c": ctypes.c_char, "p": ctypes.c_void_p}
VALUES = {"i": (7, -3, 2 ** 31 - 1), "u": (2 ** 64 - 1, 5), "l": (-2 ** 62, 9), "f": (1.5, np.float32(0.1), 3), "d": (0.1, -7, np.float64(2.5)), "c": (b"N", b"T"), "p": (0xfedcba9876543210, None, 64)}


def native(knet):
    return sys.modules["knet_jl_amd.libknet8"]


def signatures(knet):
    lk = native(knet)
    return sorted({lk._LETTERS[r] + "".join(lk._LETTERS.get(a, "p") for a in args) for n, (r, args) in knet.libknet8().decls.items() if n.endswith("_stream")})


def test_every_signature_carries_its_arguments(knet):
    lk = native(knet)
    for sig in signatures(knet):
        got = []
        proto = ctypes.CFUNCTYPE(*[CTYPES[c] for c in sig])
        cb = proto(lambda *a: (got.append(a), {"v": None, "i": -5, "f": 1.25, "d": 0.1}[sig[0]])[1])
        lib = lk.host.Library()
        assert lib._bind("f", ctypes.cast(cb, ctypes.c_void_p).value, sig)
        lib.stream = 0x1234
        for turn in range(3):
            args = [VALUES[c][(turn + i) % len(VALUES[c])] for i, c in enumerate(sig[1:-1])]
            assert lib.call("f", *args) == {"v": None, "i": -5, "f": 1.25, "d": 0.1}[sig[0]]
            want = [(CTYPES[c](a).value if c != "p" else a) for c, a in zip(sig[1:], args)] + [0x1234]
            assert list(got[-1]) == want, sig
        assert not lib._bind("g", 1, sig + "zz")


def test_what_is_not_converted_goes_to_ctypes(knet):
    """Other argument types, wrong counts and unknown names are ctypes' to convert or refuse, as before there was a native call."""
    lk = native(knet)
    seen = []

    class Lib(lk.host.Library):
        def slow_call(self, fun, *args):
            seen.append((fun,) + args)
            return "slow"
    cb = ctypes.CFUNCTYPE(None, ctypes.c_int, ctypes.c_float, ctypes.c_void_p, ctypes.c_void_p)(lambda *a: None)
    lib = Lib()
    lib._bind("fill", ctypes.cast(cb, ctypes.c_void_p).value, "vifpp")
    assert lib.call("fill", 3, 1.0, 8) is None and not seen
    for bad in ((3, ctypes.c_float(1), 8), (3.0, 1.0, 8), (np.int64(3), 1.0, 8), (3, "1.0", 8), (3, 1.0, "8"), (3, 1.0, (ctypes.c_int * 2)()), (3, 1.0), (3, 1.0, 8, 9)):
        assert lib.call("fill", *bad) == "slow" and seen[-1][1:] == bad
    assert lib.call("other", 1) == "slow"
    real = knet.libknet8()
    with pytest.raises(KeyError):
        real.call("no_such_entry", 1)
    with pytest.raises(ctypes.ArgumentError):
        real.call("fill_32", 1, "a", 0)


@pytest.mark.parametrize("dims", [(), (5,), (3, 4), (2, 1, 7, 3), (0, 4)])
def test_arrays_answer_like_their_dims(knet, dims):
    ptr = knet.KnetPtr(nbytes=4, ptr=0x10000, keep=object())
    for dt, suffix in ((np.float32, "32"), (np.float64, "64"), (np.int32, None), (np.uint8, None)):
        x = knet.KnetArray(dtype=dt, dims=[np.int64(d) for d in dims], _ptr=ptr, _offset=16)
        n = int(np.prod(dims, dtype=np.int64))
        assert x.dims == dims and all(type(d) is int for d in x.dims) and x.length == n and x.ndims == len(dims) and x.size() == dims
        assert x.dtype == np.dtype(dt) and x.suffix == suffix and x.ptr == 0x10010 and x.offset == 16 and x.kptr is ptr
        for i in range(1, len(dims) + 3):
            assert x.size(i) == (dims[i - 1] if i <= len(dims) else 1) and x.stride(i) == int(np.prod(dims[:i - 1], dtype=np.int64))
        y = x.reshape(-1) if n else x.reshape(n)
        assert y.dims == (n,) and y.kptr is ptr and y.ptr == x.ptr and copy.copy(x).ptr == x.ptr
        with pytest.raises(ValueError):
            x.reshape(n + 1)
    with pytest.raises(TypeError):
        knet.KnetArray(np.zeros(3, np.uint8))


def test_blocks_go_back_once_or_are_parked(knet):
    lk = native(knet)
    freed, blocks = [], itertools.count(0x100000, 0x1000)
    alloc = ctypes.CFUNCTYPE(ctypes.c_void_p, ctypes.c_size_t)(lambda n: 0 if n == 4 * 99 else next(blocks))
    free = ctypes.CFUNCTYPE(None, ctypes.c_void_p)(lambda p: freed.append(p))

    def refuse():
        raise MemoryError("Out of gpu memory")
    address = lambda f: ctypes.cast(f, ctypes.c_void_p).value  # noqa: E731
    real, dtypes = knet.libknet8(), tuple(np.dtype(t) for t in (np.float32, np.float64, np.int32))
    lk.host.setup(address(alloc), address(free), refuse, np.dtype, dtypes, real)
    try:
        x = knet.KnetArray(dtype=np.float32, dims=(3, 5))
        y, p = x.reshape(15), x.ptr
        del x
        assert not freed
        z = y.similar((2, 2), dtype=np.float64)
        assert z.dtype == np.float64 and z.kptr.nbytes == 32 and y.similar(dims=[4]).dims == (4,)
        freed.clear()
        del y
        assert freed == [p]
        parked = []
        lk.host.park(parked)
        q = z.ptr
        del z
        lk.host.park(None)
        assert parked == [q] and freed == [p]
        with pytest.raises(MemoryError):
            knet.KnetArray(dtype=np.float32, dims=(99,))
        knet.KnetPtr(nbytes=4, ptr=0x5000, keep=object())
        knet.KnetPtr(nbytes=4, ptr=0x6000)                     # an address without an owner is the caller's to give away
        assert freed == [p, 0x6000]
        late = knet.KnetPtr(nbytes=4, ptr=0x8000)
        late._keep = object()                                  # somebody else's after all
        del late
        assert freed == [p, 0x6000]
        # a cycle through what keeps borrowed memory alive is collected, and the memory is not given back
        class Keep:
            pass
        k = Keep()
        k.array = knet.KnetArray(dtype=np.float32, dims=(1,), _ptr=knet.KnetPtr(nbytes=4, ptr=0x7000, keep=k))
        del k
        gc.collect()
        assert not any(isinstance(o, Keep) for o in gc.get_objects()) and freed == [p, 0x6000]
    finally:
        gc.collect()
        lk.host.setup(address(real.fn["knet8_malloc"]), address(real.fn["knet8_free"]), lk._out_of_memory, np.dtype, dtypes, real)


def test_similar_refuses_what_it_refused(knet):
    x = knet.KnetArray(dtype=np.float32, dims=(2,), _ptr=knet.KnetPtr(nbytes=4, ptr=0x10000, keep=object()))
    for args, kw in (((1, 2, 3), {}), ((), {"shape": (2,)}), ((5,), {}), ((("a",),), {})):
        with pytest.raises((TypeError, ValueError)):
            x.similar(*args, **kw)


def test_block_and_element_type_can_be_replaced(knet):
    """As of the attributes they were before there was a native class."""
    a, b = (knet.KnetPtr(nbytes=64, ptr=p, keep=object()) for p in (0x10000, 0x20000))
    x = knet.KnetArray(dtype=np.float32, dims=(2, 3), _ptr=a, _offset=8)
    x.kptr = b
    assert x.kptr is b and x.ptr == 0x20008 and x.reshape(6).ptr == 0x20008
    x.dtype = np.float64
    assert x.dtype == np.float64 and x.suffix == "64" and x.view1d(1, 2).ptr == 0x20010
    x.dtype = "int32"
    assert x.suffix is None
    with pytest.raises(TypeError):
        x.kptr = 5
    with pytest.raises(TypeError):
        x.dtype = "no such type"
    assert x.kptr is b and x.dtype == np.int32
    a.nbytes = 32
    assert a.nbytes == 32
    x.note, x.offset = "kept", 16                 # any other attribute as ever
    assert x.note == "kept" and x.ptr == 0x20010
    for name in ("dtype", "kptr", "ptr", "length"):
        with pytest.raises((AttributeError, TypeError)):
            delattr(x, name)
    with pytest.raises(AttributeError):
        x.length = 5
    with pytest.raises(AttributeError):
        knet.KnetArray.__new__(knet.KnetArray).dtype


def test_module_is_for_this_interpreter(knet, monkeypatch):
    lk = native(knet)
    assert lk.HOST_PATH.endswith(importlib.machinery.EXTENSION_SUFFIXES[0]) and sys.implementation.cache_tag in lk.HOST_PATH
    monkeypatch.setattr(lk, "HOST_PATH", lk.HOST_PATH.replace(sys.implementation.cache_tag, "cpython-399"))
    with pytest.raises(OSError, match="not found"):
        lk._load_host()


@pytest.mark.parametrize("dt,suffix", [(np.float32, "32"), (np.float64, "64"), (np.int32, None)])
def test_element_types_are_told_by_equality(knet, monkeypatch, dt, suffix):
    """A pickled array comes back with a dtype object of its own, and slices, products and transposes of it carry that on."""
    a = pickle.loads(pickle.dumps(np.ones((3, 4), dt)))
    assert a.dtype == dt and a.dtype is not np.dtype(dt)
    ptr = knet.KnetPtr(nbytes=4096, ptr=0x10000, keep=object())
    for d in (a.dtype, a[1:].dtype, (a * dt(2)).dtype, a.T.dtype, pickle.loads(pickle.dumps(np.dtype(dt)))):
        x = knet.KnetArray(dtype=d, dims=(3, 4), _ptr=ptr)
        for y in (x, x.reshape(12), x.view1d(2, 5)):
            assert y.suffix == suffix and y.dtype is np.dtype(dt)
    other = knet.KnetArray(dtype=np.uint8, dims=(2,), _ptr=ptr)
    blocks, address = itertools.count(0x100000, 0x1000), lambda f: ctypes.cast(f, ctypes.c_void_p).value  # noqa: E731
    alloc, free = ctypes.CFUNCTYPE(ctypes.c_void_p, ctypes.c_size_t)(lambda n: next(blocks)), ctypes.CFUNCTYPE(None, ctypes.c_void_p)(lambda p: None)
    lk, real, dtypes = native(knet), knet.libknet8(), tuple(np.dtype(t) for t in (np.float32, np.float64, np.int32))
    lk.host.setup(address(alloc), address(free), lk._out_of_memory, np.dtype, dtypes, real)
    try:
        monkeypatch.setitem(real.fn, "knet8_memcpy", lambda *args: 0)
        monkeypatch.setattr(real, "check", lambda: None)
        x = knet.KnetArray(a)
        assert x.suffix == suffix and x.similar().suffix == suffix and x.similar((2,)).suffix == suffix
        assert other.similar((2, 2), dtype=a.dtype).suffix == suffix and x.kptr.nbytes == 12 * np.dtype(dt).itemsize
        assert knet.KnetArray(dtype=">f4", dims=(2,)).suffix is None                  # another byte order is another type
        del x
    finally:
        gc.collect()
        lk.host.setup(address(real.fn["knet8_malloc"]), address(real.fn["knet8_free"]), lk._out_of_memory, np.dtype, dtypes, real)


@pytest.mark.parametrize("dt", [np.float32, np.float64, np.int32])
@pytest.mark.parametrize("dims", [(3, 4), (5,), (2, 3, 2), (0, 4), ()])
def test_arrays_are_copied_and_pickled(knet, monkeypatch, dims, dt):
    """copy, deepcopy and pickle of arrays and of what holds them, over host memory in the place of the device's."""
    lk, real, dtypes = native(knet), knet.libknet8(), tuple(np.dtype(t) for t in (np.float32, np.float64, np.int32))
    held, address = {}, lambda f: ctypes.cast(f, ctypes.c_void_p).value  # noqa: E731

    def take(n):
        b = ctypes.create_string_buffer(n)
        held[ctypes.addressof(b)] = b
        return ctypes.addressof(b)
    alloc, free = ctypes.CFUNCTYPE(ctypes.c_void_p, ctypes.c_size_t)(take), ctypes.CFUNCTYPE(None, ctypes.c_void_p)(lambda p: held.pop(p))
    lk.host.setup(address(alloc), address(free), lk._out_of_memory, np.dtype, dtypes, real)
    try:
        monkeypatch.setitem(real.fn, "knet8_memcpy", lambda to, of, n, kind, stream: ctypes.memmove(to, of, n))
        monkeypatch.setattr(real, "check", lambda: None)
        want = np.arange(np.prod(dims, dtype=int)).reshape(dims).astype(dt)
        x = knet.KnetArray(want)
        x.note = ["mine"]
        same = copy.copy(x)
        assert same.kptr is x.kptr and same.dims == dims and same.note is x.note
        for y in (copy.deepcopy(x), *(pickle.loads(pickle.dumps(x, p)) for p in range(2, pickle.HIGHEST_PROTOCOL + 1))):
            assert type(y) is knet.KnetArray and y.ptr != x.ptr and y.dtype is x.dtype and y.suffix == x.suffix and y.dims == dims
            assert np.array_equal(y.to_numpy(), want) and y.note == x.note and y.note is not x.note
        if len(dims) == 2 and want.size:                  # a part of a block: its own elements, in a block of their size
            part = x.view1d(4, 3)
            y = copy.deepcopy(part)
            assert y.kptr.nbytes == 3 * want.itemsize and np.array_equal(y.to_numpy(), want.ravel(order="F")[4:7])
        if dt != np.int32:                                # a model and its optimizer: arrays shared within stay shared, and the copy lives by itself
            w = knet.Param(x)
            w.opt = knet.Momentum(lr=0.5)
            w.opt.velocity = x
            v = copy.deepcopy([w, w])
            assert v[0] is v[1] and v[0].value is v[0].opt.velocity and v[0].value.ptr != x.ptr
            del w, x, same
            gc.collect()
            assert np.array_equal(v[0].value.to_numpy(), want)
            del v
        x = same = y = part = None
        gc.collect()
        assert not held
    finally:
        gc.collect()
        lk.host.setup(address(real.fn["knet8_malloc"]), address(real.fn["knet8_free"]), lk._out_of_memory, np.dtype, dtypes, real)
