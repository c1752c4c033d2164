"""Small uploads in order with the launches behind them: around the staging buffer's end, the sizes that take the waiting copy, streams and threads."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# bytes / 4: one element, around a block of the copy kernel, the largest staged (64 KB) and one more
@pytest.mark.parametrize("n", [0, 1, 255, 256, 257, 16383, 16384, 16385])
def test_upload_sizes(knet, n):
    from knet_jl_amd.karray import upload
    a = np.arange(n, dtype=np.int32) * 7 - 3
    assert np.array_equal(knet.Array(upload(a)), a)
    knet.libknet8().check()


def test_many_uploads_wrap_the_buffer(knet):
    """60 x 12 KB through 256 KB, each read by a launch queued behind it and its host array overwritten at once."""
    from knet_jl_amd.karray import upload
    rng = np.random.default_rng(2)
    x = rng.standard_normal(50000).astype(np.float32)
    xd = knet.KnetArray(x)
    idx = np.empty(3000, np.int32)
    got, want = [], []
    for _ in range(60):
        idx[:] = rng.integers(1, x.size + 1, size=idx.size)
        d = upload(idx)
        y = xd.similar((idx.size,))
        knet.knet8("getents_32", idx.size, d.ptr, xd.ptr, y.ptr)
        got.append((d, y))
        want.append(x[idx - 1])
        idx[:] = 1
    for (_, y), w in zip(got, want):
        assert np.array_equal(knet.Array(y), w)
    knet.libknet8().check()


def test_streams_and_threads(knet):
    """Each stream has a buffer of its own, given back with the stream; sums from several threads on one stream keep their own results."""
    lib = knet.libknet8()
    fn = lib.fn
    streams = [fn["knet8_stream_create"]() for _ in range(3)]
    wrong = []

    def work(s, seed):
        rng = np.random.default_rng(seed)
        for _ in range(40):
            a = rng.integers(-1000, 1000, size=5000).astype(np.float32)
            p = fn["knet8_malloc"](a.nbytes)
            if fn["knet8_upload"](p, a.ctypes.data, a.nbytes, s) != 0 or fn["sum_32_20_stream"](a.size, p, s) != float(a.sum(dtype=np.float64)):
                wrong.append(seed)
            fn["knet8_synchronize"](s)
            fn["knet8_free"](p)
    knet.synchronize()
    threads = [threading.Thread(target=work, args=(streams[i % 3], i)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in streams:
        fn["knet8_stream_destroy"](s)
    assert not wrong
    fn["knet8_trim"]()
    assert float(knet.sum(knet.KnetArray(np.ones(100, np.float32)))) == 100.0
    lib.check()


def test_upload_without_staging_memory(knet):
    """No page-locked memory for a stream's buffer (knet8_tune key 5): the bytes arrive by the copy that waits, and there is no error."""
    lib = knet.libknet8()
    fn = lib.fn
    a, back = np.arange(1000, dtype=np.int32), np.empty(1000, np.int32)
    s, p = fn["knet8_stream_create"](), fn["knet8_malloc"](a.nbytes)
    old = fn["knet8_tune"](5, 1)
    try:
        assert fn["knet8_upload"](p, a.ctypes.data, a.nbytes, s) == 0
    finally:
        fn["knet8_tune"](5, old)
    fn["knet8_memcpy"](back.ctypes.data, p, a.nbytes, 2, s)
    assert np.array_equal(a, back)
    a += 5
    assert fn["knet8_upload"](p, a.ctypes.data, a.nbytes, s) == 0
    fn["knet8_memcpy"](back.ctypes.data, p, a.nbytes, 2, s)
    assert np.array_equal(a, back)
    fn["knet8_stream_destroy"](s)
    fn["knet8_free"](p)
    lib.check()


def test_per_thread_stream(knet):
    """hipStreamPerThread is one handle (2) for a stream of each thread: uploads from several threads, enough to use a staging buffer up, keep their bytes."""
    lib = knet.libknet8()
    fn = lib.fn
    wrong = []

    def work(seed):
        rng = np.random.default_rng(seed)
        p, back = fn["knet8_malloc"](60000), np.empty(15000, np.int32)
        for _ in range(30):
            a = rng.integers(-1000, 1000, size=15000).astype(np.int32)
            ok = fn["knet8_upload"](p, a.ctypes.data, a.nbytes, 2) == 0 and fn["knet8_memcpy"](back.ctypes.data, p, a.nbytes, 2, 2) == 0
            if not ok or not np.array_equal(a, back):
                wrong.append(seed)
        fn["knet8_free"](p)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    lib.check()
