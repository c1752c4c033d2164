"""Several host threads on one stream: launches that leave sums in the stream's scratch for a launch behind them are not mixed with another thread's."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_two_launch_sequences_from_threads_on_one_stream(knet):
    """Sliced products, shared softmax columns, softmax along a strided dimension, reductions by slab sums and split reductions: every thread has its own
    operands, and every call the bits that it has alone (each sums in a fixed order)."""
    lib = knet.libknet8()
    fn = lib.fn
    rng = np.random.default_rng(3)
    stream = fn["knet8_stream_create"]()
    f32 = np.float32

    def array(*dims):
        return knet.KnetArray(np.asfortranarray(rng.standard_normal(dims).astype(f32)))

    def jobs():
        m, n, k = 300, 260, 4111                                 # more than one slice of k (knet8_tune key 9)
        A, B, C = array(m, k), array(k, n), array(m, n)
        yield C, (A, B), lambda: fn["gemm_32_stream"](b"N", b"N", m, n, k, 1.0, A.ptr, m, B.ptr, k, 0.0, C.ptr, m, stream)
        X, Y = array(100000, 3), array(100000, 3)                # several workgroups to a column
        yield Y, (X,), lambda: fn["logsoftmax_32_stream"](100000, 3, X.ptr, Y.ptr, stream)
        S, T = array(64, 3000, 4), array(64, 3000, 4)            # maxima and sums per panel, then the panels
        yield T, (S,), lambda: fn["logsoftmax_strided_32_stream"](64, 3000, 4, S.ptr, T.ptr, stream)
        Z, z = array(4, 1000, 400), array(1000)                  # slabs added onto each other first
        yield z, (Z,), lambda: fn["sum_32_21_stream"](Z.length, Z.ptr, 4, 1000, z.ptr, stream)
        W, w = array(512, 8192), array(512)                      # parts met by ticket, in one launch
        yield w, (W,), lambda: fn["sum_32_21_stream"](W.length, W.ptr, 1, 512, w.ptr, stream)

    old = fn["knet8_tune"](9, 2)
    try:
        work = []
        for _ in range(4):
            mine = []
            for out, keep, call in jobs():
                knet.synchronize()
                call()
                fn["knet8_synchronize"](stream)
                mine.append((out, keep, call, knet.Array(out)))
            work.append(mine)
        wrong = []

        def run(mine, turn):
            for i in range(25):
                for j in range(len(mine)):
                    mine[(j + turn) % len(mine)][2]()
                if i % 5 == 4:
                    fn["knet8_synchronize"](stream)
                    for q, (out, _, _, want) in enumerate(mine):
                        got = np.empty(want.shape, want.dtype, order="F")
                        fn["knet8_memcpy"](got.ctypes.data, out.ptr, got.nbytes, 2, stream)
                        if not np.array_equal(got, want):
                            wrong.append((turn, i, q))
        threads = [threading.Thread(target=run, args=(mine, t)) for t, mine in enumerate(work)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong
        lib.check()
    finally:
        fn["knet8_tune"](9, old)
        fn["knet8_stream_destroy"](stream)
