"""``Fback_biasgrad_S`` where rows do not start on 16-byte boundaries: the straddling lane, the last tile of one to three rows, few rows, in place."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# rows round a vector, a wave's 64 lanes and a tile (256 rows fp32, 128 fp64); columns round a trip (16), a part and a split; place: dz apart, over dy, over y;
# shift: arrays that start one element past a 16-byte boundary
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 10, 63, 65, 67, 127, 128, 129, 130, 255, 256, 257, 258, 259, 261, 1001])
@pytest.mark.parametrize("place", ["apart", "dy", "y"])
def test_activation_gradient_and_bias_gradient_of_unaligned_rows(knet, dt, m, place):
    S, size = ("32", 4) if dt == np.float32 else ("64", 8)
    u = np.finfo(dt).eps / 2
    for n, shift in ((1, 0), (7, 1), (16, 1), (17, 0), (100, 1), (129, 0), (1000, 0), (1031, 1)):
        rng = np.random.default_rng(m * 10000 + n)
        dy, y = rng.standard_normal((2, m * n)).astype(dt)
        y = np.maximum(y, 0)
        dz = np.where(y > 0, dy, dt(0))                               # reluback.(dy, y)
        guard = np.full(8, 3.0, dt)
        a, b, c = (knet.KnetArray(np.concatenate([guard, v, guard])) for v in (dy, y, np.full(m * n, 5.0, dt)))
        # shift 0: eight guard elements keep the 16-byte boundary; shift 1: everything one element later
        at = 8 * size
        if shift:
            a, b, c = (knet.KnetArray(np.concatenate([guard, guard[:1], v, guard])) for v in (dy, y, np.full(m * n, 5.0, dt)))
            at += size
        out = {"apart": c, "dy": a, "y": b}[place]
        db = knet.KnetArray(np.full(m + 2, 3.0, dt))
        knet.knet8("reluback_biasgrad_" + S, m, n, a.ptr + at, b.ptr + at, out.ptr + at, db.ptr + size)
        got, first = knet.Array(out), 8 + shift
        assert got[first:first + m * n].tobytes() == dz.tobytes(), (n, shift)
        assert (got[:first] == 3).all() and (got[first + m * n:] == 3).all(), (n, shift)
        g = knet.Array(db)
        assert g[0] == 3 and g[-1] == 3
        z = dz.reshape(n, m).astype(np.longdouble)
        # n - 1 additions in any order: |error| <= (n - 1) u / (1 - n u) * sum |dz|
        assert (np.abs(g[1:-1] - z.sum(axis=0)) <= n * u / (1 - n * u) * np.abs(z).sum(axis=0)).all(), (n, shift)
    knet.libknet8().check()


def test_few_rows_and_very_many_columns_on_both_sides_of_the_line(knet):
    for m, n in ((10, 8192), (10, 8193), (63, 8193), (64, 8193)):
        rng = np.random.default_rng(n)
        dy, y = rng.standard_normal((2, m * n)).astype(np.float32)
        dz = np.where(y > 0, dy, np.float32(0))
        a, b, c, db = knet.KnetArray(dy), knet.KnetArray(y), knet.KnetArray(dtype=np.float32, dims=(m * n,)), knet.KnetArray(dtype=np.float32, dims=(m,))
        knet.knet8("reluback_biasgrad_32", m, n, a.ptr, b.ptr, c.ptr, db.ptr)
        assert knet.Array(c).tobytes() == dz.tobytes()
        z, u = dz.reshape(n, m).astype(np.float64), 2.0 ** -24
        assert (np.abs(knet.Array(db) - z.sum(axis=0)) <= n * u / (1 - n * u) * np.abs(z).sum(axis=0)).all()
    knet.libknet8().check()


@pytest.mark.parametrize("m,n", [(64, 100), (10, 100), (300, 64), (33, 255)])
def test_short_splits_without_scratch_go_unsplit(knet, m, n):
    fn = knet.libknet8().fn
    rng = np.random.default_rng(m)
    dy, y = rng.integers(-9, 10, size=(2, m * n)).astype(np.float32)      # whole numbers: every order of the sum gives the same bits
    dz = np.where(y > 0, dy, np.float32(0))
    a, b, c = knet.KnetArray(dy), knet.KnetArray(y), knet.KnetArray(dtype=np.float32, dims=(m * n,))
    for refuse in (1, 0):
        db = knet.KnetArray(np.full(m, -777, np.float32))
        fn["knet8_tune"](5, refuse)
        try:
            knet.knet8("reluback_biasgrad_32", m, n, a.ptr, b.ptr, c.ptr, db.ptr)
            knet.libknet8().check()
        finally:
            fn["knet8_tune"](5, 0)
        assert knet.Array(c).tobytes() == dz.tobytes() and np.array_equal(knet.Array(db), dz.reshape(n, m).sum(axis=0))


def test_the_first_call_of_a_stream_may_be_captured(knet):
    """A stream's first short split, under capture: nothing is allocated there, one workgroup walks the columns, and replays between eager splits keep their results."""
    fn = knet.libknet8().fn
    m, n = 64, 100
    rng = np.random.default_rng(8)
    dy, y = rng.integers(-9, 10, size=(2, m * n)).astype(np.float32)
    dz = np.where(y > 0, dy, np.float32(0))
    a, b, c, db = knet.KnetArray(dy), knet.KnetArray(y), knet.KnetArray(dtype=np.float32, dims=(m * n,)), knet.KnetArray(dtype=np.float32, dims=(m,))
    knet.synchronize()
    stream = fn["knet8_stream_create"]()
    try:
        stats = (ctypes.c_ulonglong * 6)()
        fn["knet8_stats"](ctypes.cast(stats, ctypes.c_void_p))
        before = stats[0]
        assert fn["knet8_graph_begin"](stream) == 0
        fn["reluback_biasgrad_32_stream"](m, n, a.ptr, b.ptr, c.ptr, db.ptr, stream)
        graph = fn["knet8_graph_end"](stream)
        fn["knet8_stats"](ctypes.cast(stats, ctypes.c_void_p))
        assert graph and stats[0] == before
        for turn in range(3):
            knet.fill(db, -777)
            knet.fill(c, -777)
            knet.synchronize()
            assert fn["knet8_graph_launch"](graph, stream) == 0 and fn["knet8_synchronize"](stream) == 0
            assert np.array_equal(knet.Array(db), dz.reshape(n, m).sum(axis=0)) and knet.Array(c).tobytes() == dz.tobytes()
            knet.fill(db, -777)
            knet.synchronize()
            fn["reluback_biasgrad_32_stream"](m, n, a.ptr, b.ptr, c.ptr, db.ptr, stream)      # eager, split: the stream's scratch is made now
            assert fn["knet8_synchronize"](stream) == 0 and np.array_equal(knet.Array(db), dz.reshape(n, m).sum(axis=0))
        fn["knet8_graph_destroy"](graph)
    finally:
        fn["knet8_stream_destroy"](stream)
    knet.libknet8().check()
