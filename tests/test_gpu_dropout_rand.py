"""``dropout_rand_S`` / ``dropout_rand_state_S``: the mask is drawn inside the launch.  They must give the bits of the two launches they stand for
(``rand_S`` or ``rand_state_S`` into a buffer, then ``dropout_S`` in place) and leave the stream at the same place (src/ops20_gpu/dropout.jl:11-16).
Equality is exact: the same draws and the same functor, so there is no tolerance to choose."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bits_equal(a, b):
    return a.tobytes() == b.tobytes()


# sizes round a vector, a workgroup of vectors (1024 fp32, 512 fp64) and a grid of many; offsets that break the 16-byte alignment of x, of y, of both
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 511, 512, 1023, 1024, 1025, 262145])
@pytest.mark.parametrize("xo,yo", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_bits_of_rand_then_dropout_and_the_stream_goes_on_from_the_same_place(knet, dt, n, xo, yo):
    S = "32" if dt == np.float32 else "64"
    c = ctypes.c_float if dt == np.float32 else ctypes.c_double
    x = np.random.default_rng(n).standard_normal(n + 1).astype(dt)
    x[::5] = [np.nan, np.inf, -np.inf, -0.0, 0.0][n % 5]
    xd, size = knet.KnetArray(x), x.dtype.itemsize
    for p in (0.2, 0.5):
        knet.seed_(99)
        u = knet.rand_(knet.KnetArray(dtype=dt, dims=(n,)))
        xv = knet.KnetArray(x[xo:xo + n])
        want = knet.Array(knet.dropout_(p, xv, u))
        after = knet.Array(knet.rand_(knet.KnetArray(dtype=dt, dims=(5,))))

        def check(call):
            y = knet.fill(knet.KnetArray(dtype=dt, dims=(n + 2,)), 7)
            call(xd.ptr + xo * size, y.ptr + yo * size)
            got = knet.Array(y)
            assert bits_equal(got[yo:yo + n], want)
            assert (got[:yo] == 7).all() and (got[yo + n:] == 7).all()      # nothing outside its range

        knet.seed_(99)
        check(lambda xp, yp: knet.knet8("dropout_rand_" + S, n, c(p), xp, yp))
        assert bits_equal(knet.Array(knet.rand_(knet.KnetArray(dtype=dt, dims=(5,)))), after)
        state = knet.RngState(99)
        check(lambda xp, yp: knet.knet8("dropout_rand_state_" + S, n, c(p), state.ptr, xp, yp))
        per = 16 // size
        assert state.get() == (99, (n + per - 1) // per)
    knet.libknet8().check()


def test_a_null_state_is_refused_and_types_without_a_generator_too(knet):
    x = knet.KnetArray(np.ones(8, np.float32))
    y = x.similar()
    with pytest.raises(RuntimeError, match="null state"):
        knet.knet8("dropout_rand_state_32", 8, 0.5, None, x.ptr, y.ptr)
        knet.libknet8().check()
    with pytest.raises(TypeError):
        knet.dropout(knet.KnetArray(np.ones(8, np.int32)), 0.5, drop=True)
