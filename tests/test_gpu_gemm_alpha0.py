"""alpha = 0: A and B are not read, as in BLAS, whichever kernel the product would take."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# the route: hipBLASLt, the library's small-product kernels (knet8_tune key 3; the last shape is the one whose k is split over workgroups), three bf16 parts (key 9)
@pytest.mark.parametrize("knob", [(3, 0), (3, 270), (9, 2)])
@pytest.mark.parametrize("S,dt", [("32", np.float32), ("64", np.float64)])
@pytest.mark.parametrize("m,n,k", [(64, 100, 784), (300, 257, 545), (16, 24, 9000)])
def test_alpha_zero(knet, m, n, k, S, dt, knob):
    lib = knet.libknet8()
    A, B = np.full((m, k), np.nan, dt), np.full((k, n), np.inf, dt)
    C, bias = np.arange(m * n, dtype=dt).reshape(m, n), np.linspace(-1, 1, m).astype(dt)
    Ad, Bd, bd = knet.KnetArray(A), knet.KnetArray(B), knet.KnetArray(bias)
    old = lib.fn["knet8_tune"](*knob)
    try:
        for beta in (0.0, 1.0, -2.0):
            got = knet.Array(knet.gemm("N", "N", 0.0, Ad, Bd, beta, knet.KnetArray(C)))
            assert np.array_equal(got, beta * C), beta
        out = knet.KnetArray(C)
        assert lib.call("gemm_bias_act_" + S, b"N", b"N", m, n, k, 0.0, Ad.ptr, m, Bd.ptr, k, bd.ptr, 1, out.ptr, m) == 0
        assert np.array_equal(knet.Array(out), np.broadcast_to(np.maximum(bias, 0)[:, None], (m, n)))
    finally:
        lib.fn["knet8_tune"](knob[0], old)
    lib.check()


@pytest.mark.parametrize("S,dt", [("32", np.float32), ("64", np.float64)])
def test_alpha_zero_in_batches(knet, S, dt):
    lib = knet.libknet8()
    m, n, k, batch = 16, 24, 9000, 3
    A, B = knet.KnetArray(np.full((m, k, batch), np.nan, dt)), knet.KnetArray(np.full((k, n, batch), np.inf, dt))
    C = np.arange(m * n * batch, dtype=dt).reshape(m, n, batch)
    for beta in (0.0, -2.0):
        out = knet.KnetArray(C)
        assert lib.call("bmm_" + S, b"N", b"N", m, n, k, 0.0, A.ptr, m, m * k, B.ptr, k, k * n, beta, out.ptr, m, m * n, batch) == 0
        assert np.array_equal(knet.Array(out), beta * C)
    lib.check()


def test_what_stays_refused(knet):
    """An activation without a bias has no kernel on any route, alpha = 0 included."""
    lib = knet.libknet8()
    A, B, C = (knet.KnetArray(np.ones(d, np.float32)) for d in ((700, 700), (700, 700), (700, 700)))
    assert lib.call("gemm_bias_act_32", b"N", b"N", 700, 700, 700, 0.0, A.ptr, 700, B.ptr, 700, None, 1, C.ptr, 700) == -1
    with pytest.raises(RuntimeError):
        lib.check()
