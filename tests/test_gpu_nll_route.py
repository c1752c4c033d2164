"""``nll`` of host labels, one pass or the chain (logsoftmax, gather, sum): what the chain accepted, refused and answered holds on both sides of the rule."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def chain(knet, x, labels):
    """Loss and gradient by the separate steps."""
    p = knet.Param(knet.KnetArray(x))
    idx = knet.findindices(knet.value(p), labels)
    J = knet.diff(lambda: knet.sum(knet.getindex(knet.logsoftmax(p, dims=1), idx)))
    n = len(idx)
    return -float(knet.value(J)) / n, -knet.Array(knet.grad(J, p)) / n


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("what", ["plain", "one_class", "tall", "images", "masked", "all_masked", "nan", "inf", "skipped", "skipped_nan", "beyond"])
def test_nll_is_the_chain(knet, what, dt):
    rng = np.random.default_rng(31)
    m, n = {"one_class": (1, 9), "tall": (40000, 5)}.get(what, (37, 50))
    x = (rng.standard_normal((m, n)) * 2).astype(dt)
    labels = rng.integers(1, m + 1, size=n)
    if what == "images":
        x, labels = x.reshape(37, 5, 10), labels.reshape(5, 10)
    if what == "masked":
        x[::3, :] = -np.inf
        x[5, 4], labels[4] = -np.inf, 6                   # the labelled score itself: an infinite loss
    if what == "all_masked":
        x[:, 7] = -np.inf
    if what in ("nan", "inf"):
        x[3, 8] = np.nan if what == "nan" else np.inf
    if what.startswith("skipped"):
        labels[::4] = 0
        if what == "skipped_nan":
            x[2, 0] = np.nan
    if what == "beyond":
        labels[0] = m + 2                                 # a row of the next column: the linear index is inside the array
    want, dwant = chain(knet, x, labels)
    p = knet.Param(knet.KnetArray(x))
    with np.errstate(all="ignore"):
        J = knet.diff(lambda: knet.nll(p, labels))
        plain = knet.nll(knet.KnetArray(x), labels)
    got, dgot = knet.value(J), knet.Array(knet.grad(J, p))
    tol = 1e-5 if dt == np.float32 else 1e-13             # the softmax kernels' contract
    assert type(got) is dt and np.allclose(float(got), want, rtol=tol, equal_nan=True) and np.allclose(float(plain), want, rtol=tol, equal_nan=True)
    assert dgot.shape == x.shape
    np.testing.assert_allclose(dgot, dwant, rtol=tol * 20, atol=tol / n, equal_nan=True)
    knet.libknet8().check()


def test_what_nll_refuses(knet):
    x = knet.KnetArray(np.zeros((4, 3), np.float32))
    for bad, err in (([1, 2], ValueError), ([1.0, 2.0, 3.0], TypeError), ([1, 2, 9], IndexError), ([-4, 1, 1], IndexError)):
        with pytest.raises(err):
            knet.nll(x, bad)
    with pytest.raises(TypeError):
        knet.nll(x, knet.KnetArray(np.array([1, 2, 3], np.int32)))
    p = knet.Param(x)
    J = knet.diff(lambda: knet.nll(p, [1, 2, 3]))
    assert abs(float(knet.value(J)) - np.log(4.0)) < 1e-6


# (m, n): one team of each size and a column that streams; labels read in host memory up to 4096 of them, copied from 4097 on and for stretches of short columns, by
# the copy that waits beyond 16384; odd columns, whose label sits in a head or tail
@pytest.mark.parametrize("m,n", [(1, 3), (10, 100), (257, 4096), (257, 4097), (10, 20000), (1000, 70), (3001, 40), (7000, 33), (16001, 20), (32000, 300), (50001, 3), (70001, 2)])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_labels_in_host_memory(knet, m, n, dt):
    rng = np.random.default_rng(m + n)
    x = (rng.standard_normal((m, n)) * 2).astype(dt)
    labels = rng.integers(1, m + 1, size=n)
    labels[0], labels[-1] = 1, m
    dx = knet.KnetArray(dtype=dt, dims=(m, n))
    xd, lib = knet.KnetArray(x), knet.libknet8()
    S = "32" if dt == np.float32 else "64"
    x64 = x.astype(np.float64)
    e = np.exp(x64 - x64.max(axis=0))
    p = e / e.sum(axis=0)
    p[labels - 1, np.arange(n)] -= 1
    tol = 1e-5 if dt == np.float32 else 1e-13             # the softmax kernels' contract
    for turn in range(2):
        got = lib.call("nll_host_%s" % S, m, n, xd.ptr, labels.ctypes.data, dx.ptr)
        lse = np.log(e.sum(axis=0)) + x64.max(axis=0)
        want = (lse - x64[labels - 1, np.arange(n)]).mean()
        assert abs(got - want) <= tol * abs(want) + tol
        np.testing.assert_allclose(knet.Array(dx), p / n, rtol=tol * 20, atol=tol / n)
        labels = labels[::-1].copy()                      # other labels through the same buffer
        p = e / e.sum(axis=0)
        p[labels - 1, np.arange(n)] -= 1
    lib.check()
    bad = labels.copy()
    for v in (0, m + 1, -1, 1 << 32):
        bad[n // 2] = v
        assert np.isnan(lib.call("nll_host_%s" % S, m, n, xd.ptr, bad.ctypes.data, dx.ptr))
    lib.check()


def test_scalars_behind_a_long_queue(knet):
    """Results that are there at once, and results that take longer than the host looks for them."""
    big, lib = knet.KnetArray(dtype=np.float64, dims=(1 << 26,)), knet.libknet8()
    for queued in (0, 1, 12, 0):
        small = knet.KnetArray(np.full(1001, 1.0 + queued))
        for _ in range(queued):
            knet.knet8("fill_64", big.length, 0.5, big.ptr)
        assert knet.sum(small) == 1001 * (1.0 + queued) and knet.maximum(small) == 1.0 + queued
    lib.check()


def test_host_labels_are_not_recorded(knet):
    x = knet.KnetArray(np.zeros((4, 3), np.float32))
    old = knet.libknet8().stream
    try:
        with pytest.raises(RuntimeError):
            knet.capture(lambda: knet.nll(x, [1, 2, 3]))
    finally:
        knet.libknet8().stream = old
    knet.libknet8().check()
    assert abs(float(knet.nll(x, [1, 2, 3])) - np.log(4.0)) < 1e-6
