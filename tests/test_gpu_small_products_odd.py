"""Small products and the layer's backward launch where columns along k start off 16-byte boundaries: the last step of a slice, arrays that start one element later."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def shifted(knet, a, off):
    """The array on the device, `off` elements past a 16-byte boundary (with NaN around it: an element read from outside shows)."""
    pad = np.full(8, np.nan, a.dtype)
    keep = knet.KnetArray(np.concatenate([pad, pad[:off], a.ravel(order="F"), pad]))
    return keep, keep.ptr + (8 + off) * a.dtype.itemsize


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("form", ["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("k", [1, 3, 4, 5, 15, 17, 31, 33, 255, 517])
def test_products_of_columns_at_any_element(knet, dt, form, k):
    S, u = ("32", 2.0 ** -24) if dt == np.float32 else ("64", 2.0 ** -53)
    lib = knet.libknet8()
    old = lib.fn["knet8_tune"](3, 270)     # the small-product kernels, whatever the rule
    try:
        for m, n, off in ((1, 1, 1), (15, 17, 0), (33, 16, 1), (100, 65, 3)):
            rng = np.random.default_rng(k + m)
            A, B = rng.standard_normal((m, k)).astype(dt), rng.standard_normal((k, n)).astype(dt)
            a, b = A.T if form[0] == "T" else A, B.T if form[1] == "T" else B
            ka, pa = shifted(knet, a, off)
            kb, pb = shifted(knet, b, off)
            c = knet.KnetArray(dtype=dt, dims=(m, n))
            assert lib.call("gemm_" + S, form[0].encode(), form[1].encode(), m, n, k, 1.0, pa, a.shape[0], pb, b.shape[0], 0.0, c.ptr, m) == 0
            A, B = A.astype(np.longdouble), B.astype(np.longdouble)
            # k products and k - 1 additions in any order: |error| <= k u / (1 - k u) * |A| |B|
            assert (np.abs(knet.Array(c) - A @ B) <= k * u / (1 - k * u) * (np.abs(A) @ np.abs(B))).all(), (m, n)
    finally:
        lib.fn["knet8_tune"](3, old)
    lib.check()


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("m,n,k", [(3, 5, 7), (17, 33, 15), (63, 100, 65), (101, 31, 130), (257, 16, 33)])
def test_layer_gradients_of_columns_at_any_element(knet, dt, m, n, k):
    S, u = ("32", 2.0 ** -24) if dt == np.float32 else ("64", 2.0 ** -53)
    lib = knet.libknet8()
    rng = np.random.default_rng(m)
    W, x, y, dy = (rng.standard_normal(d).astype(dt) for d in ((m, k), (k, n), (m, n), (m, n)))
    for off in (0, 1, 2):
        arrays = [shifted(knet, a, off) for a in (W, x, y, dy)]
        dW, db, dx = (knet.KnetArray(dtype=dt, dims=d) for d in ((m, k), (m,), (k, n)))
        assert lib.call("dense_back_" + S, 1, m, n, k, *[p for _, p in arrays], dW.ptr, db.ptr, dx.ptr) == 0
        dz, Wl, xl = np.where(y > 0, dy, 0).astype(np.longdouble), W.astype(np.longdouble), x.astype(np.longdouble)
        for got, want, size, terms in ((dW, dz @ xl.T, np.abs(dz) @ np.abs(xl).T, n), (dx, Wl.T @ dz, np.abs(Wl).T @ np.abs(dz), m),
                                       (db, dz.sum(axis=1), np.abs(dz).sum(axis=1), n)):
            assert (np.abs(knet.Array(got) - want) <= terms * u / (1 - terms * u) * size).all(), off
    lib.check()


def test_layers_beyond_the_lines_are_left_to_separate_launches(knet):
    call, ptr = knet.libknet8().call, knet.KnetArray(dtype=np.float32, dims=(4,)).ptr
    # declined on the host, nothing is read: much work over a long inner dimension, very many columns, very many tiles
    for m, n, k, dx in ((33, 1538, 819, ptr), (3293, 198, 166, ptr), (64, 1501, 100, None), (1539, 19, 2714, None)):
        assert call("dense_back_32", 1, m, n, k, ptr, ptr, ptr, ptr, ptr, ptr, dx) == 1


@pytest.mark.parametrize("m,n,k,wants", [(33, 1538, 819, True), (64, 1501, 100, False), (1539, 19, 2714, False)])
def test_a_limit_of_the_callers_own_is_the_only_one(knet, m, n, k, wants):
    """knet8_tune key 4: 0 leaves layers that are quicker so to separate launches, a value takes every layer up to it."""
    lib, u = knet.libknet8(), 2.0 ** -24
    rng = np.random.default_rng(n)
    W, x, y, dy = (rng.standard_normal(d).astype(np.float32) for d in ((m, k), (k, n), (m, n), (m, n)))
    arrays = [knet.KnetArray(a) for a in (W, x, y, dy)]
    dW, db, dx = (knet.KnetArray(np.full(d, 7, np.float32)) for d in ((m, k), (m,), (k, n)))
    call = lambda: lib.call("dense_back_32", 1, m, n, k, *[a.ptr for a in arrays], dW.ptr, db.ptr, dx.ptr if wants else None)  # noqa: E731
    assert lib.fn["knet8_tune"](4, -1) == 0 and call() == 1 and (knet.Array(dW) == 7).all()
    old = lib.fn["knet8_tune"](4, 270)
    try:
        assert call() == 0
    finally:
        lib.fn["knet8_tune"](4, old)
    assert call() == 1 and lib.call("dense_back_32", 0, m, n, k, *[a.ptr for a in arrays], None, None, None) == 0   # nothing wanted: nothing to decline
    dz = np.where(y > 0, dy, 0).astype(np.float64)
    pairs = [(dW, dz @ x.T.astype(np.float64), np.abs(dz) @ np.abs(x).T, n), (db, dz.sum(axis=1), np.abs(dz).sum(axis=1), n)]
    if wants:
        pairs.append((dx, W.T.astype(np.float64) @ dz, np.abs(W).T @ np.abs(dz), m))
    for got, want, size, terms in pairs:        # terms products and additions in any order, as above
        assert (np.abs(knet.Array(got) - want) <= terms * u / (1 - terms * u) * size).all()
    lib.check()
