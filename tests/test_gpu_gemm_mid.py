"""Products on the 32x32 kernel (knet8_tune key 11): edges of its tiles and of a lane's pair of rows, remainders of k, each number of waves, operands at any element boundary,
the output stage, and which products the rule gives to it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def knob(knet):
    fn = knet.libknet8().fn
    old = fn["knet8_tune"](11, -1)
    yield lambda v: fn["knet8_tune"](11, v)
    fn["knet8_tune"](11, old)


def run(knet, ta, tb, A, B, alpha=1.0, beta=0.0, C=None, bias=None, act=0, pad=(0, 0, 0), by=0):
    """op(A)*op(B) with leading dimensions ``pad`` larger than the rows, every array ``by`` elements off its boundary; what lies between the columns is NaN."""
    dt, lib = A.dtype, knet.libknet8()
    S = "32" if dt == np.float32 else "64"
    a, b = (A.T if ta else A), (B.T if tb else B)
    m, n, k = A.shape[0], B.shape[1], A.shape[1]

    def place(x, extra):
        full = np.full((x.shape[0] + extra, x.shape[1]), np.nan, dt)
        full[:x.shape[0]] = x
        return knet.KnetArray(np.concatenate([np.full(by, np.nan, dt), full.ravel(order="F"), np.full(1, np.nan, dt)])), x.shape[0] + extra
    (ad, lda), (bd, ldb), (cd, ldc) = place(a, pad[0]), place(b, pad[1]), place(np.zeros((m, n), dt) if C is None else C, pad[2])
    off = by * A.itemsize
    if bias is None:
        assert lib.call("gemm_%s" % S, b"T" if ta else b"N", b"T" if tb else b"N", m, n, k, alpha, ad.ptr + off, lda, bd.ptr + off, ldb, beta, cd.ptr + off, ldc) == 0
    else:
        bias_d = knet.KnetArray(bias)
        assert lib.call("gemm_bias_act_%s" % S, b"T" if ta else b"N", b"T" if tb else b"N", m, n, k, alpha, ad.ptr + off, lda, bd.ptr + off, ldb, bias_d.ptr, act, cd.ptr + off, ldc) == 0
    assert lib.fn["knet8_product_route"]() == 4
    flat = knet.Array(cd)
    out = flat[by:by + ldc * n].reshape(ldc, n, order="F")
    assert np.isnan(flat[:by]).all() and np.isnan(flat[-1]) and np.isnan(out[m:]).all()      # nothing beside the columns is touched
    return out[:m]


SHAPES = [(2, 2, 1), (3, 5, 15), (31, 33, 16), (32, 32, 17), (33, 31, 32), (34, 65, 47), (63, 64, 100), (97, 35, 255), (129, 200, 31), (40, 70, 1030), (1000, 237, 100), (700, 900, 64), (321, 1700, 40), (1601, 1030, 20)]


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_every_element_against_more_bits(knet, knob, m, n, k, ta, tb, dt):
    knob(2)
    rng = np.random.default_rng(m + 3 * n + 7 * k + 2 * ta + tb)
    A, B = rng.standard_normal((m, k)).astype(dt), rng.standard_normal((k, n)).astype(dt)
    wide = np.float64 if dt == np.float32 else np.longdouble
    want = A.astype(wide) @ B.astype(wide) if m * n * k < 2e7 or dt == np.float32 else A @ B
    size = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)
    eps = 2.0 ** -24 if dt == np.float32 else 2.0 ** -53
    for pad, by in (((0, 0, 0), 0), ((3, 1, 2), 1)):
        got = run(knet, ta, tb, A, B, pad=pad, by=by)
        # a rounding of the running sum for each of its terms, in slices of k that are added up: k + 16 of them at most, and as many in a reference of the same type
        assert (np.abs(got - want) <= 2 * (k + 16) * eps * size).all()
        assert np.linalg.norm((got - want).astype(np.float64)) <= 2 * eps * max(2.0, k ** 0.5) * np.linalg.norm(want.astype(np.float64))
    knet.libknet8().check()


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_scalars_bias_and_relu(knet, knob, dt):
    knob(2)
    rng = np.random.default_rng(5)
    m, n, k = 67, 101, 203
    A, B, C, bias = (rng.standard_normal(s).astype(dt) for s in ((m, k), (k, n), (m, n), (m,)))
    plain = run(knet, False, False, A, B, pad=(1, 0, 3))
    assert np.array_equal(run(knet, False, False, A, B, alpha=0.5, beta=2.0, C=C, pad=(0, 1, 1)), dt(0.5) * plain + dt(2) * C)
    for act in (0, 1):
        got = run(knet, False, False, A, B, bias=bias, act=act)
        assert np.array_equal(got, np.maximum(plain + bias[:, None], 0) if act else plain + bias[:, None])   # the product's bits, one rounded addition
    A[3, 7], B[5, 9], A[m - 1, k - 1] = np.nan, np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        got, want = run(knet, True, True, A, B), A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    knet.libknet8().check()


VENDOR, SMALL, SPLIT, MID = 1, 2, 3, 4
F32 = [(1000, 237, 1000, "NN", MID), (1000, 237, 1500, "NN", VENDOR), (1000, 128, 1001, "NN", MID), (250, 250, 1501, "NN", VENDOR), (512, 512, 512, "NN", MID), (100, 237, 1000, "NN", SMALL), (512, 512, 32, "NN", SMALL),
       (256, 256, 517, "TN", SMALL), (512, 320, 185, "TN", MID), (512, 320, 183, "TN", SMALL), (512, 320, 188, "TN", SMALL), (31, 4000, 500, "TN", SMALL), (1000, 1000, 252, "NT", MID), (1000, 1000, 253, "NT", VENDOR), (1000, 2048, 4096, "NN", SPLIT),
       # short k over many tiles: the line on tiles and k, m off the 128s, n off the 16s, k beyond 64
       (256, 24576, 8, "NN", VENDOR), (256, 24576, 4, "TN", MID), (264, 24576, 8, "NN", MID), (256, 24584, 8, "NT", MID), (512, 3712, 64, "NN", VENDOR), (512, 3712, 65, "NN", MID)]
F64 = [(512, 512, 512, "NN", MID), (1100, 1200, 600, "TN", MID), (100, 64, 784, "NN", SMALL), (360, 340, 149, "NN", SMALL), (360, 380, 150, "NN", MID), (2000, 2000, 90, "NN", VENDOR), (2000, 2000, 100, "NN", MID),
       (60, 60, 8193, "NN", VENDOR), (900, 1, 900, "NN", SMALL)]


@pytest.mark.parametrize("m,n,k,form,route,dt", [c + (np.float32,) for c in F32] + [c + (np.float64,) for c in F64])
def test_each_product_takes_its_route(knet, knob, m, n, k, form, route, dt):
    """By the rule whatever hipBLASLt allows; small products by theirs where that is in force (their own kernels or the vendor's otherwise)."""
    lib = knet.libknet8()
    rng = np.random.default_rng(m + n + k)
    ta, tb = form[0] == "T", form[1] == "T"
    A, B = rng.standard_normal((m, k)).astype(dt), rng.standard_normal((k, n)).astype(dt)
    a, b = knet.KnetArray(np.asfortranarray(A.T if ta else A)), knet.KnetArray(np.asfortranarray(B.T if tb else B))
    want = A.astype(np.float64) @ B.astype(np.float64)
    eps = 2.0 ** -24 if dt == np.float32 else 2.0 ** -52
    for value, expect in ((3, (route,) if route != SMALL else (SMALL, VENDOR)), (1, (VENDOR, SMALL, SPLIT))):
        knob(value)
        got = knet.Array(knet.gemm(form[0], form[1], 1, a, b, 0, knet.KnetArray(np.zeros((m, n), dt))))
        assert lib.fn["knet8_product_route"]() in expect, value
        # one rounding a step of a running sum that grows like sqrt(k); the 64-bit reference has as many
        assert np.linalg.norm(got - want) <= 2 * eps * max(2.0, k ** 0.5) * np.linalg.norm(want)
    lib.check()
