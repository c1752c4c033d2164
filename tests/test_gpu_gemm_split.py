"""Large fp32 products on the bf16 matrix cores (three bf16 parts per element): edges of the tiles, remainders of k, slices of k, the epilogue,
and what does not fit the parts (infinities, NaN, sums beyond 2^80, denormals)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def device(knet, a):
    return knet.KnetArray(np.asfortranarray(a))


def product(knet, ta, tb, A, B, alpha=1.0, beta=0.0, C=None):
    m, n = (A.shape[1] if ta else A.shape[0]), (B.shape[0] if tb else B.shape[1])
    C = np.zeros((m, n), np.float32) if C is None else C
    out = device(knet, C)
    knet.gemm("T" if ta else "N", "T" if tb else "N", alpha, device(knet, A), device(knet, B), beta, out)
    return knet.Array(out)


def operands(rng, ta, tb, m, n, k):
    A, B = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    return A, B, (np.ascontiguousarray(A.T) if ta else A), (np.ascontiguousarray(B.T) if tb else B)


@pytest.fixture
def everywhere(knet):
    """The kernel takes every product that it can (knet8_tune key 9), so that its edges are reached at small sizes."""
    fn = knet.libknet8().fn
    old = fn["knet8_tune"](9, 2)
    yield
    fn["knet8_tune"](9, old)


# (m, n, k) around the 256x128 tile and its 32 steps of k: the smallest; one row or column less and more; 1 to 3 rows in the last tile (fewer than
# one lane of the loader takes); k of less than a stage, whole stages, remainders; more than one slice of k; more tiles than
# compute units
SHAPES = [(4, 4, 1), (5, 7, 3), (63, 200, 33), (255, 127, 31), (256, 128, 32), (257, 129, 64), (258, 130, 65), (259, 131, 96), (129, 257, 127), (511, 385, 100),
          (257, 131, 1000), (1024, 1024, 2048), (300, 260, 4111), (4097, 2049, 70)]


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_every_element_against_64_bits(knet, everywhere, m, n, k, ta, tb):
    rng = np.random.default_rng(m + 3 * n + 7 * k + 2 * ta + tb)
    A, B, a, b = operands(rng, ta, tb, m, n, k)
    want = A.astype(np.float64) @ B.astype(np.float64)
    got = product(knet, ta, tb, a, b)
    # k products with a rounding of 2^-24 of the running sum each (random signs: sqrt(k) of them, running sums up to sqrt(k)); 6 standard deviations
    bound = 6 * 2.0 ** -24 * k ** 0.5 * max(1.0, k ** 0.5)
    assert np.abs(got - want).max() <= bound
    assert np.linalg.norm(got - want) <= 2.0 ** -24 * max(4.0, k ** 0.5) * np.linalg.norm(want)
    knet.libknet8().check()


@pytest.mark.parametrize("m,n,k", [(515, 390, 330), (1025, 771, 4100)])
def test_scalars_bias_and_relu(knet, everywhere, m, n, k):
    rng = np.random.default_rng(9)
    lib = knet.libknet8()
    A, B, _, _ = operands(rng, False, False, m, n, k)
    C = rng.standard_normal((m, n)).astype(np.float32)
    want = A.astype(np.float64) @ B.astype(np.float64)
    got = product(knet, False, False, A, B, alpha=0.5, beta=2.0, C=C)
    assert np.linalg.norm(got - (0.5 * want + 2.0 * C)) <= 2.0 ** -24 * k ** 0.5 * np.linalg.norm(want)
    plain = product(knet, False, False, A, B)
    bias = rng.standard_normal(m).astype(np.float32)
    Ad, Bd, bd = device(knet, A), device(knet, B), device(knet, bias)
    for act in (0, 1):
        out = knet.KnetArray(np.zeros((m, n), np.float32))
        assert lib.call("gemm_bias_act_32", b"N", b"N", m, n, k, 1.0, Ad.ptr, m, Bd.ptr, k, bd.ptr, act, out.ptr, m) == 0
        chain = plain + bias[:, None]
        assert np.array_equal(knet.Array(out), np.maximum(chain, 0) if act else chain)      # the product's bits, one rounded addition
    lib.check()


@pytest.mark.parametrize("m,n,k", [(4096, 1792, 545), (1000, 2048, 4096), (255, 3000, 8005), (64, 100, 784)])
def test_the_rule_for_large_products(knet, m, n, k):
    """Products that the rule gives to this kernel have the bits of the forced route; a small one stays where it was."""
    fn = knet.libknet8().fn
    rng = np.random.default_rng(12)
    A, B, _, _ = operands(rng, False, False, m, n, k)
    got = {}
    for knob in (0, 1, 2):
        old = fn["knet8_tune"](9, knob)
        try:
            got[knob] = product(knet, False, False, A, B)
        finally:
            fn["knet8_tune"](9, old)
    assert np.array_equal(got[0], got[1] if m == 64 else got[2])
    assert np.linalg.norm(got[1] - got[2]) <= 2.0 ** -24 * k ** 0.5 * np.linalg.norm(got[1])


def test_what_the_parts_cannot_hold(knet, everywhere):
    rng = np.random.default_rng(10)
    m, n, k = 1024, 1024, 2048
    A, B, _, _ = operands(rng, False, False, m, n, k)
    A[3, 5], A[700, 9], A[300, 17] = np.inf, np.nan, 3.4e38
    B[1, 400] = -np.inf
    with np.errstate(all="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
    got = product(knet, False, False, A, B)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
    fine = np.isfinite(want) & (np.abs(want) < 3e38)
    with np.errstate(invalid="ignore"):
        off = np.abs(got - want)
    assert off[fine].max() <= 1e-5 * np.abs(want[fine]).max()
    rest = np.ones(m, bool)
    rest[[3, 700, 300]] = False
    cols = np.ones(n, bool)
    cols[400] = False
    assert off[rest][:, cols].max() <= 6 * 2.0 ** -24 * k
    # whole rows at the ends of the range: denormals and tiny numbers, numbers whose sums pass 2^80
    A, B, _, _ = operands(rng, False, False, m, n, k)
    s = np.ones(m)
    s[:64], s[64:128], s[512:576] = 1e-36, 1e-42, 1e30
    A = (A * s[:, None]).astype(np.float32)
    want = A.astype(np.float64) @ B.astype(np.float64)
    got = product(knet, False, False, A, B)
    err = np.linalg.norm(got - want, axis=1)
    least = 2.0 ** -149 * n ** 0.5        # the spacing of denormal results
    assert np.all(err <= 2.0 ** -24 * k ** 0.5 * np.linalg.norm(want, axis=1) + least)
    knet.libknet8().check()


def with_knob(knet, value, f):
    fn = knet.libknet8().fn
    old = fn["knet8_tune"](9, value)
    try:
        return f()
    finally:
        fn["knet8_tune"](9, old)


@pytest.mark.parametrize("m,n,k", [(512, 384, 512), (300, 260, 4111)])
def test_sums_with_one_term(knet, everywhere, m, n, k):
    """One element to a row of A: each result is one product, rounded once (2^-24; the parts' own sums add at most a few roundings of numbers 2^-8 as large)."""
    rng = np.random.default_rng(21)
    A = np.zeros((m, k), np.float32)
    A[np.arange(m), rng.integers(0, k, size=m)] = rng.standard_normal(m)
    B = rng.standard_normal((k, n)).astype(np.float32)
    want = A.astype(np.float64) @ B.astype(np.float64)
    assert np.all(np.abs(product(knet, False, False, A, B) - want) <= 2.0 ** -24 * (1 + 2.0 ** -6) * np.abs(want))


def test_sums_of_equal_numbers(knet, everywhere):
    """Where what is left out has one sign in every term: 1.0038986^2, whose products of the middle and the last part make up 2^-24.01 of it.  784 of them are within
    2^-25.7 of a number that fp32 has, and that is the result."""
    v = np.array([0x3f807fc0], np.int32).view(np.float32)[0]
    m, n, k = 512, 256, 784
    want = np.float32(k * np.float64(v) * np.float64(v))
    assert np.all(product(knet, False, False, np.full((m, k), v), np.full((k, n), v)) == want)


@pytest.mark.parametrize("m,n,k", [(1000, 237, 784), (1024, 768, 2048), (512, 640, 32000)])
@pytest.mark.parametrize("what", ["normal", "positive", "relu"])
def test_no_less_precise_than_fp32(knet, m, n, k, what):
    """The error of dense products against 64 bits, beside the same product on the vendor's fp32 kernels."""
    rng = np.random.default_rng(22)
    A, B, _, _ = operands(rng, False, False, m, n, k)
    if what == "positive":
        A, B = np.abs(A), np.abs(B)
    if what == "relu":
        B = np.maximum(B, 0)
    want = A.astype(np.float64) @ B.astype(np.float64)
    off = [np.linalg.norm(with_knob(knet, v, lambda: product(knet, False, False, A, B)) - want) for v in (1, 2)]
    assert off[1] <= off[0]


def test_slices_of_k_without_scratch(knet, everywhere):
    """A product that would be cut into slices of k runs in one piece when there is no memory for their sums (knet8_tune key 5): a result, and no error."""
    lib = knet.libknet8()
    rng = np.random.default_rng(23)
    m, n, k = 300, 260, 4111
    A, B, _, _ = operands(rng, False, False, m, n, k)
    C, want = rng.standard_normal((m, n)).astype(np.float32), A.astype(np.float64) @ B.astype(np.float64)
    old = lib.fn["knet8_tune"](5, 1)
    try:
        Ad, Bd, Cd = device(knet, A), device(knet, B), device(knet, C)
        assert lib.call("gemm_32", b"N", b"N", m, n, k, 0.5, Ad.ptr, m, Bd.ptr, k, 2.0, Cd.ptr, m) == 0
    finally:
        lib.fn["knet8_tune"](5, old)
    assert np.linalg.norm(knet.Array(Cd) - (0.5 * want + 2.0 * C)) <= 2.0 ** -24 * k ** 0.5 * np.linalg.norm(want)
    lib.check()


def test_scratch_of_slices_is_bounded(knet, everywhere):
    """The slices of a product (here three of 21 MB) hold at most 64 MB of their stream."""
    import ctypes
    lib = knet.libknet8()
    m, n, k = 2304, 2304, 2048
    A, B, C = (knet.KnetArray(np.ones(d, np.float32)) for d in ((m, k), (k, n), (m, n)))

    def held():
        out = (ctypes.c_ulonglong * 6)()
        lib.fn["knet8_stats"](ctypes.addressof(out))
        return out[2]
    stream = lib.fn["knet8_stream_create"]()
    before = held()
    assert lib.fn["gemm_32_stream"](b"N", b"N", m, n, k, 1.0, A.ptr, m, B.ptr, k, 0.0, C.ptr, m, stream) == 0
    lib.fn["knet8_synchronize"](stream)
    assert 3 * 4 * m * n <= held() - before <= 64 << 20
    lib.fn["knet8_stream_destroy"](stream)
    assert held() == before and np.all(knet.Array(C) == k)
    lib.check()


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("m,n,k", [(257, 131, 31), (300, 260, 4111), (129, 257, 96)])
def test_sums_formed_again(knet, everywhere, m, n, k, ta, tb):
    """Sums that are not finite, or lie beyond 2^80, beside others: around a tile's edges, with a remainder of k and in slices, with beta, bias and relu.  They are those
    of the fp32 instruction; the sums of rows and columns without one keep their bits."""
    rng = np.random.default_rng(24)
    A, B, _, _ = operands(rng, ta, tb, m, n, k)
    C, bias = rng.standard_normal((m, n)).astype(np.float32), rng.standard_normal(m).astype(np.float32)
    lib = knet.libknet8()

    def both(A, B):
        a, b = (np.ascontiguousarray(A.T) if ta else A), (np.ascontiguousarray(B.T) if tb else B)
        Ad, Bd, bd, out = device(knet, a), device(knet, b), device(knet, bias), device(knet, C)
        assert lib.call("gemm_bias_act_32", b"T" if ta else b"N", b"T" if tb else b"N", m, n, k, 1.0, Ad.ptr, a.shape[0], Bd.ptr, b.shape[0], bd.ptr, 1, out.ptr, m) == 0
        return product(knet, ta, tb, a, b, alpha=0.5, beta=2.0, C=C), knet.Array(out)
    clean = both(A, B)
    A, B = A.copy(), B.copy()
    A[0, k // 2], A[m - 1, k - 1], A[70], B[3, n - 1] = np.nan, np.inf, A[70] * 1e28, -np.inf
    got, ref = both(A, B), with_knob(knet, 1, lambda: both(A, B))
    rest = np.ix_([i for i in range(m) if i not in (0, 70, m - 1)], range(n - 1))
    for g, r, c in zip(got, ref, clean):
        assert np.array_equal(np.isnan(g), np.isnan(r)) and np.array_equal(g[np.isinf(r)], r[np.isinf(r)])
        assert np.linalg.norm(g[70, :-1].astype(np.float64) - r[70, :-1]) <= 2.0 ** -24 * max(4.0, k ** 0.5) * np.linalg.norm(r[70, :-1].astype(np.float64))
        assert np.array_equal(g[rest], c[rest])
    lib.check()


def test_all_nan(knet, everywhere):
    got = product(knet, False, False, np.full((260, 300), np.nan, np.float32), np.ones((300, 140), np.float32))
    assert np.isnan(got).all()


@pytest.mark.parametrize("m,n,pad,first", [(256, 128, 0, 0), (259, 131, 1, 1), (258, 130, 3, 2), (5, 7, 2, 3)])
def test_stores_at_any_boundary_and_single_sums(knet, everywhere, m, n, pad, first):
    """C from any element of its array on and with any column stride: four sums a store, nothing beside the columns is touched.  Single sums beyond 2^80, in every row
    and column of a 16x16 tile, are those of the fp32 instruction; their neighbours are not formed again."""
    k, ldc = 40, m + pad
    rng = np.random.default_rng(m)
    A, B = rng.uniform(0.5, 1.0, (m, k)).astype(np.float32), rng.uniform(0.5, 1.0, (k, n)).astype(np.float32)
    # scaled by powers of two, so that a sum is beyond 2^80 only where a large row meets a large column
    A[np.arange(0, m, 17) % m] *= np.float32(2.0 ** 45)
    B[:, np.arange(0, n, 9) % n] *= np.float32(2.0 ** 45)
    want = A.astype(np.float64) @ B.astype(np.float64)
    C = np.full(first + ldc * n + 4, 7.0, np.float32)
    Ad, Bd, Cd = device(knet, A), device(knet, B), device(knet, C)
    lib = knet.libknet8()
    for beta in (0.0, 1.0):
        assert lib.call("gemm_32", b"N", b"N", m, n, k, 1.0, Ad.ptr, m, Bd.ptr, k, beta, Cd.ptr + 4 * first, ldc) == 0
    out = knet.Array(Cd)
    got = out[first:first + ldc * n].reshape(ldc, n, order="F")
    assert np.all(out[:first] == 7) and np.all(out[first + ldc * n:] == 7) and np.all(got[m:] == 7)
    # positive terms: k + 1 roundings of at most 2^-24 of the sum each in the product, one in the addition
    assert np.abs(got[:m] - 2 * want).max(initial=0, where=want < 2.0 ** 80) <= 2.0 ** -24 * (k + 2) * 2 * want[want < 2.0 ** 80].max()
    assert (np.abs(got[:m] / (2 * want) - 1)).max() <= 2.0 ** -24 * (k + 2)
    lib.check()
