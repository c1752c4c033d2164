"""Reductions of runs at any element boundary, and the variance in one launch: edges of the 16-byte loads, each route, offset operands."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def offset(knet, a, by):
    """The array on the device, starting ``by`` elements after a 256-byte boundary."""
    pad = np.zeros(a.size + by, a.dtype)
    pad[by:] = a.ravel(order="F")
    return knet.KnetArray(pad).view1d(by, a.size).reshape(a.shape)


# runs around the limit (8 vectors), with 0..3 elements over, one slab and several, one part and several; starts off the 16-byte boundary
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("dims", [(31, 5, 3), (32, 5, 3), (33, 5, 3), (35, 7, 4), (841, 9, 5), (1030, 3, 1), (4099, 2, 2), (70001, 2, 1), (15, 6, 2), (17, 6, 2), (64, 3, 2)])
@pytest.mark.parametrize("by", [0, 1])
def test_runs_of_any_length(knet, dims, by, dt):
    rng = np.random.default_rng(sum(dims))
    x = rng.standard_normal(dims).astype(dt)
    xd = offset(knet, x, by)
    want = x.astype(np.longdouble).sum(axis=(0, 2), keepdims=True)
    eps = 2.0 ** -24 if dt == np.float32 else 2.0 ** -53
    n = dims[0] * dims[2]
    bound = 4 * eps * np.sqrt(n) * np.abs(x).sum(axis=(0, 2), keepdims=True) / np.sqrt(n) + 1e-300
    assert np.all(np.abs(knet.Array(knet.sum(xd, dims=(1, 3))) - want) <= bound * 4)
    assert np.array_equal(knet.Array(knet.maximum(xd, dims=(1, 3))), x.max(axis=(0, 2), keepdims=True))
    assert np.array_equal(knet.Array(knet.minimum(xd, dims=(1, 3))), x.min(axis=(0, 2), keepdims=True))
    y = x.copy()
    y[-1, 0, -1] = np.inf                                # the last element counts, once
    assert np.array_equal(np.isinf(knet.Array(knet.sum(offset(knet, y, by), dims=(1, 3)))).ravel(), np.arange(dims[1]) == 0)
    assert np.array_equal(knet.Array(knet.countnz(xd, dims=(1, 3))), np.count_nonzero(x, axis=(0, 2), keepdims=True))
    knet.libknet8().check()


# (dims, reduced): convolution layers, columns, rows; sizes on both sides of what the kernel declines; scalars and single elements
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("dims,over", [((29, 29, 7, 3), (1, 2, 4)), ((8, 8, 5, 4), (1, 2, 4)), ((7, 9, 5, 4), (1, 2, 4)), ((3, 3, 5, 4), (1, 2, 4)), ((1023, 6), (1,)), ((1025, 6), (1,)),
                                       ((2048, 6), (1,)), ((300, 700), (2,)), ((301, 33), (2,)), ((20, 500), (2,)), ((64, 31), (2,)), ((50, 1), (1,)), ((1, 9), (2,)), ((6, 5, 4), (1,)),
                                       ((6, 5, 4), (1, 2, 3)), ((6, 5, 4), (3, 1))])
@pytest.mark.parametrize("corrected", [True, False])
def test_variance_is_the_chain(knet, dims, over, corrected, dt):
    rng = np.random.default_rng(sum(dims))
    x = (rng.standard_normal(dims) + 3).astype(dt)
    axes = tuple(d - 1 for d in over)
    xd = offset(knet, x, 1)
    m = knet.mean(xd, dims=over)
    mh = knet.Array(m)
    n = int(np.prod([dims[a] for a in axes]))
    d = x - mh
    with np.errstate(all="ignore"):
        want = (d.astype(np.float64) ** 2).sum(axis=axes, keepdims=True) / (n - int(corrected))
        got = knet.Array(knet.var(xd, dims=over, mean=m, corrected=corrected))
    eps = 2.0 ** -24 if dt == np.float32 else 2.0 ** -53
    assert got.shape == want.shape and got.dtype == dt
    np.testing.assert_allclose(got, want, rtol=8 * eps * max(4.0, np.sqrt(n)), equal_nan=True)    # one rounding a term, sums of terms of one sign
    p = knet.Param(xd)
    if np.isfinite(want).all() and n - int(corrected) > 0:
        J = knet.diff(lambda: knet.sum(knet.var(p, dims=over, mean=m, corrected=corrected)))    # recorded: through its parts
        np.testing.assert_allclose(knet.Array(knet.grad(J, p)), 2 * d / dt(n - int(corrected)), rtol=20 * eps, atol=8 * eps)
    knet.libknet8().check()


# shapes x(run, outputs, slabs) on both sides of the lines between workgroup sizes and splits: units a part 128/129, 1024/1025, 2048/2049; 160 KB an output; 224/225 and 256/257
# workgroups; more outputs than compute units; runs of whole vectors and with 1 to 3 elements over
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("dims", [(64, 5, 8), (65, 5, 8), (516, 3, 8), (512, 40, 8), (513, 40, 8), (1024, 40, 8), (1028, 40, 8), (1029, 9, 40), (1024, 9, 41), (5120, 3, 9),
                                  (260, 224, 33), (260, 225, 33), (261, 256, 33), (261, 257, 33), (400, 300, 4), (1100, 300, 9), (67, 900, 3), (3000, 60, 20)])
def test_reductions_over_slabs(knet, dims, dt):
    rng = np.random.default_rng(sum(dims))
    x = rng.standard_normal(dims).astype(dt)
    eps = 2.0 ** -24 if dt == np.float32 else 2.0 ** -53
    n = dims[0] * dims[2]
    want = x.astype(np.longdouble).sum(axis=(0, 2), keepdims=True)
    bound = 16 * eps * np.abs(x).sum(axis=(0, 2), keepdims=True)     # lanes hold partial sums of some ten terms, log2 of the lanes more on the way together
    for by in (0, 1):
        xd = offset(knet, x, by)
        got = knet.Array(knet.sum(xd, dims=(1, 3)))
        assert np.all(np.abs(got - want) <= bound)
        assert np.array_equal(knet.Array(knet.maximum(xd, dims=(1, 3))), x.max(axis=(0, 2), keepdims=True))
        m = knet.mean(xd, dims=(1, 3))
        assert np.array_equal(knet.Array(m), got * dt(1.0 / n))      # the bits of the sum and its factor
        v = knet.Array(knet.var(xd, dims=(1, 3), mean=m, corrected=False))      # terms of one sign: the bound above is relative to the sum, two more roundings a term
        np.testing.assert_allclose(v, ((x - knet.Array(m)).astype(np.longdouble) ** 2).mean(axis=(0, 2), keepdims=True), rtol=32 * eps)
    y = np.zeros(dims, dt)
    y[0, :, 0], y[-1, :, -1], y[dims[0] // 2, :, dims[2] // 2] = 1, 2, 4   # the ends of every run's walk, once
    assert np.all(knet.Array(knet.sum(offset(knet, y, 1), dims=(1, 3))) == 7)
    knet.libknet8().check()


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("dims,over", [((3, 3, 5, 4), (1, 2, 4)), ((20, 500), 2), ((64, 31), [2]), ((65, 31), (2,)), ((300, 700), 1), ((50, 1), (1,)), ((1, 9), (2,)), ((6, 5, 4), (1,)), ((6, 1, 4), (1,)),
                                       ((6, 5, 4), (1, 2, 3)), ((2000, 40), 1), ((7, 3000), 2), ((5, 4), (1, 5)), ((4000, 3), 2)])
def test_mean_is_sum_and_factor(knet, dims, over, dt):
    rng = np.random.default_rng(sum(dims))
    xd = offset(knet, rng.standard_normal(dims).astype(dt), 1)
    m, s = knet.mean(xd, dims=over), knet.sum(xd, dims=over)
    assert m.dims == s.dims and m.dtype == s.dtype
    factor, eps = dt(s.length / xd.length), 2.0 ** -24 if dt == np.float32 else 2.0 ** -53
    np.testing.assert_allclose(knet.Array(m), knet.Array(s) * factor, rtol=0, atol=16 * eps * float(np.abs(knet.Array(xd)).sum()) * float(factor))
    p = knet.Param(xd)
    J = knet.diff(lambda: knet.sum(knet.mean(p, dims=over)))
    assert np.allclose(knet.Array(knet.grad(J, p)), float(factor))
    knet.libknet8().check()


# one slab round the longest run of the stretch kernel (1024), on and off the 16-byte boundary; short runs over slabs (slab sums); rows of 256 bytes and more
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("dims,over", [((1023, 37), 1), ((1024, 37), 1), ((1024, 5000), 1), ((1025, 37), 1), ((63, 40, 50), (1, 3)), ((64, 40, 50), (1, 3)), ((32, 9000), 2), ((64, 9000), 2), ((65, 9000), 2)])
def test_mean_has_the_bits_of_the_sum_and_its_factor(knet, dims, over, dt):
    x = np.random.default_rng(sum(dims)).standard_normal(dims).astype(dt)
    for by in (0, 1):
        xd = offset(knet, x, by)
        s = knet.sum(xd, dims=over)
        assert np.array_equal(knet.Array(knet.mean(xd, dims=over)), knet.Array(s) * dt(s.length / xd.length)), by
    knet.libknet8().check()


def test_mean_without_scratch_leaves_its_output(knet):
    lib = knet.libknet8()
    x, y = knet.KnetArray(np.ones((10, 25000), np.float32)), knet.KnetArray(np.full(10, 3, np.float32))
    lib.fn["knet8_tune"](5, 1)
    try:
        knet.knet8("mean_32_21", x.length, x.ptr, 1, 10, 0.5, y.ptr)
        with pytest.raises(RuntimeError):
            lib.check()
    finally:
        lib.fn["knet8_tune"](5, 0)
    assert (knet.Array(y) == 3).all()
    knet.knet8("mean_32_21", x.length, x.ptr, 1, 10, 0.5, y.ptr)
    assert (knet.Array(y) == 12500).all()
    lib.check()


# whole vectors over several slabs, one workgroup an output, an output to (nearly) every compute unit, 128 MB and just less: places in the runs by division and in steps
@pytest.mark.parametrize("dt,dims", [(np.float32, (1024, 256, 128)), (np.float32, (1024, 256, 127)), (np.float32, (2500, 249, 55)), (np.float32, (2500, 248, 55)), (np.float64, (1026, 253, 67)), (np.float64, (514, 257, 130))])
def test_large_reductions_with_an_output_to_a_compute_unit(knet, dt, dims):
    x = np.random.default_rng(dims[2]).integers(-3, 4, dims).astype(dt)
    f = np.asfortranarray(x)
    xd = knet.KnetArray(f)
    total, squares, n = f.sum(axis=(0, 2), dtype=np.float64), (f * f).sum(axis=(0, 2), dtype=np.float64), dims[0] * dims[2]
    assert squares.max() < 2 ** 24                                                        # whole numbers below that: sums in any order are exact
    assert np.array_equal(knet.Array(knet.sum(xd, dims=(1, 3))).ravel(), total)
    assert np.array_equal(knet.Array(knet.sumabs2(xd, dims=(1, 3))).ravel(), squares)
    assert np.array_equal(knet.Array(knet.countnz(xd, dims=(1, 3))).ravel(), np.count_nonzero(f, axis=(0, 2)))
    m = knet.mean(xd, dims=(1, 3))
    assert np.array_equal(knet.Array(m).ravel(), total.astype(dt) * dt(1.0 / n))
    np.testing.assert_allclose(knet.Array(knet.var(xd, dims=(1, 3), mean=m, corrected=False)).ravel(), squares / n - (total / n) ** 2, rtol=1e-5 if dt == np.float32 else 1e-12)
    knet.libknet8().check()
