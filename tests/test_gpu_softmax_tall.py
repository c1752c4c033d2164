"""Softmax down a few columns that are too long for the registers: several workgroups to a column."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(65537, 1), (81921, 3), (100000, 100), (131073, 256), (70000, 257)])
def test_tall_columns_shared_by_workgroups(knet, oracle, m, n):
    """Columns beyond the registers with few of them (up to one a compute unit, the last shape is one more): shares with a remainder, on and off 16-byte rows."""
    rng = np.random.default_rng(m)
    x, dy = rng.standard_normal((m, n)).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    x[m // 2:, 0] = -np.inf                                  # whole shares masked
    if n > 2:
        x[7, 1], x[m - 1, 2] = np.nan, np.inf
    x64 = x[:, 3:].astype(np.float64) if n > 3 else x[:, :1].astype(np.float64)
    xd = knet.KnetArray(np.asfortranarray(x))
    y = knet.Array(knet.logsoftmax(xd, dims=1))
    if n > 2:
        assert np.isnan(y[:, 1]).all() and np.isnan(y[:, 2]).all()
    sel = slice(3, None) if n > 3 else slice(0, 1)
    mx = x64.max(axis=0)
    want = (x64 - mx) - np.log(np.exp(x64 - mx).sum(axis=0))
    fin = np.isfinite(want)
    assert np.array_equal(np.isneginf(y[:, sel]), np.isneginf(want)) and np.abs(y[:, sel][fin] - want[fin]).max() <= 1e-5 * np.abs(want[fin]).max()
    # sum of m values of N(0,1): a rounding of 2^-24 of partial sums of at most a few sqrt(m) for each of the about m/4096 additions a lane makes, times exp(y)
    got = knet.Array(knet.logsoftmaxback(knet.KnetArray(np.asfortranarray(y)), knet.KnetArray(np.asfortranarray(dy)), dims=1))
    d = dy[:, sel].astype(np.float64)
    wantb = d - np.exp(want) * d.sum(axis=0)
    assert np.abs(got[:, sel] - wantb).max() <= 1e-5 * np.abs(wantb).max()
    knet.libknet8().check()


# four shares: loads of one element, an array beyond the caches; a smaller one and shorter columns, which keep a workgroup to a column
@pytest.mark.parametrize("m,n", [(100001, 104), (170000, 104), (100000, 104), (65537, 104)])
def test_four_shares(knet, oracle, m, n):
    test_tall_columns_shared_by_workgroups(knet, oracle, m, n)


def test_tall_columns_without_scratch(knet, oracle):
    """No memory for the shares' sums (knet8_tune key 5): a workgroup to a column gives the result, and there is no error to report."""
    fn = knet.libknet8().fn
    old = fn["knet8_tune"](5, 1)
    try:
        test_tall_columns_shared_by_workgroups(knet, oracle, 81921, 3)
    finally:
        fn["knet8_tune"](5, old)
