"""Small products by default: on both sides of the rule's limits (padding, length of k, type) they match 64 bits, whichever kernel they took."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# the smallest; 16x16 tiles with remainders; at 2.7e8 flop with and without padding; k at 2048 and 8192; fp64 at k = 400 and 1.6e8 flop
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (17, 33, 5), (64, 100, 784), (100, 237, 1000), (512, 512, 514), (513, 512, 512), (16, 40, 2048), (16, 40, 2049), (8, 8, 8192),
                                   (8, 8, 8193), (576, 576, 399), (576, 576, 400)])
def test_small_products_match_64_bits(knet, m, n, k, dt):
    rng = np.random.default_rng(m + n + k)
    A, B = rng.standard_normal((m, k)).astype(dt), rng.standard_normal((k, n)).astype(dt)
    want = A.astype(np.longdouble) @ B.astype(np.longdouble) if m * n * k < 1e6 else A.astype(np.float64) @ B.astype(np.float64)
    for ta in (False, True):
        for tb in (False, True):
            a, b = (np.asfortranarray(A.T) if ta else A), (np.asfortranarray(B.T) if tb else B)
            got = knet.Array(knet.gemm("T" if ta else "N", "T" if tb else "N", 1, knet.KnetArray(a), knet.KnetArray(b), 0, knet.KnetArray(np.zeros((m, n), dt))))
            # one rounding a step of a running sum that grows like sqrt(k); the 64-bit reference has as many
            eps = 2.0 ** -24 if dt == np.float32 else 2.0 ** -52
            assert np.linalg.norm(got - want) <= 2 * eps * max(2.0, k ** 0.5) * np.linalg.norm(want), (ta, tb)
    knet.libknet8().check()


VENDOR, SMALL, SPLIT = 1, 2, 3


@pytest.fixture
def knobs(knet):
    """Sets knet8_tune keys and restores them."""
    fn = knet.libknet8().fn
    old = {}

    def put(key, value):
        old.setdefault(key, fn["knet8_tune"](key, value))
        fn["knet8_tune"](key, value)
    yield put
    for key, value in old.items():
        fn["knet8_tune"](key, value)


def test_the_other_routes(knet, knobs):
    """A limit of the caller's (key 3) comes before the rule, the forced bf16 kernel (key 9) before both of its limits; large products by their own rule."""
    lib = knet.libknet8()

    def route(m, n, k, dt=np.float32):
        A, B, C = (knet.KnetArray(np.ones(d, dt)) for d in ((m, k), (k, n), (m, n)))
        knet.gemm("N", "N", 1, A, B, 0, C)
        assert np.all(knet.Array(C) == k)
        return lib.fn["knet8_product_route"]()
    knobs(10, 1)
    assert route(10, 64, 100) == VENDOR                        # however small
    assert route(1000, 2048, 4096) == SPLIT
    knobs(3, 270)
    assert route(700, 300, 600) == SMALL and route(1000, 2048, 4096) == SPLIT
    knobs(3, 0)
    knobs(10, 2)
    knobs(9, 2)
    assert route(64, 100, 784) == SPLIT and route(64, 100, 784, np.float64) == SMALL
    knobs(9, 1)
    assert route(1000, 2048, 4096) == VENDOR
    lib.check()
