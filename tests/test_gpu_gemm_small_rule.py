"""Small products by default: on both sides of the rule's limits (padding, length of k, type) they match 64 bits, whichever kernel they took; and each takes the kernel
that the rule names."""
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


# (m, n, k, form, the route where the rule decides): each of the rule's limits from both sides
F32 = [(64, 100, 784, "NN", SMALL), (512, 512, 512, "NN", SMALL), (513, 512, 512, "NN", VENDOR), (1024, 1024, 64, "NN", SMALL),
       (1408, 1456, 32, "NN", SMALL), (1456, 1456, 32, "NN", VENDOR), (8192, 8192, 1, "NN", VENDOR), (64, 4096, 200, "NN", SMALL), (1040, 1040, 128, "NN", VENDOR),
       (32, 64, 2048, "NN", SMALL), (32, 64, 2052, "NN", VENDOR), (64, 2048, 804, "NN", VENDOR), (64, 2048, 800, "NN", SMALL), (64, 2048, 576, "NT", VENDOR), (64, 2048, 568, "NT", SMALL),
       (112, 2048, 528, "NN", VENDOR), (112, 2048, 520, "NN", SMALL), (900, 900, 72, "TN", SMALL), (900, 900, 74, "TN", VENDOR), (900, 900, 74, "NT", SMALL)]
F64 = [(64, 100, 784, "NN", SMALL), (512, 512, 112, "NN", SMALL), (512, 512, 116, "NN", VENDOR), (432, 440, 300, "NN", SMALL), (480, 480, 300, "NN", VENDOR), (480, 480, 256, "NN", SMALL),
       (512, 512, 256, "NN", VENDOR), (1024, 1024, 16, "TN", SMALL), (1040, 1024, 4, "TN", VENDOR), (16, 24, 8192, "NN", SMALL), (16, 24, 8193, "NN", VENDOR)]


@pytest.mark.parametrize("m,n,k,form,route,dt", [c + (np.float32,) for c in F32] + [c + (np.float64,) for c in F64])
def test_each_product_takes_its_route(knet, knobs, m, n, k, form, route, dt):
    rng = np.random.default_rng(m + n + k)
    lib = knet.libknet8()
    ta, tb = form[0] == "T", form[1] == "T"
    A, B = rng.standard_normal((m, k)).astype(dt), rng.standard_normal((k, n)).astype(dt)
    a, b = knet.KnetArray(np.asfortranarray(A.T if ta else A)), knet.KnetArray(np.asfortranarray(B.T if tb else B))
    eps = 2.0 ** -24 if dt == np.float32 else 2.0 ** -52
    want = A.astype(np.float64) @ B.astype(np.float64)
    for value, expect in ((2, route), (1, VENDOR)):
        knobs(10, value)
        got = knet.Array(knet.gemm(form[0], form[1], 1, a, b, 0, knet.KnetArray(np.zeros((m, n), dt))))
        assert lib.fn["knet8_product_route"]() == expect, value
        # one rounding a step of a running sum that grows like sqrt(k); the 64-bit reference has as many
        assert np.linalg.norm(got - want) <= 2 * eps * max(2.0, k ** 0.5) * np.linalg.norm(want)
    lib.check()


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
