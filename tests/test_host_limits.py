"""Calls at the limits of grids and of host memory: the host's part, on the CPU."""
import pytest

import launch_shim


# 64-bit products of which the 32x32 kernel has more tiles than fit a grid (2^32 threads), and just as many as fit: 4 waves to a tile from k = 500 on, 2 from 250 on
@pytest.mark.parametrize("m,n,k,own", [(131072, 131072, 512, False), (131072, 131040, 512, True), (262144, 131072, 250, False), (262144, 131072, 100, True), (4096, 4096, 512, True)])
def test_a_product_of_more_tiles_than_a_grid_holds_stays_with_the_vendor(knet, tmp_path, m, n, k, own):
    launch_shim.run(knet, tmp_path, """
m, n, k, own = %r
lib.knet8_tune(11, 3)                       # the 32x32 kernel by its rule
lib.knet8_tune(7, 1)
p, d, c = ctypes.c_void_p(0x7f0000000000), ctypes.c_double, ctypes.c_char
lib.gemm_64_stream(c(b"N"), c(b"N"), m, n, k, d(1), p, m, p, k, d(0), p, m, None)
assert lib.knet8_product_route() == (4 if own else 1), lib.knet8_product_route()
assert shim.shim_most_threads() < 2 ** 32, shim.shim_most_threads()
assert (shim.shim_launches() == 1) == own
print("done")
""" % ((m, n, k, own),))


def test_labels_that_no_host_memory_is_left_for_are_an_error(knet, tmp_path):
    launch_shim.run(knet, tmp_path, """
import math, resource, numpy as np
n = 1 << 26
labels = np.ones(n, np.int64)
p = ctypes.c_void_p(0x7f0000000000)
lib.nll_host_32_stream.restype = ctypes.c_float
lib.nll_host_32_stream(1, 16, p, labels.ctypes.data_as(ctypes.c_void_p), p, None)     # (what a first call sets up)
before = shim.shim_launches()
error = lib.knet8_last_error()
assert error is None, error
size = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (size + (64 << 20), resource.RLIM_INFINITY))     # the labels as 32 bits take 256 MB
loss = lib.nll_host_32_stream(1, n, p, labels.ctypes.data_as(ctypes.c_void_p), p, None)
assert math.isnan(loss) and shim.shim_launches() == before and b"host memory" in lib.knet8_last_error()
print("done")
""")
