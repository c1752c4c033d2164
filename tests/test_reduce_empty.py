"""Reductions of no elements: the host's part of every ``F_S_21`` on the CPU, launches going nowhere, and their values on the GPU."""
import numpy as np
import pytest

import launch_shim

OPS = ("sum", "prod", "maximum", "minimum", "sumabs", "sumabs2", "maxabs", "minabs", "countnz")
CALLS = """
p = ctypes.c_void_p(%d)
for op in %r:
    for S in ("32", "64"):
        for sy, ny in ((1, 1), (3, 1), (1, 5), (4, 5)):
            before = shim.shim_launches()
            if op == "noalloc": lib.sum_32_21_noalloc(0, p, sy, ny, p, None)
            elif op == "mean": getattr(lib, "mean_%%s_21_stream" %% S)(0, p, sy, ny, (ctypes.c_float if S == "32" else ctypes.c_double)(1), p, None)
            else: getattr(lib, "%%s_%%s_21_stream" %% (op, S))(0, p, sy, ny, p, None)
            assert shim.shim_launches() > before, (op, S, sy, ny)
print("done")
"""


@pytest.mark.parametrize("address", [0x10000, 0x10008])
def test_no_elements_is_a_launch_like_any_other(knet, tmp_path, address):
    launch_shim.run(knet, tmp_path, CALLS % (address, ("noalloc", "mean") + OPS))


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("dims,over,shape", [((1, 0), 2, (1, 1)), ((5, 0), 2, (5, 1)), ((0,), 1, (1,))])
def test_values_of_no_elements(knet, dims, over, shape, dt):
    x = knet.KnetArray(np.zeros(dims, dt))
    for name, want in (("sum", 0), ("prod", 1), ("maximum", -np.inf), ("minimum", np.inf), ("sumabs", 0), ("sumabs2", 0), ("maxabs", 0), ("minabs", np.inf), ("countnz", 0)):
        y = getattr(knet, name)(x, dims=over)
        got = knet.Array(y)
        assert got.shape == shape and got.dtype == dt
        assert np.array_equal(got, np.full(shape, want, dt)), (name, got)
    knet.libknet8().check()
