"""Reductions of no elements: the host's part of every ``F_S_21`` on the CPU, launches going nowhere, and their values on the GPU."""
import subprocess
import sys

import numpy as np
import pytest

OPS = ("sum", "prod", "maximum", "minimum", "sumabs", "sumabs2", "maxabs", "minabs", "countnz")

# In the place of the HIP runtime's launch calls: launches are counted and dropped.
SHIM = """
#include <stddef.h>
typedef struct { unsigned x, y, z; } d3;
static int n;
int __hipPushCallConfiguration(d3 a, d3 b, size_t s, void* st) { return 0; }
int __hipPopCallConfiguration(d3* a, d3* b, size_t* s, void** st) { return 0; }
int hipLaunchKernel(const void* f, d3 a, d3 b, void** k, size_t s, void* st) { n++; return 0; }
int shim_launches(void) { return n; }
"""
CALLS = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
p = ctypes.c_void_p(int(sys.argv[3]))
for op in sys.argv[5:]:
    for S in ("32", "64"):
        for sy, ny in ((1, 1), (3, 1), (1, 5), (4, 5)):
            before = shim.shim_launches()
            if op == "noalloc": lib.sum_32_21_noalloc(0, p, sy, ny, p, None)
            elif op == "mean": getattr(lib, "mean_%s_21_stream" % S)(0, p, sy, ny, (ctypes.c_float if S == "32" else ctypes.c_double)(1), p, None)
            else: getattr(lib, "%s_%s_21_stream" % (op, S))(0, p, sy, ny, p, None)
            assert shim.shim_launches() > before, (op, S, sy, ny)
print("done")
"""


@pytest.mark.parametrize("address", [0x10000, 0x10008])
def test_no_elements_is_a_launch_like_any_other(knet, tmp_path, address):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)])
    r = subprocess.run([sys.executable, "-c", CALLS, str(so), knet.LIB_PATH, str(address), "-", "noalloc", "mean"] + list(OPS), capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "done" in r.stdout, (r.returncode, r.stdout, r.stderr[-2000:])


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
