"""The host's part of entry points on the CPU: a small library in the place of the HIP runtime's launches and allocations.  Launches go nowhere; their number and the
largest grid are kept.  Code runs in a process of its own, where ``shim`` and ``lib`` (libknet8, by ctypes) are there already."""
import subprocess
import sys

SOURCE = """
#include <stddef.h>
#include <stdlib.h>
typedef struct { unsigned x, y, z; } d3;
static int n;
static unsigned long long most, next = 0x7000000000ull;
int __hipPushCallConfiguration(d3 g, d3 b, size_t s, void* st) {
  const unsigned long long threads = (unsigned long long)g.x * b.x;
  if (threads > most) most = threads;
  return 0;
}
int __hipPopCallConfiguration(d3* g, d3* b, size_t* s, void** st) { return 0; }
int hipLaunchKernel(const void* f, d3 g, d3 b, void** k, size_t s, void* st) { n++; return 0; }
int hipMalloc(void** p, size_t size) { *p = (void*)next; next += (size + 4095) / 4096 * 4096; return 0; }   /* never touched on the host */
int hipHostMalloc(void** p, size_t size, unsigned flags) { *p = calloc(size, 1); return *p ? 0 : 2; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetLastError(void) { return 0; }
int hipDeviceGetAttribute(int* v, int a, int d) { *v = 256; return 0; }
int hipStreamSynchronize(void* st) { return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t size, int kind, void* st) { return 0; }
int hipblasLtCreate(void** handle) { return 1; }   /* no vendor library here: its products end with an error */
int shim_launches(void) { return n; }
unsigned long long shim_most_threads(void) { return most; }
"""
PRELUDE = """
import ctypes
shim = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
shim.shim_most_threads.restype = ctypes.c_ulonglong
lib = ctypes.CDLL(%r)
lib.knet8_last_error.restype = ctypes.c_char_p
"""


def run(knet, tmp_path, code):
    """Runs ``code``, which has to print ``done`` at its end."""
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SOURCE)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)])
    r = subprocess.run([sys.executable, "-c", PRELUDE % (str(so), knet.LIB_PATH) + code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "done" in r.stdout, (r.returncode, r.stdout, r.stderr[-2000:])
