"""Dynamic LDS over 64 KB is granted to every device whose stream runs such a
kernel, on the CPU: a process in which a few runtime calls are counted instead
of made (no kernel runs, no pointer is read)."""

import os
import subprocess
import sys

import pytest

from fdfdpy_amd import _lib as L

COUNTED = r"""
#include <stddef.h>
static int current, grants[8], launches, refused = -1;
int hipGetDevice(int *d) { *d = current; return 0; }
int hipSetDevice(int d) { current = d; return 0; }
int hipStreamGetDevice(void *s, int *d) { *d = (int)((size_t)s >> 12); return (size_t)s < 4096; }
int hipFuncSetAttribute(const void *f, int a, int v) { if (current == refused) return 1; ++grants[current]; return 0; }
int hipLaunchKernel() { ++launches; return 0; }
int hipGetLastError(void) { return 0; }
int hipMemsetAsync() { return 0; }
int hipMemcpyAsync() { return 0; }
int hipStreamSynchronize(void *s) { return 0; }
int seen_grants(int d) { return grants[d]; }
int seen_launches(void) { return launches; }
void refuse(int d) { refused = d; }
"""

PROGRAM = r"""
import ctypes, sys
lib_path, counted = sys.argv[1:3]
c = ctypes.CDLL(counted, ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(lib_path)
class Grid(ctypes.Structure):
    _fields_ = [(k, ctypes.c_int32) for k in ("nx", "ny", "npml_x", "npml_y", "pol", "reserved")] + \
               [(k, ctypes.c_double) for k in ("omega", "dl", "L0")]
p = ctypes.c_void_p(256)
def factor(dev, stream=0):        # nested dissection in FP64: 67.6 KB
    c.hipSetDevice(dev)
    g = Grid(64, 64, 8, 8, 0, 0, 1.2e15, 0.02, 1e-6)
    return lib.fdfd_factor(ctypes.byref(g), p, p, 0x400, p, ctypes.c_void_p(stream))
def sweep(dev, stream=0):         # FP64 blocks of 1100 cells: 72 KB, a kernel per direction
    c.hipSetDevice(dev)
    g = Grid(1100, 1100, 8, 8, 0, 0, 1.2e15, 0.02, 1e-6)
    return lib.fdfd_sweep(ctypes.byref(g), p, p, 0x200, p, p, 1, p, ctypes.c_void_p(stream))
for call, kernels in ((factor, 1), (sweep, 2)):
    before = [c.seen_grants(d) for d in range(8)]
    new = lambda: [c.seen_grants(d) - before[d] for d in range(5)]
    assert call(0) == 0 and call(0) == 0 and new() == [kernels, 0, 0, 0, 0], new()
    assert call(1) == 0 and new() == [kernels, kernels, 0, 0, 0], new()
    assert call(1, 1) == 0 and call(1, 2) == 0 and new() == [kernels, kernels, 0, 0, 0], new()   # legacy, per thread
    assert call(0, 2 << 12) == 0 and new() == [kernels, kernels, kernels, 0, 0], new()   # a stream of device 2
    c.refuse(3)
    n = c.seen_launches()
    assert call(3) == 2 and c.seen_launches() == n        # FDFD_ERR_HIP, nothing launched
    c.refuse(-1)
    assert call(3) == 0 and new() == [kernels] * 4 + [0], new()
    d = ctypes.c_int()
    c.hipSetDevice(0), call(0, 4 << 12), c.hipGetDevice(ctypes.byref(d))
    assert d.value == 0 and new() == [kernels] * 5, (d.value, new())
print("ok")
"""


def test_every_device_is_granted(tmp_path):
    if not os.path.exists(L.LIB_PATH):
        pytest.fail("the library is not built")
    src, so = tmp_path / "counted.c", tmp_path / "libcounted.so"
    src.write_text(COUNTED)
    subprocess.run(["gcc", "-w", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    r = subprocess.run([sys.executable, "-c", PROGRAM, L.LIB_PATH, str(so)], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
