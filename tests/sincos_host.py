"""Host build of the device sincos() for system sources
(sodecl_amd/csrc/device/sincos.hip, compiled by g++ as C++ with contraction
off: the same IEEE double operations as on the GPU)."""
import ctypes
import functools
import os
import subprocess
import tempfile

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEVICE = os.path.join(ROOT, "sodecl_amd", "csrc", "device")

_HARNESS = r'''
#include <math.h>
#define SODECL_MATH_FN static inline
#include "%s/sin.hip"
#include "%s/sincos.hip"
extern "C" void sincos_host(const double* x, double* s, double* c, unsigned char* covered, long n)
{
    for (long i = 0; i < n; ++i) covered[i] = sodecl_sincos_core(x[i], s + i, c + i);
}
'''


@functools.lru_cache(None)
def _lib():
    d = tempfile.mkdtemp(prefix="sodecl_sincos_")
    cpp = os.path.join(d, "sincos_host.cpp")
    with open(cpp, "w") as f:
        f.write(_HARNESS % (DEVICE, DEVICE))
    so = os.path.join(d, "sincos_host.so")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-fno-fast-math", "-shared", "-fPIC", cpp, "-o", so],
                   check=True)
    lib = ctypes.CDLL(so)
    lib.sincos_host.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_long]
    return lib


def sincos_host(x):
    """(sine, cosine, flag: the fast path covers the argument)."""
    x = np.ascontiguousarray(x, dtype=np.float64)
    s, c = np.empty_like(x), np.empty_like(x)
    ok = np.empty(x.shape, dtype=np.uint8)
    _lib().sincos_host(x.ctypes.data, s.ctypes.data, c.ctypes.data, ok.ctypes.data, x.size)
    return s, c, ok.astype(bool)
