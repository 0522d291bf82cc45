"""The field form's sincos() marks arguments it does not cover by a NaN sine,
and only in sources that allow it."""
import ctypes
import os
import subprocess

import numpy as np

import sodecl_amd
from sodecl_amd import sodecl_interface as si
from tests.sincos_host import DEVICE, sincos_host


def test_marked_sincos(tmp_path):
    cpp, so = tmp_path / "m.cpp", str(tmp_path / "m.so")
    cpp.write_text(f'''#include <math.h>
#define SODECL_MATH_FN static inline
#include "{os.path.join(DEVICE, "sin.hip")}"
#include "{os.path.join(DEVICE, "sincos.hip")}"
extern "C" void marked(const double* x, double* s, double* c, long n)
{{
    for (long i = 0; i < n; ++i) sodecl_sincos_marked(x[i], s + i, c + i);
}}
''')
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", str(cpp), "-o", so], check=True)
    f = ctypes.CDLL(so).marked
    f.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_long]
    r = np.random.default_rng(1)
    x = np.concatenate([r.uniform(-10, 10, 20000), r.uniform(-2.0 ** 30, 2.0 ** 30, 20000),
                        np.arange(-50, 51) * (np.pi / 2), [0.0, -0.0, 2.0 ** 30 + 1, 1e22, -1e300, np.inf, np.nan]])
    s, c = np.empty_like(x), np.empty_like(x)
    f(x.ctypes.data, s.ctypes.data, c.ctypes.data, x.size)
    hs, hc, ok = sincos_host(x)
    assert 50 < (~ok).sum() < 200
    assert np.isnan(s[~ok]).all()
    np.testing.assert_array_equal(s[ok], hs[ok])
    np.testing.assert_array_equal(c[ok], hc[ok])


def test_marked_copy_only_where_the_source_allows_it():
    src = open(sodecl_amd.system_path("kuramoto")).read()
    without = "\n".join(line for line in src.split("\n") if "#define SODE_FIELD_MARKED_SINCOS" not in line)
    guarded = "#ifndef GUARD\n#define GUARD\n" + without + "\n#endif\n"   # cannot stand twice in a program
    sizes = []
    for text in (src, without, guarded):
        s = si.Session(text, 2, 500, 10, 11, 0, 0.01, 1.0, 10, 0, {}, True)
        sizes.append(s.compile_only("gfx950"))
        assert "#ifdef SODE_FIELD_MARKED_SINCOS" in s.program_source()
    assert sizes[0] != sizes[1] and sizes[1] == sizes[2]
