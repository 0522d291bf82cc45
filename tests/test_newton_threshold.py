"""The threshold that the implicit midpoint compares its squared residual norm
with: v lies below it just where sqrt(v) lies below the Newton tolerance."""
import numpy as np
import pytest

import sodecl_amd
from sodecl_amd import sodecl_interface as si


@pytest.mark.parametrize("tol", [0.0, 3.3e-5, 1e-200, 1e160])
def test_squared_threshold_is_exact(tol, tmp_path, monkeypatch):
    monkeypatch.setenv("SODECL_AMD_CACHE_DIR", str(tmp_path))
    s = si.Session(sodecl_amd.system_path("oculomotor"), 4, 64, 6, 6, 0, 1e-4, 1e-2, 10, 0,
                   dict(newton_tol=tol) if tol else {})
    s.compile_only("gfx950")
    line = next(l for l in s.program_source().splitlines() if l.startswith("#define SODECL_EPSILON1_SQUARED "))
    text = line.split()[2]
    t = np.inf if "inf" in text else float.fromhex(text)
    eps = tol or 1e-7
    with np.errstate(over="ignore"):
        around = t * (1 + np.arange(-50, 51) * 2.0 ** -52) if np.isfinite(t) else np.array([1e308, np.inf])
    around = np.concatenate([around, [0.0, np.nextafter(t, 0.0), t, np.nextafter(t, np.inf), np.inf, np.nan]])
    np.testing.assert_array_equal(around < t, np.sqrt(around) < eps)
