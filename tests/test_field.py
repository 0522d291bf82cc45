"""The field form's sincos() on the CPU, and when runs take the field form."""
import numpy as np
import pytest

import sodecl_amd
from sodecl_amd import sodecl_interface as si
from tests.sincos_host import sincos_host


@pytest.mark.skipif(np.finfo(np.longdouble).nmant < 63, reason="needs x87 long double for the references")
@pytest.mark.parametrize("reach", [0.8, 7.0, 1e4, 2.0 ** 30])
def test_sincos_error(reach):
    """Below 0.9 ulp, the bound the sine of system sources is held to, on
    random arguments and 3000 ulps around the first quadrant boundaries;
    library hand-over exactly where the reduction does not hold."""
    r = np.random.default_rng(3)
    x = np.concatenate([r.uniform(-reach, reach, 400_000),
                        (np.arange(1, 9)[:, None] * (np.pi / 4) * (1 + np.arange(-3000, 3001) * 2.0 ** -52)).ravel()])
    s, c, ok = sincos_host(x)
    assert ok.mean() > 0.98
    for got, fn in ((s, np.sin), (c, np.cos)):
        ref = fn(x.astype(np.longdouble))
        err = np.abs(got.astype(np.longdouble) - ref) / np.spacing(np.abs(ref.astype(np.float64)))
        assert err[ok].max() < 0.9
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 2.0 ** 31, -1e300, np.pi, np.pi / 2])
    assert not sincos_host(special)[2].any()


@pytest.mark.parametrize("opts,expected", [
    ({}, True), (dict(group_size=16), True), (dict(schedule="lane"), False), (dict(pairwise=-1), False),
    (dict(pairwise=4), False), (dict(fp_contract=1), False), (dict(group_size=2), False)])
def test_field_form_selected(opts, expected):
    """The automatic pairwise choice of the default arithmetic, with at most
    16 components per lane; explicit layouts, the strict arithmetic and the
    other schedules keep the pair terms or the per-component drift."""
    s = si.Session(sodecl_amd.system_path("kuramoto"), 2, 500, 40, 41, 0, 0.01, 1.0, 10, 0, opts)
    assert s.compile_only("gfx950") > 1000
    assert ("#define SODECL_USE_FIELD 1" in s.program_source()) == expected


@pytest.mark.parametrize("solver,n,orbits,lanes,cpl", [
    (2, 64, 16384, 16, 4), (2, 33, 1500, 32, 2), (1, 10, 1024, 16, 1), (1, 20, 30000, 4, 5), (0, 32, 262144, 8, 4),
    (0, 32, 20000, 16, 2), (2, 600, 100, 64, 10)])
def test_field_form_lanes(solver, n, orbits, lanes, cpl):
    """Lanes per orbit by the estimated time of the fullest SIMD (256 compute
    units assumed without a GPU); noise pairs stay with one lane."""
    nnoi = n if solver == 0 else 0
    s = si.Session(sodecl_amd.system_path("kuramoto"), solver, orbits, n, n + 1 + nnoi, nnoi, 0.01, 1.0, 10, 0,
                   {"schedule": "group"})
    s.compile_only("gfx950")
    src = s.program_source()
    assert f"#define SODECL_FL {lanes}\n#define SODECL_FC {cpl}\n" in src
