"""launch_config() is the schedule chosen, launch_geometry() what it launches:
kernel, lanes per orbit, threads per block (256 compute units assumed without a
GPU)."""
import pytest

import sodecl_amd
from sodecl_amd import sodecl_interface as si


@pytest.mark.parametrize("system,solver,orbits,n,nnoi,opts,config,geometry", [
    ("kuramoto", 2, 300, 5, 0, {}, (1, 1, 128), ("sodecl_field", 8, 64)),
    ("kuramoto", 2, 300, 5, 0, dict(schedule="lane"), (1, 1, 128), ("sodecl_lane", 1, 128)),
    ("kuramoto", 2, 16384, 64, 0, {}, (2, 64, 256), ("sodecl_field", 16, 256)),
    ("kuramoto", 2, 16384, 64, 0, dict(pairwise=-1), (2, 64, 256), ("sodecl_group", 64, 256)),
    ("oculomotor", 0, 5000, 6, 2, {}, (1, 1, 128), ("sodecl_lane", 8, 128)),
    ("oculomotor", 0, 5000, 6, 2, dict(schedule="plain"), (1, 1, 128), ("sodecl_lane", 1, 128)),
    ("oculomotor", 2, 300, 6, 0, {}, (4, 2, 128), ("sodecl_team", 2, 128)),
    ("oculomotor", 4, 300, 6, 0, {}, (1, 1, 128), ("sodecl_lane", 1, 128))])
def test_geometry(system, solver, orbits, n, nnoi, opts, config, geometry):
    npar = (n + 1 if system == "kuramoto" else 6) + nnoi
    s = si.Session(sodecl_amd.system_path(system), solver, orbits, n, npar, nnoi, 1e-3, 0.1, 10, 0, opts)
    assert s.launch_geometry() == ("", 0, 0)
    assert s.compile_only("gfx950") > 1000
    assert s.launch_config() == config
    assert s.launch_geometry() == geometry
