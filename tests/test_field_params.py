"""Field form of sources with many parameters: the adjoint's LDS for their
gradients bounds the orbits of a block."""
import pytest

import sodecl_amd
from sodecl_amd import sodecl_interface as si


# (components, parameters, orbits, group size): the orbits and automatic lanes at
# which blocks of 256 threads hold 256 orbits down to one orbit per wavefront
@pytest.mark.parametrize("n,npar,orbits,group", [(2, 81, 300000, 0), (2, 250, 300000, 0), (3, 1000, 70000, 0),
                                                 (4, 300, 300000, 4), (8, 300, 70000, 8), (3, 5000, 300, 0),
                                                 (16, 20000, 70000, 64), (40, 20000, 100, 0)])
def test_adjoint_compiles(n, npar, orbits, group):
    s = si.Session(sodecl_amd.system_path("kuramoto"), 2, orbits, n, npar, 0, 1e-3, 0.1, 10, 0,
                   dict(schedule="group", group_size=group))
    assert s.compile_only("gfx950") > 1000
    src = s.program_source()
    assert "#define SODECL_ADJOINT 1" in src
    value = lambda name: int(src.split(f"#define {name} ")[1].split()[0])
    lanes = value("SODECL_FL")
    assert lanes == group or group == 0
    assert value("SODECL_FBLOCK") // lanes * npar * 8 <= 160 * 1024


def test_few_parameters_keep_their_blocks():
    s = si.Session(sodecl_amd.system_path("kuramoto"), 2, 300000, 3, 4, 0, 1e-3, 0.1, 10, 0, dict(schedule="group"))
    s.compile_only("gfx950")
    assert "#define SODECL_FL 1\n" in s.program_source() and "#define SODECL_FBLOCK 256\n" in s.program_source()
