"""Windowed batch with more parameters than its registers hold (more than eight:
rows in LDS), up to sizes at which the orbits of a wavefront must get fewer."""
import numpy as np
import pytest

from sodecl_amd import configs, sodecl_interface as si
from tests.test_gpu_batch import check_against_oracle
from tests.test_gpu_batch_window import run


def source_and_config(npar, cells, orbits, solver=3):
    cfg = configs.brusselator_batch(orbits=orbits, seed=npar, solver=solver, cells=cells, smin=5, smax=15, ksteps=5,
                                    newton_max_iter=1000)
    src = open(cfg["system"]).read()
    for k in range(3):   # the model's parameters are the last three
        src = src.replace(f"p[{k}]", f"p[_numpar_ - {3 - k}]")
    wide = dict(cfg, npar=npar, params=np.concatenate([np.full((orbits, npar - 3), np.nan), cfg["params"]], 1))
    return src, cfg, wide


def lanes_of(program):
    return tuple(int(l.split()[2]) for l in program.splitlines() if l.startswith("#define SODECL_LPO "))


# (parameters, lanes per orbit of classes of 2, 8 and 32 equations)
@pytest.mark.parametrize("npar,lanes", [(3, (1, 1, 4)), (9, (1, 1, 4)), (31, (1, 1, 4)), (32, (2, 2, 4)), (129, (8, 8, 8)),
                                        (400, (16, 16, 16)), (3000, (64, 64, 64))])
def test_lanes_by_parameters(npar, lanes):
    src, _, _ = source_and_config(max(npar, 3), (1, 4, 16), 3)
    b = si.Batch(src, 3, 0.01, 5, npar, [2, 8, 32], 0, {}, True)
    assert b.compile_only("gfx950") > 1000
    assert lanes_of(b.program_source()) == lanes


@pytest.mark.gpu
@pytest.mark.parametrize("solver", [3, 4])
@pytest.mark.parametrize("npar,cells,orbits", [(9, (1, 4, 16), 200), (400, (1, 4, 16), 45), (9, (4, 37, 200), 9000),
                                               (130, (2, 9, 200), 17000), (1500, (1, 3, 100), 20)])
def test_many_parameters(solver, npar, cells, orbits):
    src, cfg, wide = source_and_config(npar, cells, orbits, solver)
    got, program = run(wide, src)
    assert "#define SODECL_WINDOW 1" in program
    assert np.all(np.isfinite(got[0]))
    assert check_against_oracle(cfg, *got, range(0, orbits, max(1, orbits // 40))) <= 1


@pytest.mark.gpu
def test_more_parameters_than_a_block_holds():
    src, cfg, wide = source_and_config(21000, (1, 4, 16), 3)
    with pytest.raises(RuntimeError, match="LDS"):
        run(wide, src)
