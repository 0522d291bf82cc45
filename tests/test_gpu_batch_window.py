"""The batched solver's windowed form (states, band and solve in registers)
at the edges of its lane shares, and a plugin without it, against the oracle."""
import numpy as np
import pytest
import torch

import sodecl_amd
from sodecl_amd import configs, sodecl_interface as si
from tests.test_gpu_batch import check_against_oracle

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def run(cfg, source=None):
    path = cfg["system"]
    b = si.Batch(source or open(path).read(), cfg["solver"], cfg["dt"], cfg["ksteps"], cfg["npar"], cfg["class_neq"],
                 0, {"newton_max_iter": cfg["newton_max_iter"]}, True)
    b.setup(cfg["cls"], cfg["steps"])
    y0, p = torch.tensor(cfg["y0"], device=DEV), torch.tensor(cfg["params"], device=DEV)
    out = torch.full((b.output_size(),), float("nan"), dtype=torch.float64, device=DEV)
    nu = torch.zeros(cfg["orbits"], dtype=torch.int64, device=DEV)
    b.run_device(y0.data_ptr(), p.data_ptr(), out.data_ptr(), nu.data_ptr(), 0)
    torch.cuda.synchronize()
    return (out.cpu().numpy(), nu.cpu().numpy(), *b.offsets()), b.program_source()


# (cells per class, orbits, rows per lane): one lane per orbit, lanes that come
# out even or not, the widest, past the widest (through LDS), eight rows
@pytest.mark.parametrize("solver", [3, 4])
@pytest.mark.parametrize("cells,orbits,rows", [((1, 2, 8), 45, (2, 2, 2)), ((9, 31, 65), 45, (2, 2, 4)),
                                               ((255, 256, 257), 9, (8, 8, 9)), ((15, 37, 125), 17000, (8, 8, 8))])
def test_windowed_batch_vs_oracle(solver, cells, orbits, rows):
    cfg = configs.brusselator_batch(orbits=orbits, seed=orbits, solver=solver, cells=cells, smin=10, smax=20,
                                    ksteps=5, newton_max_iter=1000)
    got, src = run(cfg)
    lanes = [int(l.split()[2]) for l in src.splitlines() if l.startswith("#define SODECL_BR ")]
    assert tuple(lanes) == rows
    assert np.all(np.isfinite(got[0]))
    assert check_against_oracle(cfg, *got, range(min(orbits, 45))) <= 1


def test_plugin_without_windowed_form():
    """Without the windowed entry points the batch runs through LDS."""
    cfg = configs.brusselator_batch(orbits=60, seed=4, solver=3, cells=(5, 20, 150), smin=10, smax=40, ksteps=10)
    source = open(sodecl_amd.system_path("brusselator")).read()
    got, src = run(cfg, source.replace("SODE_REACH", "REACH").replace("band_window", "band_at"))
    assert "#define SODECL_WINDOW 1" not in src
    assert check_against_oracle(cfg, *got, range(60)) <= 1


# (cells, orbits, rows per lane, one wavefront at a time): two rows, four and eight
# rows one at a time, four rows stacked (256 compute units)
@pytest.mark.parametrize("cells,orbits,rows,alone", [((16, 64, 256), 2300, (2, 2, 8), True),
                                                     ((16, 64, 256), 3000, (4, 4, 8), True),
                                                     ((16, 64, 256), 6000, (8, 8, 8), True),
                                                     ((16, 64, 256), 8300, (4, 4, 8), False)])
def test_rows_by_wavefronts_per_simd(cells, orbits, rows, alone):
    cfg = configs.brusselator_batch(orbits=orbits, seed=orbits, solver=3, cells=cells, smin=5, smax=15, ksteps=5,
                                    newton_max_iter=5)
    got, src = run(cfg)
    lines = src.splitlines()
    assert tuple(int(l.split()[2]) for l in lines if l.startswith("#define SODECL_BR ")) == rows
    assert all(l.endswith(" 1, 1") == alone for l in lines if l.startswith("#define SODECL_BATCH_WAVES "))
    assert check_against_oracle(cfg, *got, range(0, orbits, orbits // 40)) <= 1
