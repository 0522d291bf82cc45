"""The adjoint of a stored forward run reads that run's rows, whatever options the
session has by then."""
import numpy as np
import pytest
import torch

from sodecl_amd import configs, sodecl_interface as si

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("solver", [1, 2])
@pytest.mark.parametrize("first,then", [(dict(), dict(pairwise=-1)), (dict(pairwise=-1), dict(pairwise=0)),
                                        (dict(), dict(fp_contract=1)), (dict(group_size=64), dict(group_size=0))])
def test_options_changed_between_forward_and_adjoint(solver, first, then):
    orbits, n = 130, 12
    cfg = configs.kuramoto_rk4(orbits=orbits, n=n, seed=n, dt=0.01, tspan=0.3, ksteps=5)
    cot = None
    grads = []
    for change in (False, True):
        s = si.Session(cfg["system"], solver, orbits, n, n + 1, 0, cfg["dt"], cfg["tspan"], cfg["ksteps"], 0,
                       dict(schedule="group", **first))
        s.setup(cfg["y0"], cfg["params"])
        full = lambda *shape: torch.full(shape, float("nan"), dtype=torch.float64, device=DEV)
        y, p = torch.tensor(cfg["y0"], device=DEV), torch.tensor(cfg["params"], device=DEV)
        t, traj, work = torch.zeros(orbits, dtype=torch.float64, device=DEV), full(s.nsnap, n, orbits), full(
            s.stored_workspace_size())
        gy, gp = full(orbits, n), full(orbits, n + 1)
        if cot is None:
            cot = torch.tensor(np.random.default_rng(n).normal(size=(s.nsnap, n, orbits)), device=DEV)
        s.run_device_stored(t.data_ptr(), y.data_ptr(), p.data_ptr(), traj.data_ptr(), work.data_ptr(), 0)
        if change:
            s.set_options(then)
        s.adjoint_device_stored(p.data_ptr(), cot.data_ptr(), gy.data_ptr(), gp.data_ptr(), work.data_ptr(), 0)
        torch.cuda.synchronize()
        assert not (gy.isnan().any() or gp.isnan().any())
        grads.append((gy.cpu().numpy(), gp.cpu().numpy()))
    for a, b in zip(*grads):
        np.testing.assert_array_equal(a, b)
