"""Implicit adjoint on either side of the size up to which the transposed system
is eliminated: against the oracle's forward sensitivity at a Newton threshold of
1e-14, to 1e-9 of the largest gradient entry (as the adjoint is held to)."""
import numpy as np
import pytest
import torch

from sodecl_amd import configs
from sodecl_amd.torch_ops import Integrator
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("solver", [3, 4])
@pytest.mark.parametrize("n", [10, 11, 12])
def test_sizes(solver, n):
    orbits = 9
    cfg = configs.kuramoto_rk4(orbits=orbits, n=n, seed=n, dt=0.01, tspan=0.3, ksteps=10)
    integ = Integrator(cfg["system"], solver, orbits, n, n + 1, cfg["dt"], cfg["tspan"], cfg["ksteps"], newton_tol=1e-14)
    y0 = torch.tensor(cfg["y0"], device=DEV, requires_grad=True)
    p = torch.tensor(cfg["params"], device=DEV, requires_grad=True)
    cot = np.random.default_rng(n).normal(size=(integ.nsnap, n, orbits))
    got = torch.autograd.grad(integ(y0, p), (y0, p), torch.tensor(cot, device=DEV))
    ref = Oracle("kuramoto").sensitivity_gradient({3: "ie", 4: "im"}[solver], cfg["y0"], cfg["params"], cot, cfg["dt"],
                                                  cfg["tspan"], cfg["ksteps"], newton_tol=1e-14)
    for g, r in zip(got, ref):
        assert np.abs(g.cpu().numpy() - r).max() <= 1e-9 * np.abs(r).max()
