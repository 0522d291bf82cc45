"""Adjoint in field form with many parameters (fewer orbits per block, more
lanes per orbit): the gradients of the same system without the unused ones, and
zeros for those."""
import numpy as np
import pytest
import torch

from sodecl_amd import configs
from sodecl_amd.torch_ops import Integrator

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("n,npar,orbits", [(2, 250, 40000), (3, 1000, 500), (3, 3000, 17)])
def test_unused_parameters(n, npar, orbits):
    cfg = configs.kuramoto_rk4(orbits=orbits, n=n, seed=n, dt=0.01, tspan=0.2, ksteps=5)
    cot = None
    grads = []
    for m in (n + 1, npar):
        integ = Integrator(cfg["system"], 2, orbits, n, m, cfg["dt"], cfg["tspan"], cfg["ksteps"], schedule="group")
        y0 = torch.tensor(cfg["y0"], device=DEV, requires_grad=True)
        p = torch.zeros(orbits, m, dtype=torch.float64, device=DEV)
        p[:, :n + 1] = torch.tensor(cfg["params"], device=DEV)
        p.requires_grad_(True)
        if cot is None:
            cot = torch.tensor(np.random.default_rng(n).normal(size=(integ.nsnap, n, orbits)), device=DEV)
        grads.append(torch.autograd.grad(integ(y0, p), (y0, p), cot))
    (gy, gp), (hy, hp) = grads
    # another split of sums of up to n terms over 20 steps
    assert (gy - hy).abs().max() <= 1e-12 * gy.abs().max()
    assert (gp - hp[:, :n + 1]).abs().max() <= 1e-12 * gp.abs().max()
    assert (hp[:, n + 1:] == 0).all()
