"""The field form of the group schedule on the GPU: against the oracle at the
edges of its lane shares, and its adjoint against the forward sensitivity."""
import numpy as np
import pytest
import torch

from sodecl_amd import configs, sodecl_interface as si
from sodecl_amd.torch_ops import Integrator
from oracle.oracle import Oracle
from tests.parity import assert_traj_close
from tests.sincos_host import sincos_host

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

# one component per lane, shares that come out even or not, spare lanes, one
# lane per orbit, the most components per lane; odd noise counts and steps
EDGES = [(1, 3, 4, 10), (2, 33, 32, 7), (2, 20, 4, 10), (2, 64, 4, 10), (1, 8, 1, 10), (2, 17, 16, 3), (1, 5, 64, 1),
         (0, 5, 8, 7), (0, 6, 2, 10), (0, 7, 2, 3), (0, 33, 16, 10), (0, 2, 2, 1)]


@pytest.mark.parametrize("solver,n,group,ksteps", EDGES)
def test_field_form_vs_oracle(solver, n, group, ksteps):
    orbits = 67
    if solver == 0:
        cfg = configs.kuramoto_em(orbits=orbits, n=n, seed=n, tspan=0.1, ksteps=ksteps)
        cfg["counters"] = np.random.default_rng(n).integers(0, 2 ** 40, orbits).astype(np.float64)
        cfg["counters"][::9] += 0.5          # whole and fractional counters in one wavefront
    else:
        cfg = configs.kuramoto_rk4(orbits=orbits, n=n, seed=n, dt=0.01, tspan=0.6, ksteps=ksteps)
        cfg["solver"] = solver
    s = configs.session_for(cfg, schedule="group", group_size=group)
    s.setup(cfg["y0"], cfg["params"], None, cfg.get("counters"))
    out = s.run().reshape(s.nsnap, n, orbits)
    assert "#define SODECL_USE_FIELD 1" in s.program_source()
    ref = Oracle("kuramoto").run({0: "em", 1: "euler", 2: "rk4"}[solver], cfg["y0"], cfg["params"], cfg["dt"],
                                 cfg["tspan"], cfg["ksteps"], counters=cfg.get("counters"), nnoi=cfg["nnoi"])
    assert_traj_close(out, ref["out"], what=f"solver {solver} N={n} G={group}")
    if solver == 0:
        np.testing.assert_array_equal(s.counters(), ref["counters"])


def test_field_form_large_and_exact_phases():
    """Phases beyond the reduction's range and at multiples of pi/2 take the
    library's sincos, also next to ordinary ones: the pairwise drift's steps to
    one last place of the phase per step either way."""
    n, orbits, steps = 12, 40, 20
    cfg = configs.kuramoto_rk4(orbits=orbits, n=n, seed=2, dt=0.01, tspan=0.2, ksteps=steps)
    cfg["y0"][::3] += 2.0 ** 31
    cfg["y0"][1::3, :4] = np.array([0.0, -0.0, np.pi, -np.pi / 2])
    got = []
    for mode in (0, -1):
        s = configs.session_for(cfg, schedule="group", pairwise=mode)
        s.setup(cfg["y0"], cfg["params"])
        got.append(s.run().reshape(s.nsnap, n, orbits)[-1])
    spacing = np.spacing(np.abs(got[1]) + 1.0)
    assert np.all(np.abs(got[0] - got[1]) <= 2 * steps * spacing)
    assert np.abs(got[0] - cfg["y0"].T)[:, ::3].max() > 0.1   # the large phases moved


def test_sincos_in_a_source_matches_host_build():
    """f = (sin p, cos p) of one Euler step from -0 with dt = 1 stores both
    values; library_sin = 1 gives the device library's."""
    src = """
void sode_system(double t, double y[_numeq_], double yout[_numeq_], double p[_numpar_])
{
    for (int i = 0; i < _numpar_; i++) sincos(p[i], &yout[2 * i], &yout[2 * i + 1]);
}
"""
    r = np.random.default_rng(5)
    x = np.concatenate([r.uniform(-8, 8, 40000), r.uniform(-2.0 ** 30, 2.0 ** 30, 8000),
                        np.arange(-400, 400) * (np.pi / 2), [0.0, -0.0, 2.0 ** 31, np.inf, -np.inf, np.nan, 1e22, 3.0]])
    x = x.reshape(-1, 8)
    got = []
    for lib in (0, 1):
        s = si.Session(src, 1, len(x), 16, 8, 0, 1.0, 1.0, 1, 0, dict(schedule="lane", library_sin=lib), True)
        s.setup(np.full((len(x), 16), -0.0), x)
        got.append(s.run().reshape(2, 8, 2, len(x))[1].transpose(2, 0, 1))
    hs, hc, ok = sincos_host(x)
    for k, host in ((0, hs), (1, hc)):
        np.testing.assert_array_equal(got[0][:, :, k][ok].view(np.uint64), host[ok].view(np.uint64))
        np.testing.assert_array_equal(got[0][:, :, k][~ok].view(np.uint64), got[1][:, :, k][~ok].view(np.uint64))


@pytest.mark.parametrize("solver,n,group,stored", [(1, 3, 4, False), (2, 33, 32, False), (2, 20, 4, True),
                                                   (2, 64, 16, True), (1, 17, 2, False), (2, 6, 1, False)])
def test_field_adjoint_vs_forward_sensitivity(solver, n, group, stored):
    """1e-9 of the largest gradient entry, as the pairwise adjoint is held to."""
    orbits, k = 19, 5
    cfg = configs.kuramoto_rk4(orbits=orbits, n=n, seed=n, dt=0.01, tspan=0.3, ksteps=5)
    integ = Integrator(cfg["system"], solver, orbits, n, n + 1, cfg["dt"], cfg["tspan"], cfg["ksteps"],
                       store_stages=stored, schedule="group", group_size=group)
    y0 = torch.tensor(cfg["y0"], device=DEV, requires_grad=True)
    p = torch.tensor(cfg["params"], device=DEV, requires_grad=True)
    cot = np.random.default_rng(n).normal(size=(integ.nsnap, n, orbits))
    gy, gp = torch.autograd.grad(integ(y0, p), (y0, p), torch.tensor(cot, device=DEV))
    ry, rp = Oracle("kuramoto").sensitivity_gradient({1: "euler", 2: "rk4"}[solver], cfg["y0"], cfg["params"], cot,
                                                     cfg["dt"], cfg["tspan"], cfg["ksteps"], orbit_range=(0, k))
    for g, ref in ((gy, ry), (gp, rp)):
        assert np.max(np.abs(g.cpu().numpy()[:k] - ref)) <= 1e-9 * np.max(np.abs(ref))
