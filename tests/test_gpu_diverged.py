"""Implicit solvers on orbits that diverge: components that no coefficient
couples become NaN together, as in the reference's sweep (0 * NaN), in the
default arithmetic as in the strict one."""
import numpy as np
import pytest

from sodecl_amd import configs, sodecl_interface as si

pytestmark = pytest.mark.gpu

# component 0 overflows; the others decay on their own, their couplings are
# constant zeros
SOURCE = """
void sode_system(double t, double y[_numeq_], double yout[_numeq_], double p[_numpar_])
{
    yout[0] = p[0] * y[0] * y[0] * y[0];
    for (int i = 1; i < _numeq_; i++) yout[i] = -y[i];
}
void calc_jacobian(double y[_numeq_], double jac[_numeq_][_numeq_], double p[_numpar_])
{
    for (int i = 0; i < _numeq_; i++)
        for (int j = 0; j < _numeq_; j++) jac[i][j] = 0;
    jac[0][0] = 3 * p[0] * y[0] * y[0];
    for (int i = 1; i < _numeq_; i++) jac[i][i] = -1;
}
"""


def run(make, strict, y0, p):
    s = make(dict(fp_contract=strict, newton_max_iter=20))
    s.setup(y0, p)
    return s.run().reshape(s.nsnap, y0.shape[1], len(y0))


@pytest.mark.parametrize("solver,ksteps", [(3, 1), (4, 1), (3, 4), (4, 4)])
@pytest.mark.parametrize("n", [2, 3, 5])
def test_uncoupled_components(solver, n, ksteps):
    orbits = 70
    r = np.random.default_rng(n)
    y0, p = r.normal(size=(orbits, n)), np.ones((orbits, 1))
    y0[1:20, 0] = 1e120        # the drift overflows
    y0[20:25, n - 1] = np.nan
    y0[25:30, 1] = np.inf
    y0[30:33, 0] = 1e200
    make = lambda opts: si.Session(SOURCE, solver, orbits, n, 1, 0, 0.01, 0.04 * ksteps, ksteps, 0, opts, True)
    a, b = run(make, 0, y0, p), run(make, 1, y0, p)
    np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
    assert np.isnan(b[-1][:, 1:33]).all() and not np.isnan(b[-1][:, 33:]).any()
    # where dt 3 y^2 stays below 0.03 (near 1 the Newton matrix is singular)
    mild = np.abs(b[:, 0]).max(0) < 1
    assert mild[33:].sum() > 10
    np.testing.assert_allclose(a[:, :, mild], b[:, :, mild], rtol=1e-10, atol=1e-12)


@pytest.mark.parametrize("solver", [3, 4])
def test_oculomotor(solver):
    cfg = configs.oculomotor_rk4(orbits=64, seed=1, dt=1e-5, tspan=5e-5, ksteps=1)
    cfg["solver"] = solver
    cfg["y0"][:, 5] += 1.0
    for k in range(6):
        cfg["y0"][k, k] = np.nan
        cfg["y0"][10 + k, k] = np.inf
    cfg["y0"][20:24, 3] = 1e120   # y3 y4^2 overflows
    cfg["y0"][20:24, 4] = 1e120
    make = lambda opts: configs.session_for(cfg, **opts)
    a, b = run(make, 0, cfg["y0"], cfg["params"]), run(make, 1, cfg["y0"], cfg["params"])
    np.testing.assert_array_equal(np.isnan(a), np.isnan(b))
    assert not np.isnan(b[:, :, 24:]).any()
