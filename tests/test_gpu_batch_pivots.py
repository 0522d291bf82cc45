"""The batched solver's two-level solve (paired reciprocals, no elimination)
and its general windowed solve against the same plugins through LDS, with
pivots whose products leave the range of a double and a pivot of zero."""
import numpy as np
import pytest
import torch

from sodecl_amd import sodecl_interface as si

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
DT = 1.0 / 128

# two species per cell: y[2k]' = p0 y[2k] + p1 y[2k+1], y[2k+1]' = p2 y[2k+1]
TWO = """
#define SODE_REACH 1
double sode_system_window(int i, double t, double w[], double p[_numpar_])
{
    return (i & 1) ? p[2] * w[0] : p[0] * w[0] + p[1] * w[1];
}
void calc_jacobian_band_window(int i, double w[], double p[_numpar_], double* lower, double* diag, double* upper)
{
    *diag = (i & 1) ? p[2] : p[0];
    *upper = (i & 1) ? 0.0 : p[1];
    *lower = 0.0;
}
"""
# a chain: y[i]' = p0 y[i] + p1 (y[i-1] + y[i+1])
CHAIN = """
#define SODE_REACH 1
double sode_system_window(int i, double t, double w[], double p[_numpar_])
{
    const double left = i > 0 ? w[-1] : 0.0;
    const double right = i < _numeq_ - 1 ? w[1] : 0.0;
    return p[0] * w[0] + p[1] * (left + right);
}
void calc_jacobian_band_window(int i, double w[], double p[_numpar_], double* lower, double* diag, double* upper)
{
    *diag = p[0];
    *upper = p[1];
    *lower = p[1];
}
"""
REST = """
double sode_system_i(int i, double t, double y[_numeq_], double p[_numpar_])
{
    return sode_system_window(i, t, y + i, p);
}
void sode_system(double t, double y[_numeq_], double yout[_numeq_], double p[_numpar_])
{
    for (int i = 0; i < _numeq_; i++)
        yout[i] = sode_system_window(i, t, y + i, p);
}
void calc_jacobian_band_i(int i, double y[_numeq_], double p[_numpar_], double* lower, double* diag, double* upper)
{
    calc_jacobian_band_window(i, y + i, p, lower, diag, upper);
}
void calc_jacobian_band(double y[_numeq_], double lower[_numeq_], double diag[_numeq_], double upper[_numeq_], double p[_numpar_])
{
    for (int i = 0; i < _numeq_; i++)
        calc_jacobian_band_window(i, y + i, p, &lower[i], &diag[i], &upper[i]);
}
void calc_jacobian(double y[_numeq_], double jac[_numeq_][_numeq_], double p[_numpar_])
{
    for (int i = 0; i < _numeq_; i++)
        for (int j = 0; j < _numeq_; j++)
            jac[i][j] = 0.0;
    for (int i = 0; i < _numeq_; i++)
    {
        double lo, di, up;
        calc_jacobian_band_window(i, y + i, p, &lo, &di, &up);
        jac[i][i] = di;
        if (i + 1 < _numeq_)
        {
            jac[i][i + 1] = up;
            jac[i + 1][i] = lo;
        }
    }
}
"""


def run(source, solver, sizes, cls, y0, params):
    b = si.Batch(source, solver, DT, 4, 3, sizes, 0, {"newton_max_iter": 4}, True)
    b.setup(cls, np.full(len(cls), 4, np.int32))
    out = torch.full((b.output_size(),), -1.0, dtype=torch.float64, device=DEV)
    nu = torch.zeros(len(cls), dtype=torch.int64, device=DEV)
    y, p = torch.tensor(y0, device=DEV), torch.tensor(params, device=DEV)
    b.run_device(y.data_ptr(), p.data_ptr(), out.data_ptr(), nu.data_ptr(), 0)
    torch.cuda.synchronize()
    assert ("#define SODECL_WINDOW 1" in b.program_source()) == ("SODE_REACH" in source)
    return out.cpu().numpy(), nu.cpu().numpy(), b.offsets()


@pytest.mark.parametrize("solver", [3, 4])
@pytest.mark.parametrize("plugin", ["two", "chain"])
def test_windowed_solve_vs_lds(plugin, solver):
    """Linear systems: the Newton updates are x = M^-1 r with a residual as
    large as y, so each unknown carries a few units of 2^-53 of the largest
    state per step from either solve; 4 steps, and M within a factor of ten
    of its diagonal: 1e-13 of the largest initial state."""
    sizes = [2, 18, 130, 512]   # one lane, ragged, lanes half used, all lanes
    # (two: products of pivots that overflow or underflow to none, pivots of
    # opposite signs, and a pivot of zero; chain: diagonally dominant)
    rates = {"two": [(-3.0, -0.3, -2.0), (-1e200, -1e199, -1e190), (-1e160, 1e159, -1e170), (-5.0, 0.2, 40.0),
                     (-1e300, 1e298, -2.0), (1.0 / DT if solver == 3 else 2.0 / DT, 0.5, -2.0), (-1e4, 0.0, -1e-4)],
             "chain": [(-3.0, 0.7, 0.0), (-1e5, 2e4, 0.0), (-50.0, -10.0, 0.0)]}[plugin]
    rng = np.random.default_rng(7)
    orbits = 60
    cls = (np.arange(orbits) % 4).astype(np.int32)
    params = np.array([rates[(o // 4) % len(rates)] for o in range(orbits)])
    y0 = np.concatenate([rng.uniform(0.5, 1.0, sizes[c]) for c in cls])
    window = (TWO if plugin == "two" else CHAIN) + REST
    got, updates, (_, off) = run(window, solver, sizes, cls, y0, params.ravel())
    want, updates_lds, _ = run(window.replace("SODE_REACH", "REACH").replace("band_window", "band_at"), solver, sizes,
                               cls, y0, params.ravel())
    broken = np.array([plugin == "two" and (o // 4) % len(rates) == 5 for o in range(orbits)])
    for o in range(orbits):
        a, b = (v[off[o]:off[o] + 2 * sizes[cls[o]]].reshape(2, -1) for v in (got, want))
        np.testing.assert_array_equal(a[0], b[0])
        assert np.all(np.isnan(a[1])) if broken[o] else np.all(np.isfinite(a[1]))
        if not broken[o]:
            assert np.max(np.abs(a[1] - b[1])) <= 1e-13
            # (four midpoint steps of an infinitely stiff component return to its start)
            assert np.max(np.abs(a[1] - a[0])) > 1e-3 or np.abs(params[o]).max() > 100
