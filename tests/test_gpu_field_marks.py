"""Field form of sources whose features do not carry a NaN of sincos() to the
sums: phases where the fast sincos() does not hold (0, the multiples of pi/2,
beyond 2^30), against numpy."""
import numpy as np
import pytest

from sodecl_amd import sodecl_interface as si

pytestmark = pytest.mark.gpu

SOURCE = """
void sode_system(double t, double y[_numeq_], double yout[_numeq_], double p[_numpar_])
{ for (int i = 0; i < _numeq_; i++) yout[i] = 0; }
double sode_system_i(int i, double t, double y[_numeq_], double p[_numpar_]) { return 0; }
#ifdef SODECL_FIELD_API
#define SODE_FIELDS 1
#define SODE_FIELD_SHARED 1
#define SODE_FIELD_OWN 0
int sode_field_own_param(int i, int k) { return 0; }
void sode_field(int i, double t, double yi, double ps[], double po[], double phi[])
{
    double s, c;
    sincos(yi, &s, &c);
    phi[0] = FEATURE;
}
double sode_system_field(int i, double t, double yi, double ps[], double po[], double phi[], double sum[])
{ return ps[0] * sum[0]; }
#endif
"""
FEATURES = {"fmin(s, 0.5)": lambda s, c: np.minimum(s, 0.5), "c": lambda s, c: c,
            "s >= 0 ? 1.0 : -1.0": lambda s, c: np.where(s >= 0, 1.0, -1.0),
            "fmax(c, 0.25)": lambda s, c: np.maximum(c, 0.25)}


@pytest.mark.parametrize("feature", sorted(FEATURES))
@pytest.mark.parametrize("n,group", [(3, 0), (12, 0), (40, 64), (40, 4)])
def test_features_that_drop_nan(feature, n, group):
    special = np.array([0.0, -0.0, np.pi / 2, -np.pi / 2, np.pi, 3 * np.pi / 2, 2.0 ** 30 + 1.5, -1e12, 1e22, 1.0, 2.5])
    orbits = 50
    r = np.random.default_rng(n)
    y0 = r.choice(special, (orbits, n))
    y0[0] = 0.0
    p = r.uniform(0.5, 1.5, (orbits, 1))
    opts = dict(group_size=group, schedule="group") if group else {}
    s = si.Session(SOURCE.replace("FEATURE", feature), 1, orbits, n, 1, 0, 1.0, 1.0, 1, 0, opts, True)
    s.setup(y0, p)
    out = s.run().reshape(2, n, orbits)
    assert "#define SODECL_USE_FIELD 1" in s.program_source()
    total = FEATURES[feature](np.sin(y0), np.cos(y0)).sum(1)
    ref = y0 + p * total[:, None]
    # the sums' roundings (n of them, terms of at most 1) and the last addition's
    tol = 4e-16 * (1.5 * n * n + np.abs(ref))
    assert (np.abs(out[1].T - ref) <= tol).all()
