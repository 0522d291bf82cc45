"""Small Euler-Maruyama launches of the lane schedule: the lanes of an orbit call
a plugin's team entry point in teams of two, however many draw the noise."""
import numpy as np
import pytest

from sodecl_amd import sodecl_interface as si

pytestmark = pytest.mark.gpu

# the team entry point of a source written for pairs: each lane adds up half of
# eight terms
SOURCE = """
double term(int k, double y[_numeq_], double p[_numpar_]) { return p[0] * y[k & 1] / (k + 2); }
void sode_system(double t, double y[_numeq_], double yout[_numeq_], double p[_numpar_])
{
    double lo = 0, hi = 0;
    for (int k = 0; k < 4; k++) { lo += term(k, y, p); hi += term(k + 4, y, p); }
    yout[0] = -(lo + hi);
    yout[1] = lo - hi;
}
#ifdef SODECL_TEAM_API
void sode_system_team(double t, double y[_numeq_], double yout[_numeq_], double p[_numpar_])
{
    const int odd = sodecl_lane() == 1;
    double mine = 0;
    for (int k = 0; k < 8 / sodecl_group_size(); k++) mine += term(odd ? k + 4 : k, y, p);
    const double other = sodecl_group_xor(mine, 1);
    yout[0] = -(odd ? other + mine : mine + other);
    yout[1] = odd ? other - mine : mine - other;
}
#endif
void sode_system_stoch(double t, double y[_numeq_], double st[_numeq_], double p[_numpar_], double noise[_numnoi_])
{ st[0] = p[1] * noise[0]; st[1] = 0; }
"""


@pytest.mark.parametrize("orbits", [5, 3000, 9000, 30000])
def test_teams_of_two(orbits):
    r = np.random.default_rng(orbits)
    y0, p = r.normal(size=(orbits, 2)), r.uniform(0.5, 1.5, (orbits, 2))
    counters = r.integers(0, 10 ** 11, orbits).astype(np.float64)
    outs = []
    for schedule in ("lane", "plain"):
        s = si.Session(SOURCE, 0, orbits, 2, 2, 1, 1e-3, 0.06, 20, 0, dict(schedule=schedule, fp_contract=1), True)
        s.setup(y0, p, None, counters)
        assert ("#define SODECL_NOISE_TEAM 1" in s.program_source()) == (schedule == "lane")
        outs.append(s.run().copy())
    np.testing.assert_array_equal(outs[0], outs[1])
