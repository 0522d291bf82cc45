"""Euler-Maruyama counters that are no whole numbers, or reach 2^53 during a run:
the reference adds 1 per Threefry call, so a counter sticks at 2^53 and a
fraction rounds call by call.  Noise and final counters as in the oracle."""
import numpy as np
import pytest

from sodecl_amd import configs, sodecl_interface as si
from oracle.oracle import Oracle
from tests.parity import assert_traj_close

pytestmark = pytest.mark.gpu

EDGE = [2.0 ** 53 - 70, 2.0 ** 53 - 1, 2.0 ** 53, 2.0 ** 53 + 2, 2.0 ** 60, 0.7, 1.0 - 2.0 ** -53, 2.0 ** 50 + 0.375, 2.0 ** 52 - 40.5,
        -3.0, 17.0]


def counters(orbits, edge):
    c = np.random.default_rng(orbits).integers(0, 10 ** 11, orbits).astype(np.float64)
    if edge:
        c[:len(EDGE)] = EDGE
    else:
        c[7] = 2.0 ** 53 - 64 * 30   # whole and below 2^53 to the end
    return c


@pytest.mark.parametrize("edge", [True, False])
@pytest.mark.parametrize("orbits,ksteps", [(40, 13), (3000, 20), (20000, 7)])
def test_lane_schedule(orbits, ksteps, edge):
    cfg = configs.oculomotor_rk4(orbits=orbits, seed=orbits, dt=2e-6, tspan=2e-6 * 3 * ksteps, ksteps=ksteps)
    cfg["y0"][:, 5] += 1.0
    nnoi, k = 3, 40
    params = np.concatenate([cfg["params"], np.random.default_rng(3).uniform(0, 0.2, (orbits, nnoi))], 1)
    cnt = counters(orbits, edge)
    s = si.Session(cfg["system"], 0, orbits, 6, 6 + nnoi, nnoi, cfg["dt"], cfg["tspan"], ksteps, 0, {})
    s.setup(cfg["y0"], params, None, cnt)
    out = s.run().reshape(-1, 6, orbits)
    ref = Oracle("oculomotor").run("em", cfg["y0"], params, cfg["dt"], cfg["tspan"], ksteps, counters=cnt, nnoi=nnoi,
                                   orbit_range=(0, k))
    assert_traj_close(out[:, :, :k], ref["out"])
    np.testing.assert_array_equal(s.counters()[:k], ref["counters"][:k])


@pytest.mark.parametrize("edge", [True, False])
@pytest.mark.parametrize("n,group", [(3, 0), (5, 0), (12, 16), (33, 64), (32, 8), (33, 4)])
def test_field_form(n, group, edge):
    orbits = 40
    cfg = configs.kuramoto_em(orbits=orbits, n=n, seed=n, tspan=0.021, ksteps=7)
    cfg["counters"] = counters(orbits, edge)
    s = configs.session_for(cfg, **(dict(schedule="group", group_size=group) if group else {}))
    s.setup(cfg["y0"], cfg["params"], None, cfg["counters"])
    out = s.run().reshape(-1, n, orbits)
    assert "#define SODECL_USE_FIELD 1" in s.program_source()
    ref = Oracle("kuramoto").run("em", cfg["y0"], cfg["params"], cfg["dt"], cfg["tspan"], cfg["ksteps"],
                                 counters=cfg["counters"], nnoi=n)
    assert_traj_close(out, ref["out"])
    np.testing.assert_array_equal(s.counters(), ref["counters"])
