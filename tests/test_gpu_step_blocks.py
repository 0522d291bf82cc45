"""Segments whose length is not a multiple of the steps per block of the lane
and team schedules' step loops, and checkpoints inside them, against the
oracle: 1e-10 of each component's scale."""
import numpy as np
import pytest

from sodecl_amd import configs, sodecl_interface as si
from oracle.oracle import Oracle
from tests.parity import assert_traj_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ksteps", [7, 8, 9, 10, 11, 13])
@pytest.mark.parametrize("solver,schedule", [(0, "lane"), (1, "lane"), (2, "lane"), (2, "team")])
def test_segment_remainders(solver, schedule, ksteps):
    orbits, dt, segments = 130, 2.0 ** -19, 5
    tspan = segments * ksteps * dt
    cfg = configs.oculomotor_rk4(orbits=orbits, seed=ksteps, dt=dt, tspan=tspan, ksteps=ksteps)
    cfg["y0"][:, 5] += 1.0
    params, nnoi, counters = cfg["params"], 0, None
    if solver == 0:
        rng = np.random.default_rng(ksteps)
        nnoi = 2
        params = np.concatenate([params, rng.uniform(0, 0.2, (orbits, nnoi))], 1)
        counters = rng.integers(0, 10 ** 11, orbits).astype(np.float64)
    s = si.Session(cfg["system"], solver, orbits, 6, params.shape[1], nnoi, dt, tspan, ksteps, 0,
                   dict(schedule=schedule))
    s.setup(cfg["y0"], params, None, counters)
    out = s.run().reshape(s.nsnap, 6, orbits)
    assert ("#define SODECL_ONE_WAVE 1" in s.program_source())
    ref = Oracle("oculomotor").run({0: "em", 1: "euler", 2: "rk4"}[solver], cfg["y0"], params, dt, tspan, ksteps,
                                   counters=counters, nnoi=nnoi)
    assert_traj_close(out, ref["out"], what=f"solver {solver} {schedule} ksteps {ksteps}")
    if solver == 0:
        np.testing.assert_array_equal(s.counters(), ref["counters"])


@pytest.mark.parametrize("ksteps", [3, 4, 7, 9])
def test_field_segment_remainders(ksteps):
    """The field form's Euler steps with one component per lane."""
    orbits, n, dt = 67, 10, 2.0 ** -7
    tspan = 5 * ksteps * dt
    cfg = configs.kuramoto_rk4(orbits=orbits, n=n, seed=ksteps, dt=dt, tspan=tspan, ksteps=ksteps)
    s = si.Session(cfg["system"], 1, orbits, n, n + 1, 0, dt, tspan, ksteps, 0, {})
    s.setup(cfg["y0"], cfg["params"])
    out = s.run().reshape(s.nsnap, n, orbits)
    assert "#define SODECL_FL 16\n#define SODECL_FC 1\n" in s.program_source()
    ref = Oracle("kuramoto").run("euler", cfg["y0"], cfg["params"], dt, tspan, ksteps)
    assert_traj_close(out, ref["out"], what=f"field Euler ksteps {ksteps}")
