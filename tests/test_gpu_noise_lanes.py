"""Lanes that draw an orbit's noise together (small Euler-Maruyama launches of
the lane schedule): in the strict arithmetic the bits of the reference's launch
design (one lane per orbit; the default arithmetic may contract a source's
sums differently in the two programs), in the default one the oracle at the
parity tolerance, counters exact in both."""
import numpy as np
import pytest

from sodecl_amd import configs, sodecl_interface as si
from oracle.oracle import Oracle
from tests.parity import assert_traj_close

pytestmark = pytest.mark.gpu


# (orbits, ksteps, block, lanes): step counts below and not a multiple of the
# lanes, a block that allows fewer lanes, orbits for eight, two and one
@pytest.mark.parametrize("orbits,ksteps,block,lanes", [(3, 3, 0, 16), (67, 7, 0, 16), (50, 50, 24, 8), (6000, 9, 0, 8),
                                                       (20001, 5, 0, 2), (40000, 4, 0, 1)])
@pytest.mark.parametrize("odd", [False, True])
def test_noise_lanes(orbits, ksteps, block, lanes, odd):
    cfg = configs.oculomotor_rk4(orbits=orbits, seed=orbits, dt=2e-6, tspan=2e-6 * 4 * ksteps, ksteps=ksteps)
    cfg["y0"][:, 5] += 1.0
    rng = np.random.default_rng(orbits)
    # a third, unused noise process makes the last call's second half idle
    nnoi = 3 if odd else 2
    params = np.concatenate([cfg["params"], rng.uniform(0, 0.2, (orbits, nnoi))], 1)
    counters = rng.integers(0, 10 ** 11, orbits).astype(np.float64)
    outs = []
    for schedule, strict in (("lane", 1), ("plain", 1), ("lane", 0)):
        s = si.Session(cfg["system"], 0, orbits, 6, 6 + nnoi, nnoi, cfg["dt"], cfg["tspan"], ksteps, 0,
                       dict(schedule=schedule, block_size=block, fp_contract=strict))
        s.setup(cfg["y0"], params, None, counters)
        src = s.program_source().split("#line")[0]
        assert (f"#define SODECL_NL {lanes}\n" in src) == (schedule == "lane" and lanes > 1)
        outs.append((s.run().copy(), s.run().copy(), s.counters()))
    for a, b in zip(outs[0], outs[1]):
        np.testing.assert_array_equal(a, b)
    k = min(orbits, 20)
    ref = Oracle("oculomotor").run("em", cfg["y0"], params, cfg["dt"], cfg["tspan"], ksteps, counters=counters,
                                   nnoi=nnoi, orbit_range=(0, k))
    assert_traj_close(outs[2][0].reshape(-1, 6, orbits)[:, :, :k], ref["out"], what="default arithmetic")
    calls = (nnoi + 1) // 2 * ref["launches"] * ksteps
    np.testing.assert_array_equal(outs[0][2], counters + 2 * calls)
    np.testing.assert_array_equal(outs[2][2], counters + 2 * calls)
