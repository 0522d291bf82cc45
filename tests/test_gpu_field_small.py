"""Systems of two to seven components in the field form, which the automatic
schedule takes where the lane schedule used to run: against the oracle, and
what keeps the lane schedule."""
import numpy as np
import pytest

from sodecl_amd import configs
from oracle.oracle import Oracle
from tests.parity import assert_traj_close

pytestmark = pytest.mark.gpu


# few and many orbits (one component per lane up to all on one), odd noise counts
@pytest.mark.parametrize("solver", [0, 1, 2])
@pytest.mark.parametrize("n,orbits", [(2, 67), (2, 70000), (3, 67), (3, 70000), (5, 9001), (7, 67), (7, 70000)])
def test_small_systems_vs_oracle(solver, n, orbits):
    if solver == 0:
        cfg = configs.kuramoto_em(orbits=orbits, n=n, seed=n, tspan=0.02, ksteps=10)
        cfg["counters"] = np.random.default_rng(n).integers(0, 2 ** 40, orbits).astype(np.float64)
    else:
        cfg = configs.kuramoto_rk4(orbits=orbits, n=n, seed=n, dt=0.01, tspan=0.2, ksteps=5)
        cfg["solver"] = solver
    s = configs.session_for(cfg)
    s.setup(cfg["y0"], cfg["params"], None, cfg.get("counters"))
    out = s.run().reshape(s.nsnap, n, orbits)
    assert s.launch_config()[0] == 1
    assert "#define SODECL_USE_FIELD 1" in s.program_source()
    some = np.unique(np.r_[0:40, orbits - 20:orbits])
    ref = Oracle("kuramoto").run({0: "em", 1: "euler", 2: "rk4"}[solver], cfg["y0"], cfg["params"], cfg["dt"],
                                 cfg["tspan"], cfg["ksteps"], counters=cfg.get("counters"), nnoi=cfg["nnoi"])
    assert_traj_close(out[:, :, some], ref["out"][:, :, some], what=f"solver {solver} N={n}")
    if solver == 0:
        np.testing.assert_array_equal(s.counters(), ref["counters"])


@pytest.mark.parametrize("opts", [dict(schedule="lane"), dict(schedule="plain"), dict(pairwise=-1), dict(fp_contract=1),
                                  dict(group_size=4), dict(block_size=64)])
def test_explicit_choices_keep_the_lane_schedule(opts):
    cfg = configs.kuramoto_rk4(orbits=50, n=5, seed=1, dt=0.01, tspan=0.1, ksteps=5)
    s = configs.session_for(cfg, **opts)
    s.setup(cfg["y0"], cfg["params"])
    out = s.run().reshape(s.nsnap, 5, 50)
    assert "#define SODECL_USE_FIELD 1" not in s.program_source()
    ref = Oracle("kuramoto").run("rk4", cfg["y0"], cfg["params"], cfg["dt"], cfg["tspan"], cfg["ksteps"])
    assert_traj_close(out, ref["out"], what=str(opts))


@pytest.mark.parametrize("solver", [0, 2])
def test_host_share_beside_the_field_form(solver):
    """The GPU's orbits of an automatic run have the bits of a run without host
    share; the host's, which the lane arithmetic integrates, match the oracle."""
    orbits, n = 200, 5
    if solver == 0:
        cfg = configs.kuramoto_em(orbits=orbits, n=n, seed=3, tspan=0.1, ksteps=10)
    else:
        cfg = configs.kuramoto_rk4(orbits=orbits, n=n, seed=3, dt=0.01, tspan=0.5, ksteps=5)
    out = []
    for share in (0.0, 0.3):
        s = configs.session_for(cfg, host_share=share)
        s.setup(cfg["y0"], cfg["params"], None, cfg.get("counters"))
        out.append(s.run().reshape(s.nsnap, n, orbits))
        assert "#define SODECL_USE_FIELD 1" in s.program_source()
    assert s.host_stats()[1] == 60
    np.testing.assert_array_equal(out[0][:, :, :140], out[1][:, :, :140])
    ref = Oracle("kuramoto").run({0: "em", 2: "rk4"}[solver], cfg["y0"], cfg["params"], cfg["dt"], cfg["tspan"],
                                 cfg["ksteps"], counters=cfg.get("counters"), nnoi=cfg["nnoi"])
    assert_traj_close(out[1], ref["out"], what="host share")
    if solver == 0:
        np.testing.assert_array_equal(s.counters(), ref["counters"])
