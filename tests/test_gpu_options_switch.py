"""Options changed on a live session: every run afterwards is the run of a fresh
session with those options, whichever programs the session holds already (two
option sets may agree in schedule, group and block size and still need
different kernels)."""
import numpy as np
import pytest
import torch

from sodecl_amd import configs, sodecl_interface as si

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def oculomotor_em(orbits):
    cfg = configs.oculomotor_rk4(orbits=orbits, seed=orbits, dt=2e-6, tspan=2e-6 * 40, ksteps=10)
    cfg["y0"][:, 5] += 1.0
    rng = np.random.default_rng(orbits)
    cfg.update(solver=0, nnoi=2, npar=8, params=np.concatenate([cfg["params"], rng.uniform(0, 0.2, (orbits, 2))], 1),
               counters=rng.integers(0, 10 ** 11, orbits).astype(np.float64))
    return cfg


def kuramoto(orbits, n):
    return configs.kuramoto_rk4(orbits=orbits, n=n, seed=n, dt=0.01, tspan=0.1, ksteps=5)


OFF = dict(schedule="auto", group_size=0, block_size=0)
CASES = [(oculomotor_em(5000), dict(), dict(schedule="plain")),
         (oculomotor_em(300), dict(schedule="lane"), dict(schedule="plain")),
         (kuramoto(16384, 64), dict(group_size=64), dict()),
         (kuramoto(700, 33), dict(group_size=64, block_size=256), dict()),
         (kuramoto(300, 5), dict(), dict(schedule="lane")),
         (kuramoto(300, 5), dict(), dict(schedule="plain"))]


def session(cfg, opts):
    return si.Session(cfg["system"], cfg["solver"], cfg["orbits"], cfg["neq"], cfg["npar"], cfg["nnoi"], cfg["dt"],
                      cfg["tspan"], cfg["ksteps"], 0, opts)


@pytest.mark.parametrize("forward", [True, False])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_switched_run_equals_a_fresh_one(case, forward):
    cfg, a, b = CASES[case]
    order = (a, b, a) if forward else (b, a, b)
    live = session(cfg, order[0])
    live.setup(cfg["y0"], cfg["params"], None, cfg.get("counters"))
    y0, p = torch.tensor(cfg["y0"], device=DEV), torch.tensor(cfg["params"], device=DEV)

    def device_run(s):
        y, t = y0.clone(), torch.zeros(cfg["orbits"], dtype=torch.float64, device=DEV)
        cnt = torch.tensor(cfg["counters"], device=DEV) if cfg["solver"] == 0 else None
        traj = torch.full((s.nsnap, cfg["neq"], cfg["orbits"]), float("nan"), dtype=torch.float64, device=DEV)
        s.run_device(t.data_ptr(), y.data_ptr(), p.data_ptr(), 0 if cnt is None else cnt.data_ptr(), traj.data_ptr(), 0)
        torch.cuda.synchronize()
        return [v.cpu().numpy() for v in (y, t, traj) + (() if cnt is None else (cnt,))]

    for k, opts in enumerate(order):
        live.set_options(dict(OFF, **opts))
        fresh = session(cfg, opts)
        fresh.setup(cfg["y0"], cfg["params"], None, cfg.get("counters"))
        for one, other in zip(device_run(live), device_run(fresh)):
            np.testing.assert_array_equal(one, other, err_msg=f"{opts}, switch {k}")
        assert not np.isnan(device_run(live)[2]).any()


def test_switched_adjoint_equals_a_fresh_one():
    cfg = kuramoto(4100, 64)
    a, b = dict(schedule="group", group_size=64), dict(schedule="group", group_size=0)

    def gradients(s):
        every = s.default_checkpoint_interval()
        n, o = cfg["neq"], cfg["orbits"]
        y, p = torch.tensor(cfg["y0"], device=DEV), torch.tensor(cfg["params"], device=DEV)
        full = lambda *shape: torch.full(shape, float("nan"), dtype=torch.float64, device=DEV)
        t, traj = torch.zeros(o, dtype=torch.float64, device=DEV), full(s.nsnap, n, o)
        k = s.checkpoint_count(every)
        ck_t, ck_y, gy, gp = full(k, o), full(k, n, o), full(o, n), full(o, n + 1)
        work, cot = full(s.adjoint_workspace_size(every)), torch.ones_like(traj)
        s.run_device_checkpointed(t.data_ptr(), y.data_ptr(), p.data_ptr(), 0, traj.data_ptr(), ck_t.data_ptr(),
                                  ck_y.data_ptr(), every, 0)
        s.adjoint_device(ck_t.data_ptr(), ck_y.data_ptr(), p.data_ptr(), cot.data_ptr(), gy.data_ptr(), gp.data_ptr(),
                         work.data_ptr(), every, 0)
        torch.cuda.synchronize()
        assert not (gy.isnan().any() or gp.isnan().any())
        return gy.cpu().numpy(), gp.cpu().numpy()

    live = session(cfg, a)
    live.setup(cfg["y0"], cfg["params"])
    for opts in (a, b, a):
        live.set_options(opts)
        fresh = session(cfg, opts)
        fresh.setup(cfg["y0"], cfg["params"])
        for one, other in zip(gradients(live), gradients(fresh)):
            np.testing.assert_array_equal(one, other, err_msg=str(opts))


def test_graph_recorded_for_other_options_is_not_replayed():
    cfg = oculomotor_em(300)
    kw = dict(segments_per_launch=1, use_graph=1)
    live = session(cfg, dict(kw, schedule="lane"))
    live.setup(cfg["y0"], cfg["params"], None, cfg["counters"])
    y0, p = torch.tensor(cfg["y0"], device=DEV), torch.tensor(cfg["params"], device=DEV)
    y, t, cnt = torch.empty_like(y0), torch.empty(300, dtype=torch.float64, device=DEV), torch.tensor(cfg["counters"],
                                                                                                    device=DEV)
    traj = torch.empty(live.nsnap, 6, 300, dtype=torch.float64, device=DEV)
    for schedule in ("lane", "plain", "lane"):
        live.set_options(dict(kw, schedule=schedule))
        fresh = session(cfg, dict(schedule=schedule, segments_per_launch=1))
        fresh.setup(cfg["y0"], cfg["params"], None, cfg["counters"])
        outs = []
        for s in (live, fresh, live):   # the live session's second run replays
            y.copy_(y0)
            t.zero_()
            cnt.copy_(torch.tensor(cfg["counters"], device=DEV))
            traj.fill_(float("nan"))
            s.run_device(t.data_ptr(), y.data_ptr(), p.data_ptr(), cnt.data_ptr(), traj.data_ptr(), 0)
            torch.cuda.synchronize()
            outs.append(traj.cpu().numpy().copy())
        np.testing.assert_array_equal(outs[0], outs[2], err_msg=schedule)
        np.testing.assert_array_equal(outs[0], outs[1], err_msg=schedule)
