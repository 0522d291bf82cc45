"""A trajectory for host memory that streams in chunks against the same run in
one launch on device memory, around the size where streaming begins: the same
bits, whatever the chunks."""
import numpy as np
import pytest
import torch

import sodecl_amd
from sodecl_amd import sodecl_interface as si

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


# (solver, orbits, snapshots): 16 orbits' snapshot is 768 bytes; below and above
# the line, chunks of one snapshot with a rest, and many in a chunk
@pytest.mark.parametrize("solver,orbits,snaps", [(2, 16384, 8), (2, 16384, 9), (0, 30011, 7), (2, 700, 400)])
def test_streamed_run_matches_one_launch(solver, orbits, snaps):
    ks, dt = 2, 2.0 ** -19
    tspan = (snaps - 1) * ks * dt
    noise = 2 if solver == 0 else 0
    rng = np.random.default_rng(orbits)
    y0 = 1e-3 * rng.standard_normal((orbits, 6))
    y0[:, 5] += 1.0
    p = np.array([120.0, 1.5, 0.0045, 0.05, 600.0, 9.0]) * rng.uniform(0.8, 1.25, (orbits, 6))
    if noise:
        p = np.concatenate([p, rng.uniform(0.0, 0.2, (orbits, noise))], axis=1)
    counters = np.floor(rng.uniform(0, 1e11, orbits)) if noise else None
    s = si.Session(sodecl_amd.system_path("oculomotor"), solver, orbits, 6, p.shape[1], noise, dt, tspan, ks, 0, {})
    assert s.launches + 1 == snaps
    s.setup(y0, p, None, counters)
    got = s.run().reshape(snaps, 6, orbits)
    t = torch.zeros(orbits, dtype=torch.float64, device=DEV)
    y, q = torch.tensor(y0, device=DEV), torch.tensor(p, device=DEV)
    c = torch.tensor(counters, device=DEV) if noise else None
    out = torch.empty(snaps, 6, orbits, dtype=torch.float64, device=DEV)
    s.run_device(t.data_ptr(), y.data_ptr(), q.data_ptr(), c.data_ptr() if noise else 0, out.data_ptr(), 0)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(got.view(np.uint64), out.cpu().numpy().view(np.uint64))
