"""The sampler at the edges of its row tiles and column chunks against its
CPU restatement: uniform columns bit for bit, the others to the few ulps the
sampler is held to, neighbouring memory untouched."""
import numpy as np
import pytest
import torch

from sodecl_amd.sampling import sample, table
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 1), (63, 1), (64, 16), (65, 3), (1025, 1), (130, 120), (129, 121), (70, 245),
                                       (150000, 2)])
def test_sampler_tile_edges(rows, cols):
    kinds = [("normal", 0.3, 1.7), ("uniform", -1.0, 2.0), ("log_uniform", 0.2, 0.9), ("constant", 4.5)]
    dists = [kinds[(c * 7 + cols) % 4] for c in range(cols)]
    whole = torch.full((rows * cols + 16,), -7.0, dtype=torch.float64, device="cuda:0")
    out = whole[:rows * cols].view(rows, cols)
    got = sample(dists, rows, 12345, out=out).cpu().numpy()
    ref = Oracle("oculomotor").sample(table(dists), rows, 12345)
    for c, d in enumerate(dists):
        if d[0] in ("uniform", "constant"):
            np.testing.assert_array_equal(got[:, c], ref[:, c])
        else:
            np.testing.assert_allclose(got[:, c], ref[:, c], rtol=0, atol=64e-16 * max(abs(d[1]), abs(d[2])))
    assert (whole[rows * cols:] == -7.0).all()


@pytest.mark.parametrize("rows,cols", [(20000, 17), (40000, 61), (65473, 64), (65472, 65), (66000, 5)])
def test_sampler_column_splits(rows, cols):
    """Tables on either side of the size up to which columns spread over
    blocks, with columns that do not come out even, and of each chunk's width:
    the uniform columns bit for bit."""
    dists = [("uniform", float(c), c + 2.0) if c % 3 else ("constant", float(c)) for c in range(cols)]
    got = sample(dists, rows, 77).cpu().numpy()
    np.testing.assert_array_equal(got, Oracle("oculomotor").sample(table(dists), rows, 77))
