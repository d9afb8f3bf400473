"""GPU test of the grid-interpolated Widom path that packs the corners of every
cell side by side (1e6 insertions and more): energies equal the oracle's
trilinear interpolation bit for bit at sampled insertions, on grids whose sizes
are at the edges of the packing's blocks (16 by 64) and on either side of the
size rule, with blocked 1e13 K nodes; the sums are those of the energies."""
import numpy as np
import pytest

from emptyroom_amd import api
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(2, 2, 2), (16, 65, 64), (17, 30, 66), (33, 40, 129), (64, 64, 64),
                               (65, 64, 64), (110, 110, 108), (128, 97, 130)])
def test_packed_corners(ctx, n):
    print(f"tri faces n={n}", flush=True)
    rng = np.random.default_rng(sum(n))
    g = rng.uniform(-2000.0, 3000.0, n).astype(np.float32)
    g[rng.random(n) < 0.1] = 1e13
    grid = api.Grid.upload(ctx, g)
    nins, seed, temp = 1_000_000, 41, 298.0
    sb, seb, m, e = api.widom_grid(ctx, grid, nins, temp, seed, energies=True)
    grid.close()
    assert m == nins
    pick = np.concatenate([np.arange(200), rng.integers(0, nins, 2000), [nins - 1]])
    frac = np.array([api.widom_point(seed, 1, int(i)) for i in pick])
    assert np.array_equal(e[pick], oracle.trilinear_points(g.astype(np.float64), frac))
    b = np.exp(-e / temp)
    assert abs(sb - b.sum()) <= 1e-12 * b.sum()
    eb = np.where(b == 0, 0.0, e * b)
    assert abs(seb - eb.sum()) <= 1e-12 * np.abs(eb).sum()
