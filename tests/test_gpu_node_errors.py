"""GPU test: the far field from nodes brings fine FP32 grids no further off the
direct FP64 sums than direct tiles are.

The same grid is computed in the default tile (nodes) and in tiles of another shape
(no nodes).  The nodes' FP64 sums replace the FP32 rounding of about half the pairs
by an interpolation error a tenth as large, so where that rounding is what is seen
(|E| < 1000 K) the rms error must be below 0.9 of the direct tiles', and nowhere
above it.
"""
import numpy as np
import pytest

from emptyroom_amd import api, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("atoms,cell,ntypes", [(300, (16.5, 16.1, 17.6, 80.0, 95.0, 100.0), 6),
                                               (450, (17.0, 16.2, 16.4, 90.0, 90.0, 90.0), 3)])
def test_errors_beside_direct_tiles(atoms, cell, ntypes):
    print(f"node errors atoms={atoms} cell={cell}", flush=True)
    n = [int(10 * x) for x in cell[:3]]
    f = synth.small_framework(62, n_atoms=atoms, cell=cell, ntypes=ntypes)
    f.frac[:, 0] *= 0.55  # a channel: points of low energy
    a = f.particles()
    args = (a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
    grids = []
    with api.Context(0) as c:
        for tile in ((8, 8, 8), (4, 8, 16)):
            tu = api.default_tuning()
            tu.tile[0], tu.tile[1], tu.tile[2] = tile
            c.tuning = tu
            fw = api.Framework(c, *args)
            grids.append(api.compute_grid(c, fw, n, api.ER_FP32).astype(np.float64))
            fw.close()
        ref = api.direct_grid(c, *args, n)
    for most, bound in ((1e3, 0.9), (1e4, 1.0)):
        m = np.abs(ref) < most
        assert m.sum() > 1000
        rms = [np.sqrt(np.mean((g[m] - ref[m]) ** 2)) for g in grids]
        print(f"|E| < {most:g}: nodes {rms[0]:.3e}, direct tiles {rms[1]:.3e}", flush=True)
        assert rms[0] <= bound * rms[1]
