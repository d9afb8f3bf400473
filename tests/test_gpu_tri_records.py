"""GPU test: trilinear Widom runs that pack the corners of every cell give the bits of
runs that do not.

Grid sizes are at the edges of the packing's blocks (16 by 64), with enough insertions
that the rule packs them; the same run in a context whose cap leaves no room for the
packed corners takes the plain kernel.  Sampled energies equal the oracle's.
"""
import numpy as np
import pytest

from emptyroom_amd import api
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nins", [((2, 2, 2), 1_100_000), ((16, 65, 64), 1_300_000),
                                    ((17, 30, 66), 1_200_001), ((33, 40, 129), 1_700_000),
                                    ((64, 64, 64), 2_100_000), ((128, 97, 130), 3_300_000),
                                    ((129, 128, 130), 1_100_000)])
def test_packed_corners_and_plain(n, nins):
    print(f"tri records n={n} insertions={nins}", flush=True)
    rng = np.random.default_rng(sum(n))
    g = rng.uniform(-2000.0, 3000.0, n).astype(np.float32)
    g[rng.random(n) < 0.1] = 1e13
    f = api.lib()["_ZN2er15tri_faces_bytesEPKim"]
    f.restype, f.argtypes = api.ctypes.c_size_t, [api.ctypes.POINTER(api.ctypes.c_int),
                                                  api.ctypes.c_uint64]
    records = f((api.ctypes.c_int * 3)(*n), nins)
    assert records > 0
    seed, temp = 41, 298.0
    got = []
    # a context holds ~32 MiB itself; a run the energies, the partials and the grid
    room = (33 << 20) + (1 << 19) + 8 * nins + g.nbytes + (2 << 20)
    for cap in (0, room):
        with api.Context(0, hbm_cap=cap) as c:
            grid = api.Grid.upload(c, g)
            got.append(api.widom_grid(c, grid, nins, temp, seed, energies=True))
            assert api.widom_grid(c, grid, nins, temp, seed) == got[-1][:3]
            grid.close()
    assert got[0][:3] == got[1][:3] and np.array_equal(got[0][3], got[1][3])
    pick = np.concatenate([np.arange(100), rng.integers(0, nins, 1000), [nins - 1]])
    frac = np.array([api.widom_point(seed, 1, int(i)) for i in pick])
    assert np.array_equal(got[0][3][pick], oracle.trilinear_points(g.astype(np.float64), frac))
