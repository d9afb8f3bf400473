"""GPU parity of small jobs, whose cells (grid tiles, Widom bins) are shared out
to four workgroups of eight waves (up to 128 cells) or of four (up to 320).

Point counts are at the edges of tiles, of a part's quadrant and of the two
limits, with cells whose points share y and z and rotated ones, no atoms at all,
and lists of several passes; bins hold less and more than the 512 insertions of
one round.  Tolerances as for every grid and Widom test: FP64 grid 1e-9
relative, FP32 grid 1e-3 K where E < 1e4 K and 1e-6 relative above, energies
1e-3 K.  A batch of small and large jobs gives the plain path's bits.
"""
import numpy as np
import pytest

from emptyroom_amd import api, synth
from oracle import oracle

pytestmark = pytest.mark.gpu

CELL = (12.0, 11.0, 13.0, 80.0, 100.0, 95.0)
FLT_MAX = float(np.finfo(np.float32).max)


@pytest.fixture(scope="module")
def sctx():
    c = api.Context(0)
    yield c
    c.close()


def make(n_atoms, rotated=False, seed=31):
    f = synth.small_framework(seed, n_atoms=n_atoms, cell=CELL)
    t = f.t
    if rotated:
        q, _ = np.linalg.qr(np.random.default_rng(2).normal(size=(3, 3)))
        t = q @ f.t
    return f, t, f.particles()


@pytest.mark.parametrize("n,atoms,rotated", [
    ((2, 2, 2), 30, False), ((8, 8, 8), 30, True), ((9, 5, 12), 30, False),
    ((17, 4, 23), 30, True), ((40, 39, 33), 30, False), ((32, 32, 64), 20, False),
    ((33, 32, 64), 20, True), ((32, 64, 80), 12, False), ((33, 64, 80), 12, False),
    ((12, 13, 20), 700, False), ((10, 9, 8), 0, False),
])
def test_small_grids(sctx, n, atoms, rotated):
    print(f"small grid n={n} atoms={atoms} rotated={rotated}", flush=True)
    f, t, a = make(atoms, rotated)
    fw = api.Framework(sctx, a[:, :3], a[:, 3], a[:, 4], t, f.rep, f.rc2)
    ref = oracle.lj_grid(t, a, f.rep, f.rc2, n)
    g64 = api.compute_grid(sctx, fw, n, api.ER_FP64)
    assert np.max(np.abs(g64 - ref) / np.maximum(1.0, np.abs(ref))) < 1e-9
    g32 = api.compute_grid(sctx, fw, n, api.ER_FP32).astype(np.float64)
    low = ref < 1e4
    assert np.max(np.abs(g32[low] - ref[low]), initial=0.0) <= 1e-3
    high = np.minimum(ref[~low], FLT_MAX)
    assert np.all(np.abs(g32[~low] - high) <= 1e-6 * high)
    fw.close()


@pytest.mark.parametrize("nins,per_bin,atoms", [(1, 480, 30), (700, 480, 30), (61000, 480, 30),
                                                (62500, 480, 30), (30000, 4000, 30),
                                                (3000, 30, 700), (5000, 16, 30)])
def test_small_widom(sctx, nins, per_bin, atoms):
    print(f"small widom n={nins} per_bin={per_bin} atoms={atoms}", flush=True)
    f, t, a = make(atoms)
    tu = sctx.tuning
    tu.widom_per_bin = per_bin
    sctx.tuning = tu
    try:
        fw = api.Framework(sctx, a[:, :3], a[:, 3], a[:, 4], t, f.rep, f.rc2)
        sb, seb, n, e = api.widom(sctx, fw, nins, 300.0, 9, energies=True)
        sums = api.widom(sctx, fw, nins, 300.0, 9)
        fw.close()
    finally:
        tu.widom_per_bin = 480
        sctx.tuning = tu
    rb, reb, re = oracle.widom(t, a, f.rep, f.rc2, 300.0, 9, 0, nins, energies=True)
    low = re < 1e4
    assert np.max(np.abs(e[low] - re[low]), initial=0.0) <= 1e-3
    assert np.all(np.abs(e[~low] - re[~low]) <= 1e-6 * re[~low])
    assert sums == (sb, seb, n)  # an insertion that stops early adds the same 0
    assert abs(sb - rb) <= 1e-4 * rb


def test_batch_of_small_and_large(sctx):
    print("small batch", flush=True)
    f, t, a = make(60)
    fw = api.Framework(sctx, a[:, :3], a[:, 3], a[:, 4], t, f.rep, f.rc2)
    dims = [(9, 9, 9), (48, 48, 48), (70, 70, 70), (20, 10, 30), (60, 40, 50)]
    tasks = [dict(fw=fw, grid_n=n, precision=k % 2, n_insertions=10 ** (k + 2), seed=k,
                  temperature=300.0) for k, n in enumerate(dims)]
    for graph in (False, True):
        b = api.Batch(sctx, tasks, use_graph=graph)
        for _ in range(3):
            b.run()
            b.wait()
        for k, n in enumerate(dims):
            assert np.array_equal(b.grid(k), api.compute_grid(sctx, fw, n, k % 2))
            assert b.widom(k) == api.widom(sctx, fw, 10 ** (k + 2), 300.0, k)
        b.close()
    fw.close()
