"""GPU parity of grids of 321 to 512 tiles, which give a tile one workgroup of eight
waves, two for each quarter of its points.

Point counts lie at both limits, with edge tiles that leave one, two or three of
their quarters without a point, cells whose points share y and z and rotated ones,
and lists of several passes.  The grids are compared with the reference's direct
method on the GPU (bit-identical to the oracle): FP64 1e-9 relative, FP32 1e-3 K
where E < 1e4 K and 1e-6 relative above.  A batch gives the plain path's bits.
"""
import numpy as np
import pytest

from emptyroom_amd import api, synth
pytestmark = pytest.mark.gpu

CELL = (12.0, 11.0, 13.0, 80.0, 100.0, 95.0)
FLT_MAX = float(np.finfo(np.float32).max)


@pytest.fixture(scope="module")
def mctx():
    c = api.Context(0)
    yield c
    c.close()


def make(n_atoms, rotated=False):
    f = synth.small_framework(37, n_atoms=n_atoms, cell=CELL)
    t = f.t
    if rotated:
        q, _ = np.linalg.qr(np.random.default_rng(4).normal(size=(3, 3)))
        t = q @ f.t
    return f, t, f.particles()


@pytest.mark.parametrize("n,atoms,rotated", [
    ((64, 64, 48), 30, False),        # 384 cells
    ((49, 52, 53), 30, False),        # 343, edges of 1, 4 and 5 points
    ((57, 57, 57), 30, True),         # 512, edges of one point
    ((64, 64, 64), 20, True),         # 512
    ((24, 856, 8), 12, False),        # 321
    ((56, 55, 54), 700, False),       # several passes
    ((50, 51, 49), 0, False),
    ((64, 64, 65), 20, False),        # 576: one workgroup of four waves
])
def test_mid_grids(mctx, n, atoms, rotated):
    print(f"mid grid n={n} atoms={atoms} rotated={rotated}", flush=True)
    f, t, a = make(atoms, rotated)
    args = (a[:, :3], a[:, 3], a[:, 4], t, f.rep, f.rc2)
    fw = api.Framework(mctx, *args)
    ref = api.direct_grid(mctx, *args, n) if atoms else np.zeros(n)
    g64 = api.compute_grid(mctx, fw, n, api.ER_FP64)
    assert np.max(np.abs(g64 - ref) / np.maximum(1.0, np.abs(ref))) < 1e-9
    g32 = api.compute_grid(mctx, fw, n, api.ER_FP32).astype(np.float64)
    low = ref < 1e4
    assert np.max(np.abs(g32[low] - ref[low]), initial=0.0) <= 1e-3
    high = np.minimum(ref[~low], FLT_MAX)
    assert np.all(np.abs(g32[~low] - high) <= 1e-6 * high)
    fw.close()


def test_batch(mctx):
    print("mid batch", flush=True)
    f, t, a = make(60)
    fw = api.Framework(mctx, a[:, :3], a[:, 3], a[:, 4], t, f.rep, f.rc2)
    dims = [(57, 64, 60), (9, 9, 9), (50, 52, 54), (70, 70, 70), (49, 49, 49)]
    tasks = [dict(fw=fw, grid_n=n, precision=k % 2, n_insertions=170000, seed=k,
                  temperature=300.0) for k, n in enumerate(dims)]
    for graph in (False, True):
        b = api.Batch(mctx, tasks, use_graph=graph)
        for _ in range(3):
            b.run()
            b.wait()
        for k, n in enumerate(dims):
            assert np.array_equal(b.grid(k), api.compute_grid(mctx, fw, n, k % 2))
            assert b.widom(k) == api.widom(mctx, fw, 170000, 300.0, k)
        b.close()
    fw.close()
