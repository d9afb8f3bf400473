"""GPU test of the far field of fine FP32 grids, which blocks of 2 x 2 x 2 tiles
take from Chebyshev nodes.

The path is chosen for grids of at least 1024 blocks of 16 x 16 x 16 points with
enough far atoms, so the grids here have 4-6 million points and are compared
with the reference's direct method on the GPU (bit-identical to the oracle):
1e-3 K where |E| < 1e4 K and 1e-6 relative beyond, as for every FP32 grid (the
interpolation itself is good to ~2e-5 K).  Point counts put one, three, eight,
nine and sixteen points into the last block of an axis, and an odd number of
tiles along it; cells are right-angled and triclinic; one framework has 40 pair
types.  Batch, server and the call without allocation give the same bits.
"""
import ctypes

import numpy as np
import pytest

from emptyroom_amd import api, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nctx():
    c = api.Context(0)
    yield c
    c.close()


def framework(seed, n_atoms, cell, ntypes=6, cluster=0):
    f = synth.small_framework(seed, n_atoms=n_atoms, cell=cell, ntypes=ntypes)
    if cluster:
        rng = synth.Rng(seed + 1)
        f.frac[:cluster] = 0.5 + 0.04 * (rng.uniform(3 * cluster).reshape(cluster, 3) - 0.5)
    return f


def check(g, ref):
    low = np.abs(ref) < 1e4
    assert low.any()
    assert np.max(np.abs(g[low] - ref[low])) <= 1e-3
    rel = np.abs(g[~low] - np.minimum(ref[~low], float(np.finfo(np.float32).max)))
    assert np.all(rel <= 1e-6 * np.abs(np.minimum(ref[~low], float(np.finfo(np.float32).max))))


@pytest.mark.parametrize("n,cell,atoms,ntypes", [
    ((161, 163, 168), (16.0, 16.2, 16.7, 90.0, 90.0, 90.0), 330, 6),
    ((169, 176, 161), (17.0, 17.6, 16.1, 84.0, 97.0, 105.0), 400, 6),
    ((177, 164, 165), (17.7, 16.5, 16.4, 90.0, 101.0, 90.0), 480, 40),
])
def test_fine_grid_against_direct(nctx, n, cell, atoms, ntypes):
    print(f"nodes n={n} cell={cell} atoms={atoms} types={ntypes}", flush=True)
    f = framework(61, atoms, cell, ntypes)
    a = f.particles()
    fw = api.Framework(nctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
    g = api.compute_grid(nctx, fw, n, api.ER_FP32)
    ref = api.direct_grid(nctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2, n)
    check(g.astype(np.float64), ref)
    fw.close()


def test_lists_that_overflow(nctx):
    """2500 atoms in a ball of 0.3 A: regions and blocks near it overflow their
    lists and fall back to direct tiles.  Its field is -3e4 K deep and nearly all
    of it comes from one place, so the FP32 rounding of the pairs (a few ulp,
    4e-7) is common to them: 1e-6 of 1e4 K instead of the usual 1e-3 K."""
    n, cell = (170, 163, 164), (17.0, 16.3, 16.4, 90.0, 95.0, 90.0)
    print("nodes overflow", flush=True)
    f = framework(61, 2600, cell, 4, 2500)
    a = f.particles()
    fw = api.Framework(nctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
    g = api.compute_grid(nctx, fw, n, api.ER_FP32).astype(np.float64)
    ref = np.minimum(api.direct_grid(nctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2, n),
                     float(np.finfo(np.float32).max))
    assert np.all(np.abs(g - ref) <= 1e-6 * np.maximum(np.abs(ref), 1e4))
    fw.close()


def test_same_bits_on_every_path(nctx):
    print("nodes paths", flush=True)
    n, cell = (165, 161, 176), (16.5, 16.1, 17.6, 80.0, 95.0, 100.0)
    f = framework(62, 420, cell)
    a = f.particles()
    fw = api.Framework(nctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
    g = api.compute_grid(nctx, fw, n, api.ER_FP32)
    h = ctypes.CDLL("libamdhip64.so.7", mode=ctypes.RTLD_GLOBAL)  # the library's own runtime
    h.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    out, buf = np.empty_like(g), ctypes.c_void_p()
    assert h.hipMalloc(ctypes.byref(buf), ctypes.c_size_t(out.nbytes)) == 0
    assert api.lib().er_grid_compute_noalloc(nctx.h, fw.h, (ctypes.c_int * 3)(*n), api.ER_FP32,
                                             buf) == 0
    assert h.hipMemcpy(out.ctypes.data, buf, out.nbytes, 2) == 0
    assert h.hipFree(buf) == 0
    assert np.array_equal(out, g)
    small = (21, 22, 23)
    tasks = [dict(fw=fw, grid_n=small), dict(fw=fw, grid_n=n, n_insertions=5000),
             dict(fw=fw, grid_n=small, precision=api.ER_FP64)]
    for graph in (False, True):
        b = api.Batch(nctx, tasks, use_graph=graph)
        for _ in range(3):
            b.run()
            b.wait()
        assert np.array_equal(b.grid(1), g)
        assert np.array_equal(b.grid(0), api.compute_grid(nctx, fw, small, api.ER_FP32))
        assert np.array_equal(b.grid(2), api.compute_grid(nctx, fw, small, api.ER_FP64))
        b.close()
    with api.Context(0) as c:
        s = api.Server(c)
        args = (a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
        tickets = [s.submit(*args, grid_n=k)[1] for k in (n, small)]
        for t, k in zip(tickets, (n, small)):
            assert s.poll(t, -1.0).state == api.RQ_DONE
            assert np.array_equal(s.fetch_grid(t, k), api.compute_grid(nctx, fw, k, api.ER_FP32))
        s.close()
    fw.close()
