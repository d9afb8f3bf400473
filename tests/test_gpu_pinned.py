"""GPU test of results that kernels write to pinned host memory: trilinear energies
of up to 98304 positions and grids of up to 128 KiB that stay on the host.  On either
side of the limits they are the bits of the calls that copy: the same positions in
one large call, the same grid kept on the device and downloaded.
"""
import numpy as np
import pytest

from emptyroom_amd import api, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup():
    c = api.Context(0)
    f = synth.small_framework(41, n_atoms=25, cell=(12.0, 11.0, 13.0, 85.0, 97.0, 90.0))
    a = f.particles()
    fw = api.Framework(c, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
    yield c, fw
    fw.close()
    c.close()


@pytest.mark.parametrize("precision", [api.ER_FP32, api.ER_FP64])
def test_energies(setup, precision):
    print(f"pinned energies precision={precision}", flush=True)
    c, fw = setup
    g = api.Grid.compute(c, fw, (30, 28, 33), precision)
    p = np.random.default_rng(3).uniform(-0.5, 1.5, (200000, 3))
    e = api.grid_energies(c, g, p)
    for n in (1, 255, 98303, 98304, 98305):
        assert np.array_equal(api.grid_energies(c, g, p[:n]), e[:n])
    g.close()


@pytest.mark.parametrize("n,precision", [
    ((32, 32, 32), api.ER_FP32), ((32, 32, 33), api.ER_FP32),
    ((16, 32, 32), api.ER_FP64), ((17, 32, 32), api.ER_FP64), ((2, 2, 2), api.ER_FP32)])
def test_grids(setup, n, precision):
    print(f"pinned grid n={n} precision={precision}", flush=True)
    c, fw = setup
    g = api.Grid.compute(c, fw, n, precision)
    kept = g.download()
    g.close()
    assert np.array_equal(api.compute_grid(c, fw, n, precision), kept)
