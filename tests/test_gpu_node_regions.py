"""GPU test: the values of fine FP32 grids (far field from nodes) do not depend on
the regions their blocks are worked on in.

Regions decide which candidate list a block reads (a region's, or the framework's),
so the chunks of the source and the room beside a region's list differ; the grids
must be equal to the bit.  Dense frameworks have more far atoms a block than one
pass over the list takes; two balls of 2900 atoms, 9 A apart, give blocks near one
of them a list that has no room in a slice beside their region's.
"""
import numpy as np
import pytest

from emptyroom_amd import api, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rctx():
    c = api.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("atoms,ball,ntypes,edge", [(1000, 0, 6, 16.4), (1100, 0, 1, 16.4),
                                                    (1000, 0, 40, 16.4), (5900, 2900, 4, 27.0)])
def test_same_bits_in_every_region(rctx, atoms, ball, ntypes, edge):
    # 17^3 blocks: regions of two blocks leave the 2048 work items a grid alone has
    n, cell = (264, 260, 258), (edge + 0.1, edge, edge - 0.1, 90.0, 95.0, 90.0)
    print(f"node regions atoms={atoms} ball={ball} types={ntypes}", flush=True)
    f = synth.small_framework(61, n_atoms=atoms, cell=cell, ntypes=ntypes)
    if ball:
        u = synth.Rng(62).uniform(6 * ball).reshape(2, ball, 3)
        for k in range(2):
            f.frac[k * ball:(k + 1) * ball] = 0.4 + 0.02 * u[k] + [k * 9.0 / edge, 0.0, 0.0]
    a = f.particles()
    grids = []
    try:
        for length in (api.default_tuning().region_len, 0.0, 2.5):
            tu = api.default_tuning()
            tu.region_len = length
            rctx.tuning = tu
            fw = api.Framework(rctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
            grids.append(api.compute_grid(rctx, fw, n, api.ER_FP32))
            fw.close()
    finally:
        rctx.tuning = api.default_tuning()
    for g in grids[1:]:
        differ = int(np.sum(g != grids[0]))
        assert differ == 0
