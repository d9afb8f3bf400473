"""GPU test of batches of many small jobs.

A small job alone shares the records of a point out to several waves; in a batch
that fills the device one wave makes the same sums.  Every grid and every Widom sum
must have the bits it has alone, over jobs of eight, four and two parts, both
precisions, lists of several passes, bins of one, two and several rounds and
saturated insertions; and the batch must not cost what idle waves are for: its time
is compared with the same grids at one point per lane, which have no parts (a
quarter of the difference that sharing out makes there is allowed).
"""
import statistics
import time

import numpy as np
import pytest

from emptyroom_amd import api, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def bctx():
    c = api.Context(0)
    yield c
    c.close()


def frameworks(ctx):
    got = []
    for k, (atoms, cell) in enumerate([(40, (11.0, 12.0, 13.0, 80.0, 95.0, 105.0)),
                                       (150, (14.0, 13.0, 15.0, 90.0, 90.0, 90.0)),
                                       (700, (12.0, 14.0, 13.0, 85.0, 101.0, 90.0)),
                                       (60, (20.0, 18.0, 19.0, 90.0, 97.0, 90.0))]):
        f = synth.small_framework(80 + k, n_atoms=atoms, cell=cell, ntypes=1 + 2 * k)
        a = f.particles()
        got.append(api.Framework(ctx, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2))
    return got


def run(ctx, tasks, graph):
    b = api.Batch(ctx, tasks, use_graph=graph)
    for _ in range(3):
        b.run()
        b.wait()
    return b


@pytest.mark.parametrize("per_bin", [480, 200, 1700])
def test_bits_of_each_job_alone(bctx, per_bin):
    print(f"small batch per_bin={per_bin}", flush=True)
    tu = api.default_tuning()
    tu.widom_per_bin = per_bin
    bctx.tuning = tu
    try:
        fws = frameworks(bctx)
        dims = [(9, 9, 9), (20, 17, 30), (33, 40, 37), (48, 41, 50), (57, 49, 52), (64, 63, 60)]
        tasks = [dict(fw=fws[k % 4], grid_n=dims[k % 6], precision=(k // 2) % 2,
                      n_insertions=(500, 9000, 61000, 150000)[(k + k // 4) % 4], seed=k,
                      temperature=(300.0, 15.0)[k % 2]) for k in range(48)]
        for graph in (False, True):
            b = run(bctx, tasks, graph)
            for k, t in enumerate(tasks):
                alone = api.compute_grid(bctx, t["fw"], t["grid_n"], t["precision"])
                differ = int(np.sum(b.grid(k) != alone))
                assert differ == 0, (k, differ)
                assert b.widom(k) == api.widom(bctx, t["fw"], t["n_insertions"], t["temperature"],
                                               t["seed"]), k
            b.close()
        for fw in fws:
            fw.close()
    finally:
        bctx.tuning = api.default_tuning()


def test_many_small_grids_cost_no_more_than_unshared(bctx):
    def us(tasks):
        b = run(bctx, tasks, True)
        v = []
        for _ in range(9):
            t = time.perf_counter()
            b.run()
            b.wait()
            v.append(1e6 * (time.perf_counter() - t))
        b.close()
        return statistics.median(v)

    got = []
    try:
        for ppl, tile in ((2, (8, 8, 8)), (1, (8, 8, 4))):
            tu = api.default_tuning()
            tu.points_per_lane = ppl
            tu.tile[0], tu.tile[1], tu.tile[2] = tile
            bctx.tuning = tu
            fws = frameworks(bctx)
            got.append(us([dict(fw=fws[k % 4], grid_n=(40, 33, 37)) for k in range(128)]))
            for fw in fws:
                fw.close()
    finally:
        bctx.tuning = api.default_tuning()
    print(f"128 small grids: {got[0]:.0f} us, one point per lane {got[1]:.0f} us", flush=True)
    assert got[0] <= 1.25 * got[1]
