"""GPU test of the Widom binning: jobs of few bins are sorted in one step, jobs
of many bins into groups of bins and then within the groups.

The insertions-per-bin knob puts a run on either side of the one-step limit of
4096 bins (a mean of one insertion per bin gives about as many bins as
insertions).  Every insertion must reach the bin its point lies in exactly
once, so every energy must be the oracle's: 1e-3 K where E < 1e4 K, as for every
Widom test; an insertion in a wrong bin would miss its own atoms.  A batch of
runs from both sides gives the plain path's sums bit for bit.
"""
import numpy as np
import pytest

from emptyroom_amd import api, synth
from oracle import oracle

pytestmark = pytest.mark.gpu

CELL = (14.0, 15.0, 13.0, 80.0, 100.0, 95.0)


@pytest.fixture(scope="module")
def setup():
    c = api.Context(0)
    f = synth.small_framework(23, n_atoms=30, cell=CELL)
    a = f.particles()
    fw = api.Framework(c, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
    yield c, f, a, fw
    fw.close()
    c.close()


def per_bin(c, v):
    t = c.tuning
    t.widom_per_bin = v
    c.tuning = t


@pytest.mark.parametrize("nins,mean", [(1, 1), (255, 480), (4000, 1), (4500, 1), (20011, 1),
                                       (60001, 7)])
def test_every_insertion_in_its_bin(setup, nins, mean):
    print(f"binning nins={nins} per_bin={mean}", flush=True)
    c, f, a, fw = setup
    per_bin(c, mean)
    try:
        sb, seb, n, e = api.widom(c, fw, nins, 300.0, 77, energies=True)
    finally:
        per_bin(c, 480)
    rb, reb, re = oracle.widom(f.t, a, f.rep, f.rc2, 300.0, 77, 0, nins, energies=True)
    assert n == nins
    mask = re < 1e4
    assert np.max(np.abs(e[mask] - re[mask]), initial=0.0) <= 1e-3
    assert np.all(e[~mask] > 0.99e4)
    assert abs(sb - rb) <= 1e-4 * rb


def test_batch_of_one_and_two_step_jobs(setup):
    print("binning batch", flush=True)
    c, f, a, fw = setup
    per_bin(c, 2)
    try:
        counts = [300, 30000, 5000, 12345]
        tasks = [dict(fw=fw, n_insertions=k, temperature=300.0, seed=5 + i)
                 for i, k in enumerate(counts)]
        plain = [api.widom(c, fw, k, 300.0, 5 + i) for i, k in enumerate(counts)]
        b = api.Batch(c, tasks, use_graph=True)
        for _ in range(3):
            b.run()
            b.wait()
            assert [b.widom(i) for i in range(len(counts))] == plain
        b.close()
    finally:
        per_bin(c, 480)
