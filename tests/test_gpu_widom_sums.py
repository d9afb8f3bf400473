"""GPU test of the Boltzmann sums of a Widom run and of the second binning step's
two ways through a group's pairs.

The sums take a block per 2048 energies, up to 1024 blocks; the sizes lie on both
sides of one block, of two and of the most.  They are compared with the sums of the
energies the same run returns, made in numpy: two orders of n FP64 terms of which the
first sum's are positive differ by n 2^-53 at most, and by much less where both are
trees (1e-12); a lost or doubled block would be 5e-4 or more.

Groups of more than 20480 pairs are read again by the second pass: a run of 2.2e7
insertions in 45000 bins (two steps) against the same run in 3600 (one step), whose
energies differ by FP32 rounding only (1e-3 K where E < 1e4 K); an insertion that
reached no bin keeps a pair of integers for its energy.
"""
import numpy as np
import pytest

from emptyroom_amd import api, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup():
    c = api.Context(0)
    f = synth.small_framework(29, n_atoms=12, cell=(15.0, 14.0, 16.0, 90.0, 100.0, 90.0))
    a = f.particles()
    fw = api.Framework(c, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
    yield c, fw
    fw.close()
    c.close()


@pytest.mark.parametrize("nins", [1, 2047, 2048, 2049, 4097, 300001, 2048 * 1024 + 1])
def test_sums_of_the_energies(setup, nins):
    print(f"sums nins={nins}", flush=True)
    c, fw = setup
    sb, seb, n, e = api.widom(c, fw, nins, 300.0, 5, energies=True)
    assert n == nins
    b = np.exp(-e / 300.0)
    eb = np.where(b == 0.0, 0.0, e * b)
    assert abs(sb - b.sum()) <= 1e-12 * b.sum()
    assert abs(seb - eb.sum()) <= 1e-12 * np.abs(eb).sum()


def test_groups_past_the_kept_pairs(setup):
    print("large groups", flush=True)
    c, fw = setup
    got = []
    try:
        for mean in (480, 6000):
            t = c.tuning
            t.widom_per_bin = mean
            c.tuning = t
            got.append(api.widom(c, fw, 22_000_000, 300.0, 6, energies=True)[3])
    finally:
        t = c.tuning
        t.widom_per_bin = 480
        c.tuning = t
    low = got[1] < 1e4
    assert np.array_equal(low, got[0] < 1e4)
    assert np.max(np.abs(got[0][low] - got[1][low])) <= 1e-3
