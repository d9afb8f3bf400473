"""The bins of a Widom run stay within what the binning kernels histogram in LDS.

3e8 insertions at one insertion a bin ask for 3e8 bins; the binning takes at most
7168 groups of 15360 bins.  The host code runs against a stand-in of the HIP runtime
(tests/host/fake_hip.cpp), whose device memory is never touched: what the run
allocates (three words a bin, three an insertion) tells the bins.
"""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import fake  # noqa: E402


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return fake.build(tmp_path_factory.mktemp("fake"))


@pytest.mark.parametrize("n,most", [(300_000_000, 7168 * 15360), (50_000_000, 51_000_000)])
def test_bins_of_tiny_occupancy(lib, n, most):
    fake.run(lib, f"""
    ctx = api.Context(0)
    tu = api.default_tuning()
    tu.widom_per_bin = 1
    ctx.tuning = tu
    fw = api.Framework(ctx, *ARGS)
    held = fake.fake_device_used()
    api.widom(ctx, fw, {n}, 300.0, 5)
    bins = (fake.fake_device_used() - held - 12 * {n}) // 12
    assert 0.9 * min({n}, {most}) <= bins <= {most} + 1_000_000, bins
    fw.close(); ctx.close()
    """)
