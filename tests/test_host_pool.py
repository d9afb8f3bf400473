"""Device memory of a context: optional blocks (the corner records of a trilinear Widom
run, four times the grid) must not cost a program memory or calls that it needs.

The host code runs against a stand-in of the HIP runtime with a device of a chosen
size (tests/host/fake_hip.cpp); no kernel runs.
"""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import fake  # noqa: E402


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return fake.build(tmp_path_factory.mktemp("fake"))


def test_grids_of_many_sizes_keep_one_block_of_records(lib):
    fake.run(lib, """
    ctx = api.Context(0)
    most = 0
    for k in range(8):
        n = (118 + 4 * k, 112, 110)            # 5.8 to 7.2 MB, records 23 to 29 MB
        most = 16 * n[0] * n[1] * n[2]
        g = api.Grid.upload(ctx, np.zeros(n, np.float32))
        before = fake.fake_mallocs()
        api.widom_grid(ctx, g, 2_000_000, 300.0, 5)
        assert k > 0 or fake.fake_mallocs() > before   # (records were asked for)
        g.close()
    grids = sum(4 * (118 + 4 * k) * 112 * 110 for k in range(8))
    assert fake.fake_device_used() < grids + most + (96 << 20), fake.fake_device_used()
    held = fake.fake_device_used()
    ctx.close()
    ctx = api.Context(0)
    empty = fake.fake_device_used()
    ctx.close()
    assert held - empty < grids + most + (24 << 20), (held, empty)
    """)


def test_records_that_do_not_fit_leave_the_cache_and_the_error_alone(lib):
    fake.run(lib, """
    probe = api.Context(0)
    base = fake.fake_device_used()             # what a context itself holds
    probe.close()
    ctx = api.Context(0, hbm_cap=base + (20 << 20))  # the grid, not its records
    n = (118, 112, 110)
    g = api.Grid.upload(ctx, np.zeros(n, np.float32))
    keep = api.Grid.upload(ctx, np.zeros((50, 50, 50), np.float32))
    try:
        api.Grid.upload(ctx, np.zeros((400, 400, 400), np.float32))
        raise SystemExit("no refusal")
    except api.EmptyRoomError:
        pass
    said = api.lib().er_last_error()
    keep.close()                               # a cached block
    frees = fake.fake_frees()
    for k in range(3):
        sb, seb, count = api.widom_grid(ctx, g, 2_000_000, 300.0, 5)
        assert count == 2_000_000
    assert fake.fake_frees() == frees
    assert api.lib().er_last_error() == said
    g.close(); ctx.close()
    """)


def test_cached_blocks_are_given_back_before_a_refusal(lib):
    fake.run(lib, """
    ctx = api.Context(0)
    fake.fake_device_limit(fake.fake_device_used() + (100 << 20))
    big = api.Grid.upload(ctx, np.zeros((256, 256, 256), np.float32))      # 64 MiB
    big.close()                                                            # now cached
    other = api.Grid.upload(ctx, np.zeros((300, 256, 256), np.float32))    # 75 MiB
    other.close(); ctx.close()
    """)
