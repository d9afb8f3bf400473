"""A large result's copy to the host starts when the kernels before it have ended.

While a grid is computed neither the caller nor the copy's helping threads may use
the host's cores, nor may the copy hold the slots that every context of the device
shares.  The host code runs against a stand-in of the HIP runtime whose kernels
only take time (tests/host/fake_hip.cpp).
"""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import fake  # noqa: E402


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return fake.build(tmp_path_factory.mktemp("fake"))


@pytest.mark.parametrize("n", [(100, 90, 80), (180, 170, 160)])
def test_no_core_waits_for_a_kernel(lib, n):
    fake.run(lib, f"""
    ctx = api.Context(0)
    fw = api.Framework(ctx, *ARGS)
    api.compute_grid(ctx, fw, {n!r})          # buffers and threads are made
    fake.fake_kernel_ms(400)
    wall, cpu = time.perf_counter(), time.process_time()
    api.compute_grid(ctx, fw, {n!r})
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert wall > 0.4, wall
    assert cpu < 0.2, cpu                  # (a core that waits uses 0.4 and more)
    fw.close(); ctx.close()
    """)


def test_slots_are_free_while_a_kernel_runs(lib):
    fake.run(lib, """
    n = (180, 170, 160)
    one, two = api.Context(0), api.Context(0)
    fw = [api.Framework(c, *ARGS) for c in (one, two)]
    for c, w in zip((one, two), fw):
        api.compute_grid(c, w, n)
    done = threading.Event()
    def long():
        api.compute_grid(one, fw[0], n)
        done.set()
    fake.fake_kernel_ms(1500)
    t = threading.Thread(target=long)
    t.start()
    time.sleep(0.3)
    fake.fake_kernel_ms(0)
    before = fake.fake_ring_copies()
    api.compute_grid(two, fw[1], n)
    assert not done.is_set()
    assert fake.fake_ring_copies() - before >= 9, fake.fake_ring_copies() - before
    t.join()
    for w in fw: w.close()
    one.close(); two.close()
    """)
