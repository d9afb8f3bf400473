"""The server's grids can be fetched from any thread, whatever its current device, and
after a fetch that failed.

The host code runs against a stand-in of the HIP runtime with two devices
(tests/host/fake_hip.cpp), which refuses, as HIP does, an event that is recorded on
a stream of another device.
"""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host"))
import fake  # noqa: E402


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return fake.build(tmp_path_factory.mktemp("fake"))


# small buffer, ring, ring with helping threads
@pytest.mark.parametrize("n", [(20, 20, 20), (100, 90, 80), (180, 170, 160)])
def test_fetch_from_a_thread_of_another_device(lib, n):
    fake.run(lib, f"""
    n = {n!r}
    ctx = api.Context(1)
    srv = api.Server(ctx)
    ticket = srv.submit(*ARGS, grid_n=n)[1]
    assert srv.poll(ticket, -1.0).state == api.RQ_DONE
    got = []
    def client():   # a new thread: its current device is 0, and stays so
        got.append(srv.fetch_grid(ticket, n))
        d = ctypes.c_int(-1)
        fake.hipGetDevice(ctypes.byref(d))
        assert d.value == 0
        got.append(True)
    t = threading.Thread(target=client)
    t.start(); t.join()
    assert len(got) == 2 and got[0].shape == n
    srv.release(ticket)
    srv.close(); ctx.close()
    """)


def test_fetch_that_runs_out_of_host_memory(lib):
    """The copy may throw (its buffers are made by the first one); the ticket can
    then be fetched again and released."""
    fake.run(lib, """
    n = (100, 90, 80)
    ctx = api.Context(0)
    srv = api.Server(ctx)
    ticket = srv.submit(*ARGS, grid_n=n)[1]
    assert srv.poll(ticket, -1.0).state == api.RQ_DONE
    fake.fake_host_malloc_throws(1)
    try:
        srv.fetch_grid(ticket, n)
        raise SystemExit("fetched")
    except api.EmptyRoomError as e:
        print(e)
    fake.fake_host_malloc_throws(0)
    assert srv.fetch_grid(ticket, n).shape == n
    srv.release(ticket)      # waits for copies that have not ended
    srv.close(); ctx.close()
    """, timeout=30.0)
