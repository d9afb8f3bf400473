"""GPU test of the transfer buffers that contexts share: contexts (and their streams)
come and go while another one keeps the buffers alive.  Uploads, captured batches and
downloads through every path (pinned results, one buffer, ring) must go on working,
with the bits they had at first, whatever the memory of a closed stream is used for
next."""
import numpy as np
import pytest

from emptyroom_amd import api, synth

pytestmark = pytest.mark.gpu


def use(c, f, a):
    fw = api.Framework(c, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
    small = api.compute_grid(c, fw, (9, 8, 7), api.ER_FP32)
    one = api.compute_grid(c, fw, (40, 41, 42), api.ER_FP64)
    ring = api.compute_grid(c, fw, (80, 81, 82), api.ER_FP64)
    b = api.Batch(c, [dict(fw=fw, grid_n=(20, 20, 20), n_insertions=2000, temperature=300.0)],
                  use_graph=True)
    for _ in range(2):
        b.run()
        b.wait()
    got = [small, one, ring, b.grid(0), np.array(b.widom(0)[:2])]
    b.close()
    fw.close()
    return got


def test_contexts_come_and_go():
    print("lifetimes", flush=True)
    f = synth.small_framework(43, n_atoms=20, cell=(12.0, 11.0, 13.0, 85.0, 97.0, 90.0))
    a = f.particles()
    with api.Context(0) as keep:
        ref = use(keep, f, a)
        for k in range(40):
            others = [api.Context(0) for _ in range(1 + k % 3)]
            for c in others:
                assert all(np.array_equal(x, y) for x, y in zip(use(c, f, a), ref))
            for c in others:
                c.close()
            if k % 4 == 0:
                assert all(np.array_equal(x, y) for x, y in zip(use(keep, f, a), ref))
    with api.Context(0) as c:  # the buffers were given back
        assert all(np.array_equal(x, y) for x, y in zip(use(c, f, a), ref))


def test_batch_closed_while_it_runs():
    """A run writes its sums to the batch's own memory: closing waits for it."""
    print("batch closed early", flush=True)
    f = synth.small_framework(44, n_atoms=40, cell=(14.0, 13.0, 12.0, 85.0, 97.0, 90.0))
    a = f.particles()
    with api.Context(0) as c:
        fw = api.Framework(c, a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
        tasks = [dict(fw=fw, grid_n=(60, 60, 60), n_insertions=100000, temperature=300.0, seed=k)
                 for k in range(8)]
        ref = api.widom(c, fw, 100000, 300.0, 3)
        for k in range(10):
            b = api.Batch(c, tasks, use_graph=bool(k % 2))
            b.run()
            b.close()
        b = api.Batch(c, tasks, use_graph=True)
        b.run()
        b.wait()
        assert b.widom(3) == ref
        b.close()
        fw.close()


def test_server_closed_with_work_done():
    """Requests' and launches' events go before the streams they were recorded on."""
    print("server closed", flush=True)
    f = synth.small_framework(45, n_atoms=30, cell=(12.0, 13.0, 12.0, 85.0, 97.0, 90.0))
    a = f.particles()
    args = (a[:, :3], a[:, 3], a[:, 4], f.t, f.rep, f.rc2)
    for k in range(6):
        with api.Context(0) as c:
            s = api.Server(c)
            tickets = [s.submit(*args, grid_n=(20, 20, 20), n_insertions=5000, temperature=300.0,
                                seed=j)[1] for j in range(4)]
            for t in tickets[:k % 4]:
                assert s.poll(t, -1.0).state == api.RQ_DONE
            s.close()
