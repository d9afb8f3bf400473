"""GPU test of the copies to and from the caller's arrays: sizes at the edges of
the small buffer (1 MiB), of the ring's slots (2 MiB) and of the size from which
threads help (16 MiB), into arrays that begin at odd addresses, from several
threads at once, and after the last context that shares the buffers is gone.
Every byte must arrive; none beyond the array may change."""
import ctypes
import threading

import numpy as np
import pytest

from emptyroom_amd import api

pytestmark = pytest.mark.gpu

MB = 1 << 18  # floats per MiB


def roundtrip(ctx, n, offset, seed):
    h = np.random.default_rng(seed).random(n, dtype=np.float32)
    g = api.Grid.upload(ctx, h)
    room = np.full(h.nbytes + offset + 64, 7, np.uint8)
    api._check(api.lib().er_grid_download(g.h, ctypes.c_void_p(room.ctypes.data + offset)))
    g.close()
    got = room[offset:offset + h.nbytes]
    assert np.array_equal(got, h.reshape(-1).view(np.uint8))
    assert np.all(room[:offset] == 7) and np.all(room[offset + h.nbytes:] == 7)


@pytest.mark.parametrize("n", [(2, 2, 2), (3, 5, 7), (2, 2, MB // 4), (2, 4, MB // 8 + 1),
                               (2, 16, MB // 16), (2, 16, MB // 16 + 1), (5, 16, MB // 16),
                               (16, 16, MB // 16 - 1), (16, 16, MB // 16), (37, 19, MB // 17)])
@pytest.mark.parametrize("offset", [0, 12])
def test_every_byte_arrives(n, offset):
    print(f"transfer n={n} offset={offset}", flush=True)
    with api.Context(0) as c:
        roundtrip(c, n, offset, 1)


def test_threads_and_contexts():
    print("transfer threads", flush=True)
    errors = []

    def client(k):
        try:
            for r in range(3):
                with api.Context(0) as c:
                    for i, n in enumerate([(2, 2, 100 + k), (3, 16, MB // 16), (27, 16, MB // 16)]):
                        roundtrip(c, n, 4 * k, 10 * k + i)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=client, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
