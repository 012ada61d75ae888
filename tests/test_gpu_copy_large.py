"""smith_copy_d2h through the pinned slots (4 MB and up): every byte, at the
edges of the threshold, the 1 MB chunks and the eight slots, from an offset,
in order with work enqueued before it, and from two threads at once."""
import threading

import numpy as np
import pytest

from smith_amd import device

pytestmark = pytest.mark.gpu
MB = 1 << 20


@pytest.mark.parametrize("nbytes", [4 * MB - 4, 4 * MB, 4 * MB + 4, 8 * MB, 8 * MB + 8, 9 * MB - 4, 33 * MB + 12])
@pytest.mark.parametrize("offset", [0, 260])
def test_bytes(nbytes, offset):
    a = np.random.default_rng(nbytes + offset).integers(0, 2**32, (nbytes + offset) // 4, dtype=np.uint32)
    b = device.alloc(a.nbytes)
    device.upload(b, a)
    for _ in range(2):
        got = device.download(b, nbytes, np.uint32, offset)
        assert np.array_equal(got, a[offset // 4:])
    # ordered after the kernel enqueued just before
    device.check(device.lib.smith_fill_zero(device.ops_ctx(), b, a.nbytes))
    assert not device.download(b, nbytes, np.uint32, offset).any()
    device.release_buffer(b)


def test_two_threads():
    n = 6 * MB + 4
    data = [np.random.default_rng(i).integers(0, 2**32, n // 4, dtype=np.uint32) for i in range(2)]
    bufs = [device.alloc(n) for _ in data]
    for b, a in zip(bufs, data):
        device.upload(b, a)
    ok = [False, False]

    def work(i):
        ok[i] = all(np.array_equal(device.download(bufs[i], n, np.uint32), data[i]) for _ in range(5))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert ok == [True, True]
    for b in bufs:
        device.release_buffer(b)
