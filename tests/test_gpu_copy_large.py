"""smith_copy_d2h through the pinned slots (4 MB and up): every byte, at the
edges of the threshold, the 1 MB chunks and the eight slots, from an offset,
in order with work enqueued before it, and from two threads at once; into pinned memory, directly;
and behind a long queue of earlier work."""
import ctypes
import threading
import time

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


def test_pinned_destination():
    """Pinned memory is written by the DMA itself: a copy takes as long as the
    runtime's own (1.4 times that: room for the clocks), not that of the slots
    and a copy on the host."""
    n = 64 * MB
    a = np.random.default_rng(3).integers(0, 2**32, n // 4, dtype=np.uint32)
    b = device.alloc(n)
    device.upload(b, a)
    hip, dst = ctypes.CDLL("libamdhip64.so.7"), ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(dst), ctypes.c_size_t(n), 0) == 0
    out = np.ctypeslib.as_array((ctypes.c_uint32 * (n // 4)).from_address(dst.value))
    calls = {"runtime": lambda: hip.hipMemcpy(dst, ctypes.c_void_p(b), ctypes.c_size_t(n), 2),
             "smith": lambda: device.download_into(out, b)}
    best = {}
    for name, call in calls.items():
        out[:] = 0
        for _ in range(6):
            t = time.perf_counter()
            call()
            t = time.perf_counter() - t
            best[name] = min(best.get(name, t), t)
        assert np.array_equal(out, a), name
    print(best)
    assert best["smith"] <= 1.4 * best["runtime"], best
    # memory in the middle of a pinned allocation
    out[:] = 0
    device.download_into(out[1000:], b, 4000)
    assert np.array_equal(out[1000:], a[1000:]) and not out[:1000].any()
    device.release_buffer(b)
    hip.hipHostFree(dst)


def test_waits_in_one_thread():
    """While the stream still works on what was enqueued before the copy, one
    thread waits (the helpers would make it four)."""
    M, N, K = 2048, 4096, 4096
    a, out, b = device.alloc(M * K * 4), device.alloc(M * N * 4), device.alloc(8 * MB)
    w = device.alloc(K // 32 * N * 24)
    for buf, n in ((a, M * K * 4), (w, K // 32 * N * 24), (b, 8 * MB)):
        device.check(device.lib.smith_fill_zero(device.ops_ctx(), buf, n))
    device.download(b, 8 * MB, np.uint32)
    for _ in range(2):  # the first round makes the scratch
        device.sync()
        wall, cpu = time.perf_counter(), time.process_time()
        for _ in range(400):
            device.check(device.lib.smith_matmul_q4(device.ops_ctx(), a, w, out, M, N, K, K // 32))
        queued = time.perf_counter() - wall
        device.download(b, 8 * MB, np.uint32)
        wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    print("waits", queued, wall, cpu)
    assert wall > 2 * queued  # the copy did wait for the GPU
    assert cpu <= 1.6 * wall, (cpu, wall)
    for buf in (a, out, b, w):
        device.release_buffer(buf)
