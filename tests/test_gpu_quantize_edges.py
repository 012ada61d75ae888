"""quantizeQ4 on the GPU where its f32 quotient must hand over to the f64
arithmetic: ties and values next to them, ranges at the ends of what f32
quotients are used for, NaN / infinities, zero ranges; and at the edges of its
256-column blocks and 32-row groups.  Bytes equal the oracle's."""
import numpy as np
import pytest

import smith_amd as S
from oracle import oracle as O
from smith_amd import device, prng

pytestmark = pytest.mark.gpu


def check(w):
    q = S.quantizeQ4(w)
    got = device.download(q["buffer"], q["totalBytes"], np.uint8)
    device.release_buffer(q["buffer"])
    assert np.array_equal(got, O.quantize_q4s(w))


@pytest.mark.parametrize("K", [1, 31, 32, 33, 64, 95])
@pytest.mark.parametrize("N", [1, 3, 255, 256, 257, 700])
def test_block_and_group_edges(K, N):
    check(prng.randn((K, N), 811, std=0.02))


@pytest.mark.parametrize("K", [32, 63, 8192, 8225])
@pytest.mark.parametrize("N", [1, 2, 7, 85, 86, 127, 128, 129])
def test_narrow(K, N):
    """Several groups to a workgroup up to 128 columns: its last workgroup
    short of groups, its last group short of rows."""
    check(prng.randn((K, N), 812, std=0.02))


@pytest.mark.parametrize("N", [2, 8])
def test_narrow_time(N):
    """A narrow matrix fills the workgroups: quantizing K = 131072 of N columns
    takes no longer than the same weights as 32 times the columns (1.6 times:
    its reads are short)."""
    K = 131072
    us = []
    L, ctx = device.lib, device.ops_ctx()
    w, out = device.alloc(K * N * 4), device.alloc(K // 32 * N * 24)
    device.check(L.smith_fill_zero(ctx, w, K * N * 4))
    for k, n in ((K, N), (K // 32, N * 32)):
        device.check(L.smith_quantize_q4(ctx, w, out, k, n))
        device.profile_kernels(True)
        for _ in range(5):
            device.check(L.smith_quantize_q4(ctx, w, out, k, n))
        ms, cnt = device.profile_read("smith_quantize_q4s")
        device.profile_kernels(False)
        us.append(ms / cnt * 1e3)
    print(N, us)
    assert us[0] <= 1.6 * us[1], us
    for b in (w, out):
        device.release_buffer(b)


@pytest.mark.parametrize("K", [32, 45])
def test_ties_and_ranges(K):
    rng = np.random.default_rng(812)
    cols = []
    for e in (-140, -101, -99, -20, 0, 10, 98, 99, 100, 120):
        s = np.float64(2.0) ** e
        for off in (0.0, -7.25, 3.0, 1e6):
            # levels i and ties i + 0.5 of the 0..15 grid, some one step off
            v = (rng.integers(0, 31, K) * 0.5 + off) * s
            v[0], v[1] = off * s, (15 + off) * s
            f = v.astype(np.float32)
            for k in range(2, K, 3):
                f[k] = np.nextafter(f[k], np.float32(rng.choice([-np.inf, np.inf])))
            cols.append(np.clip(f, f[0], f[1]))
    for sp in (np.nan, np.inf, -np.inf):  # among ordinary values, first and later
        for at in (0, 7):
            c = prng.randn((K, 1), 813)[:, 0].copy()
            c[at] = sp
            cols.append(c)
    cols += [np.zeros(K, np.float32), np.full(K, 3.5, np.float32), np.full(K, -0.0, np.float32),
             np.full(K, np.nan, np.float32), np.full(K, 3e38, np.float32) * np.where(np.arange(K) % 2, 1, -1)]
    with np.errstate(over="ignore", invalid="ignore"):
        check(np.ascontiguousarray(np.stack(cols, 1).astype(np.float32)))
