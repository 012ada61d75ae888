"""smith_lmhead_{q4_0,q6_k}_rows: the logits of several rows against the
float64 product of the oracle's weights, at the edges of its 16 / 32 / 64-row
tiles, 256-column blocks and 32-row K steps, and against the single-row heads
where a result is not finite.

Bar, relative 2-norm: each operand is held to 22 bits (2^-23 rms at most) and
the sums are f32 over at most K / 32 MFMAs per wave: 2e-6 leaves room for
K = 8192 (the single-row heads, plain f32 sums, are held to the same)."""
import numpy as np
import pytest

from oracle import oracle as O
from smith_amd import device, prng

pytestmark = pytest.mark.gpu
BAR = 2e-6
EPS = 1e-5


def _buf(a):
    a = np.ascontiguousarray(a)
    b = device.alloc(max(a.nbytes, 4))
    device.upload(b, a)
    return b


class Head:
    def __init__(self, kind, K, N, seed, scale=0.02, w=None):
        L, ctx = device.lib, device.ops_ctx()
        if w is None:
            w = prng.randn((K, N), seed, std=scale)
        t = O.GGML_Q4_0 if kind == "q4_0" else O.GGML_Q6_K
        blocks = O.quantize_rows(t, w)  # blocks run along vocab
        self.w = O.dequantize_tensor(t, blocks, K * N).reshape(K, N).astype(np.float64)
        self.kind, self.K, self.N = kind, K, N
        src = _buf(blocks)
        if kind == "q4_0":
            self.bufs = (device.alloc(K * N // 2), device.alloc(K * N // 16))
            device.check(L.smith_repack_lmhead_q4_0(ctx, src, *self.bufs, K, N))
        else:
            self.bufs = (device.alloc(int(L.smith_lmhead_q6_k_bytes(K, N))),)
            device.check(L.smith_repack_lmhead_q6_k(ctx, src, *self.bufs, K, N))
        device.sync()
        device.release_buffer(src)

    def run(self, x, gamma, rows=True):
        L, ctx = device.lib, device.ops_ctx()
        M = x.shape[0]
        xb, gb, y = _buf(x), None if gamma is None else _buf(gamma), device.alloc(M * self.N * 4)
        if rows:
            f = L.smith_lmhead_q4_0_rows if self.kind == "q4_0" else L.smith_lmhead_q6_k_rows
            device.check(f(ctx, xb, M, gb, EPS, *self.bufs, y, self.K, self.N))
        else:
            f = L.smith_lmhead_q4_0_nb if self.kind == "q4_0" else L.smith_lmhead_q6_k_nb
            for m in range(M):
                device.check(f(ctx, xb + m * self.K * 4, gb, EPS, *self.bufs, y + m * self.N * 4, self.K, self.N))
        out = device.download(y, M * self.N * 4, np.float32).reshape(M, self.N)
        for b in (xb, y) + (() if gb is None else (gb,)):
            device.release_buffer(b)
        return out

    def ref(self, x, gamma):
        x = x.astype(np.float64)
        if gamma is not None:
            x = x / np.sqrt((x * x).mean(1, keepdims=True) + EPS) * gamma
        return x @ self.w

    def close(self):
        for b in self.bufs:
            device.release_buffer(b)


def rel2(y, ref):
    return float(np.linalg.norm(y - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("kind,K,N", [("q4_0", 8, 32), ("q4_0", 40, 96), ("q4_0", 1032, 288), ("q4_0", 3072, 1024),
                                      ("q6_k", 16, 256), ("q6_k", 48, 512), ("q6_k", 1040, 768),
                                      ("q6_k", 8192, 256)])
def test_rows_match_reference(kind, K, N):
    h = Head(kind, K, N, 821)
    for M in (1, 2, 15, 16, 17, 33, 64, 65, 131):
        x = prng.randn((M, K), 822 + M)
        for gamma in (None, 1 + prng.randn((K,), 823, std=0.1)):
            assert rel2(h.run(x, gamma), h.ref(x, gamma)) <= BAR, (M, gamma is None)
    h.close()


# 2e-5 gives Q4_0 subnormal f16 scales; a Q6_K scale is 1/4064 of the largest
# weight, so 2e-4 (2e-5 would round every scale, and the weights, to zero)
@pytest.mark.parametrize("kind,scale", [("q4_0", 2e-5), ("q4_0", 0.02), ("q4_0", 200.0), ("q6_k", 2e-4),
                                        ("q6_k", 0.02), ("q6_k", 200.0)])
def test_rows_scales(kind, scale):
    """Weights down to f16-subnormal scales and rows of very different sizes:
    every row to its own bar (subnormal scales leave the single-row heads'
    f32 products and these exact splits alike)."""
    K, N = 1024, 512
    h = Head(kind, K, N, 824, scale)
    x = prng.randn((6, K), 825) * np.float32([[1e-20], [1e-4], [1.0], [300.0], [1e6], [1e20]])
    x[2, 5] = 3e4  # one element far above its row
    y, ref = h.run(x, None), h.ref(x, None)
    for m in range(6):
        assert rel2(y[m], ref[m]) <= BAR, m
    h.close()


@pytest.mark.parametrize("kind", ["q4_0", "q6_k"])
def test_rows_of_any_size(kind):
    """Rows from next to the smallest f32 numbers to next to the largest."""
    K, N = 1024, 512
    h = Head(kind, K, N, 828)
    x = prng.randn((6, K), 829) * np.float32([[1e-36], [1e-33], [1e-32], [1e-30], [1e33], [3e35]])
    y, ref = h.run(x, None), h.ref(x, None)
    for m in range(6):
        assert rel2(y[m].astype(np.float64), ref[m]) <= BAR, m
    h.close()


@pytest.mark.parametrize("kind", ["q4_0", "q6_k"])
def test_rows_outlier_at_zero_weights(kind):
    """An element far above its row that meets zero weights: the outputs of
    those columns come from the other elements alone, which keep their bits."""
    K, N, at = 1024, 1024, 5
    w = prng.randn((K, N), 830, std=0.02)
    w[at, :N // 2] = 0.0
    h = Head(kind, K, N, 0, w=w)
    assert not h.w[at, :N // 2].any()
    x = prng.randn((4, K), 831)
    x[:, at] = [1e2, 1e4, 1e6, 1e8]
    y, ref = h.run(x, None), h.ref(x, None)
    for m in range(4):
        assert rel2(y[m, :N // 2], ref[m, :N // 2]) <= BAR, m
        assert rel2(y[m, N // 2:], ref[m, N // 2:]) <= BAR, m
    h.close()


@pytest.mark.parametrize("kind", ["q4_0", "q6_k"])
def test_rows_not_finite(kind):
    K, N = 64, 512
    h = Head(kind, K, N, 826)
    x = prng.randn((20, K), 827)
    x[3, 7], x[4, 1], x[18, 63] = np.inf, np.nan, -np.inf
    x[5] = 0.0
    for gamma in (None, np.ones(K, np.float32)):
        y, want = h.run(x, gamma), h.run(x, gamma, rows=False)
        for m in range(20):
            if np.isfinite(want[m]).all():
                assert np.allclose(y[m], want[m], rtol=0, atol=4e-6 * max(1e-30, np.abs(want[m]).max())), m
            else:
                assert np.array_equal(np.isnan(y[m]), np.isnan(want[m])), m
                f = ~np.isnan(want[m])
                assert np.array_equal(y[m][f], want[m][f]), m
    h.close()


@pytest.mark.parametrize("kind", ["q4_0", "q6_k"])
@pytest.mark.parametrize("M", [17, 64])
def test_rows_not_finite_time(kind, M):
    """Rows that are redone in f32 cost no more than the same rows through the
    single-row head (twice that: room for the clocks)."""
    K, N = 2048, 16384
    h = Head(kind, K, N, 832)
    x = prng.randn((M, K), 833)
    x[:, 9] = np.nan
    us = []
    for rows, name in ((True, "smith_lmhead_%s_rows_m" % kind), (False, "smith_lmhead_%s_nb" % kind)):
        assert np.isnan(h.run(x, None, rows)).all()
        device.profile_kernels(True)
        h.run(x, None, rows)
        ms, _ = device.profile_read(name)
        device.profile_read("")
        device.profile_kernels(False)
        us.append(ms)
    assert us[0] <= 2 * us[1], us
    h.close()


@pytest.mark.parametrize("kind", ["q4_0", "q6_k"])
def test_rows_weights_beyond_f16(kind):
    """Weights above the f16 range: every row is redone in f32."""
    K, N = 264 if kind == "q4_0" else 272, 768
    h = Head(kind, K, N, 834, 6e4)
    assert np.abs(h.w).max() > 65504
    for M in (5, 33, 70):
        x = prng.randn((M, K), 835)
        g = 1 + prng.randn((K,), 836, std=0.1)
        assert rel2(h.run(x, g), h.ref(x, g)) <= BAR, M
    h.close()


@pytest.mark.parametrize("kind", ["q4_0", "q6_k"])
@pytest.mark.parametrize("M,K,N", [(2, 3072, 1024), (3, 4096, 2048), (5, 8192, 256), (2, 1024, 32768), (16, 3072, 8192)])
def test_few_rows_time(kind, M, K, N):
    """A few rows cost no more than through the single-row head (30 % above
    it: room for the clocks), and agree with it."""
    h = Head(kind, K, N, 837)
    x = prng.randn((M, K), 838)
    us, out = [], []
    for rows in (True, False):
        h.run(x, None, rows)
        device.profile_kernels(True)
        out.append(h.run(x, None, rows).astype(np.float64))
        ms, _ = device.profile_read("smith_lmhead_")
        device.profile_read("")
        device.profile_kernels(False)
        us.append(ms * 1e3)
    print(kind, M, K, N, us)
    assert us[0] <= 1.3 * us[1], us
    assert rel2(out[0], out[1]) <= BAR
    h.close()
