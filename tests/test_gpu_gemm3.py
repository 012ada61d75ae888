"""smith_gemm3_* (M >= 64, K % 64 == 0 on (g, n) records) at the edges of its
tiles, ring and splits, against the float64 product of the oracle's weights.

Bar, relative 2-norm: an f16 rounding is uniform within 2^-11, 2.8e-4 rms of
the value; activations and weights are each rounded once (4e-4 together), a
Q4S weight also carries its zero point's product (|scale * zero| of about two
weights' rms) rounded apart: 7e-4.  Three times that: 2e-3.
"""
import numpy as np
import pytest

import smith_amd as S
from oracle import oracle as O
from smith_amd import device, prng

pytestmark = pytest.mark.gpu
BAR = 2e-3


def rel2(y, ref):
    return float(np.linalg.norm(y.astype(np.float64) - ref) / np.linalg.norm(ref))


def weights(fmt, K, N, seed):
    """(device arguments, f64 weights [K, N], buffers to release)"""
    w = prng.randn((K, N), seed, std=0.02)
    if fmt == "q40":
        blocks = O.quantize_rows(O.GGML_Q4_0, np.ascontiguousarray(w.T))
        src, nib, d = device.alloc(blocks.size), device.alloc(N * K // 2), device.alloc(N * K // 16)
        device.upload(src, blocks)
        device.check(device.lib.smith_repack_q4_0(device.ops_ctx(), src, nib, d, N, K))
        wd = O.dequantize_tensor(O.GGML_Q4_0, blocks, N * K).reshape(N, K).T
        return (nib, d), wd.astype(np.float64), (src, nib, d)
    q = (S.quantizeQ4 if fmt == "q4s" else S.quantizeQ8)(w)
    raw = device.download(q["buffer"], q["totalBytes"], np.uint8)
    wd = (O.dequant_q4s if fmt == "q4s" else O.dequant_q8)(raw, K, N)
    return (q["buffer"],), wd.astype(np.float64), (q["buffer"],)


# one to three stages (fewer than the ring holds), a last split that is
# shorter, every row-tile count, one row past a tile, columns of one lane to
# one past the tile, odd N (records that start off a dword)
@pytest.mark.parametrize("fmt", ["q4s", "q8", "q40"])
@pytest.mark.parametrize("M,N,K", [(64, 1, 64), (65, 17, 128), (70, 255, 192), (97, 257, 256), (129, 300, 1088),
                                   (161, 33, 4096), (190, 512, 320), (224, 6, 2048), (257, 511, 448),
                                   (300, 1029, 1024)])
def test_gemm3_edges(fmt, M, N, K):
    wa, wd, bufs = weights(fmt, K, N, 701)
    a = prng.randn((M, K), 702)
    at, out = S.tensor(a), S.create([M, N])
    L, ctx = device.lib, device.ops_ctx()
    device.profile_kernels(True)
    if fmt == "q40":
        device.check(L.smith_matmul_q4_0(ctx, at.buffer, *wa, out.buffer, M, N, K))
    else:
        device.check((L.smith_matmul_q4 if fmt == "q4s" else L.smith_matmul_q8)(ctx, at.buffer, *wa, out.buffer, M, N, K,
                                                                              K // 32))
    _, n = device.profile_read("smith_gemm3_%s_" % fmt)
    device.profile_read("")
    device.profile_kernels(False)
    assert n == 1
    assert rel2(out.data, a.astype(np.float64) @ wd) <= BAR
    for b in bufs:
        device.release_buffer(b)


@pytest.mark.parametrize("fmt", ["q8", "q40"])
@pytest.mark.parametrize("epi", [1, 2])
@pytest.mark.parametrize("M,N,K", [(66, 254, 64), (66, 252, 64), (130, 600, 2048), (514, 4098, 128)])
def test_gemm3_epilogues(fmt, epi, M, N, K):
    """Residual and SwiGLU with a fused RMSNorm, stored by the GEMM itself
    (short K) and by the K-split reduce; N % 4 != 0 takes the scalar stores."""
    wa, wd, bufs = weights(fmt, K, N, 703)
    x = prng.randn((M, K), 704)
    g = 1 + prng.randn((K,), 705, std=0.1)
    r = prng.randn((M, N), 706)
    x64 = x.astype(np.float64)
    y = (x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-5) * g) @ wd
    if epi == 1:
        y = y + r
    else:
        y = y[:, 0::2] / (1 + np.exp(-y[:, 0::2])) * y[:, 1::2]
    xt, gt, rt = S.tensor(x), S.tensor(g), S.tensor(r)
    out = S.create(list(y.shape))
    entry = device.lib.smith_linear_q4_0 if fmt == "q40" else device.lib.smith_linear_q8
    device.check(entry(device.ops_ctx(), xt.buffer, *wa, out.buffer, M, N, K, gt.buffer, 1e-5, rt.buffer, epi))
    # silu(g) * u moves by up to 1.1 |dg| |u| + |silu(g)| |du|: twice the bar
    assert rel2(out.data, y) <= (BAR if epi == 1 else 2 * BAR)
    for b in bufs:
        device.release_buffer(b)


# tile planes: row tiles from 32 rows, tiles past the last column, one to a few
# stages, rows on either side of the 65 .. 128 that Q4_K / Q6_K leave to gemm2
@pytest.mark.parametrize("t", [O.GGML_Q4_0, O.GGML_Q4_1, O.GGML_Q5_0, O.GGML_Q4_K, O.GGML_Q6_K])
@pytest.mark.parametrize("M,N,K", [(2, 16, 256), (33, 272, 512), (64, 528, 768), (129, 48, 2048), (200, 1040, 256),
                                   (257, 8208, 256)])
def test_gemm3_tiles(t, M, N, K):
    if t == O.GGML_Q4_0 and M < 64:
        M = 64  # fewer rows of Q4_0 tiles run the GEMVs
    w = prng.randn((N, K), 711, std=0.02)
    blocks = O.quantize_rows(t, w)
    wd = O.dequantize_tensor(t, blocks, N * K).reshape(N, K).astype(np.float64)
    L, ctx = device.lib, device.ops_ctx()
    src, pl = device.alloc(blocks.size), device.alloc(int(L.smith_gguf_tiles_bytes(t, N, K)))
    device.upload(src, blocks)
    device.check(L.smith_repack_gguf_tiles_into(ctx, t, src, pl, N, K, 0, 1, N))
    x = prng.randn((M, K), 712)
    xt, out = S.tensor(x), S.create([M, N])
    device.profile_kernels(True)
    device.check(L.smith_linear_gguf_tiles(ctx, t, xt.buffer, pl, out.buffer, M, N, K, None, 0.0, None, 0))
    _, n = device.profile_read("smith_gemm3_")
    device.profile_read("")
    device.profile_kernels(False)
    assert n == 1
    assert rel2(out.data, x.astype(np.float64) @ wd.T) <= BAR
    for b in (src, pl):
        device.release_buffer(b)
