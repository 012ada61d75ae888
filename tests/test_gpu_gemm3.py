"""The prefill GEMM: smith_gemm3_* (K % 64 == 0) at the edges of its tiles, ring
and splits and in every row-tile count, smith_gemm2_* at the edges of its
rule, and the register-staged kernels that K % 64 == 32 leaves to; against the
float64 product of the oracle's weights, each with the kernel's name.

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


class launched:
    """with launched(prefix, n): exactly n GEMM kernels run, all named prefix*"""

    def __init__(self, prefix, n=1):
        self.prefix, self.n = prefix, n

    def __enter__(self):
        device.profile_kernels(True)

    def __exit__(self, exc, *_):
        _, n = device.profile_read(self.prefix)
        other = sum(device.profile_read("smith_gemm%s_%s" % (v, f))[1] for v in ("", "2", "3") for f in ("q4", "q5", "q6", "q8"))
        device.profile_read("")
        device.profile_kernels(False)
        if exc is None:
            assert (n, other) == (self.n, 0), (self.prefix, n, other)


class Tiles:
    """GGUF tile planes of random weights [N, K]"""

    def __init__(self, t, N, K, seed):
        blocks = O.quantize_rows(t, prng.randn((N, K), seed, std=0.02))
        self.w = O.dequantize_tensor(t, blocks, N * K).reshape(N, K).astype(np.float64)
        self.t, self.N, self.K = t, N, K
        L, src = device.lib, device.alloc(blocks.size)
        self.planes = device.alloc(int(L.smith_gguf_tiles_bytes(t, N, K)))
        device.upload(src, blocks)
        device.check(L.smith_repack_gguf_tiles_into(device.ops_ctx(), t, src, self.planes, N, K, 0, 1, N))
        device.sync()
        device.release_buffer(src)

    def run(self, x, M):
        out = S.create([M, self.N])
        device.check(device.lib.smith_linear_gguf_tiles(device.ops_ctx(), self.t, x.buffer, self.planes, out.buffer, M,
                                                        self.N, self.K, None, 0.0, None, 0))
        return out

    def close(self):
        device.release_buffer(self.planes)


def matmul(fmt, at, wa, M, N, K):
    """a [M, K] times the weights of `weights`"""
    out = S.create([M, N])
    L, ctx = device.lib, device.ops_ctx()
    if fmt == "q40":
        device.check(L.smith_matmul_q4_0(ctx, at.buffer, *wa, out.buffer, M, N, K))
    else:
        device.check((L.smith_matmul_q4 if fmt == "q4s" else L.smith_matmul_q8)(ctx, at.buffer, *wa, out.buffer, M, N, K,
                                                                              K // 32))
    return out


# one to three stages (fewer than the ring holds), a last split that is
# shorter, one row past a tile, columns of one lane to one past the tile, odd N
# (records that start off a dword); the plan takes 64-row tiles for all of them
@pytest.mark.parametrize("fmt", ["q4s", "q8", "q40"])
@pytest.mark.parametrize("M,N,K", [(64, 1, 64), (65, 17, 128), (70, 255, 192), (97, 257, 256), (129, 300, 1088),
                                   (161, 33, 4096), (190, 512, 320), (224, 6, 2048), (257, 511, 448),
                                   (300, 1029, 1024)])
def test_gemm3_edges(fmt, M, N, K):
    wa, wd, bufs = weights(fmt, K, N, 701)
    a = prng.randn((M, K), 702)
    at = S.tensor(a)
    with launched("smith_gemm3_%s_m4" % fmt):
        out = matmul(fmt, at, wa, M, N, K)
    assert rel2(out.data, a.astype(np.float64) @ wd) <= BAR
    for b in bufs:
        device.release_buffer(b)


def check_epilogue(fmt, epi, M, N, K, kernel):
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
    with launched(kernel):
        device.check(entry(device.ops_ctx(), xt.buffer, *wa, out.buffer, M, N, K, gt.buffer, 1e-5, rt.buffer, epi))
    # silu(g) * u moves by up to 1.1 |dg| |u| + |silu(g)| |du|: twice the bar
    assert rel2(out.data, y) <= (BAR if epi == 1 else 2 * BAR)
    for b in bufs:
        device.release_buffer(b)


@pytest.mark.parametrize("fmt", ["q8", "q40"])
@pytest.mark.parametrize("epi", [1, 2])
@pytest.mark.parametrize("M,N,K", [(66, 254, 64), (66, 252, 64), (130, 600, 2048), (514, 4098, 128)])
def test_gemm3_epilogues(fmt, epi, M, N, K):
    """Residual and SwiGLU with a fused RMSNorm, stored by the GEMM itself
    (short K) and by the K-split reduce; N % 4 != 0 takes the scalar stores."""
    check_epilogue(fmt, epi, M, N, K, "smith_gemm3_%s_m" % fmt)


# rows whose plan over 65 column tiles takes each row-tile count: the last
# tile short, exactly one row past two tiles, and in between
TM_ROWS = ((4, 190), (6, 193), (8, 300), (10, 385), (12, 500), (14, 577), (16, 700))


@pytest.mark.parametrize("K", [64, 128, 192, 320])
@pytest.mark.parametrize("fmt", ["q4s", "q8", "q40"])
def test_gemm3_row_tiles(fmt, K):
    """Every row-tile count (a ring, loads per wave and MFMA order of its own)
    at one to five stages, the last column tile of one column."""
    N = 16385
    wa, wd, bufs = weights(fmt, K, N, 721)
    a = prng.randn((700, K), 722)
    at, ref = S.tensor(a), a.astype(np.float64) @ wd
    for tm, M in TM_ROWS:
        print(fmt, K, tm, M, flush=True)
        with launched("smith_gemm3_%s_m%d" % (fmt, tm)):
            out = matmul(fmt, at, wa, M, N, K)
        assert rel2(out.data, ref[:M]) <= BAR, (tm, M)
    for b in bufs:
        device.release_buffer(b)


@pytest.mark.parametrize("t,K", [(t, K) for t in (O.GGML_Q4_0, O.GGML_Q4_1, O.GGML_Q5_0) for K in (64, 192, 320)] + [
    (t, K) for t in (O.GGML_Q4_K, O.GGML_Q6_K) for K in (256, 512)])
def test_gemm3_tiles_row_tiles(t, K):
    """As above on the tile planes, the last column tile of 16 columns."""
    tag = {O.GGML_Q4_0: "q40t", O.GGML_Q4_1: "q41t", O.GGML_Q5_0: "q50t", O.GGML_Q4_K: "q4kt", O.GGML_Q6_K: "q6kt"}[t]
    w = Tiles(t, 16400, K, 723)
    a = prng.randn((700, K), 724)
    at, ref = S.tensor(a), a.astype(np.float64) @ w.w.T
    for tm, M in TM_ROWS:
        print(tag, K, tm, M, flush=True)
        with launched("smith_gemm3_%s_m%d" % (tag, tm)):
            out = w.run(at, M)
        assert rel2(out.data, ref[:M]) <= BAR, (tm, M)
    w.close()


@pytest.mark.parametrize("fmt,tm,M,N,K", [("q8", 6, 258, 3095, 1280), ("q8", 8, 196, 5413, 1280),
                                          ("q8", 10, 257, 7270, 1792), ("q8", 14, 197, 8212, 2560),
                                          ("q4s", 6, 260, 2085, 2304), ("q4s", 8, 200, 5382, 1600)])
def test_gemm3_row_tiles_splits(fmt, tm, M, N, K):
    """Wider row tiles with K splits (4 to 9 of them)."""
    wa, wd, bufs = weights(fmt, K, N, 725)
    a = prng.randn((M, K), 726)
    at = S.tensor(a)
    with launched("smith_gemm3_%s_m%d" % (fmt, tm)):
        out = matmul(fmt, at, wa, M, N, K)
    assert rel2(out.data, a.astype(np.float64) @ wd) <= BAR
    for b in bufs:
        device.release_buffer(b)


# K % 64 == 32, the last stage half empty: each tile of the register-staged
# kernels (from 256 rows 256 x 256 with 1, 2, 4 and 8 K splits), rows and
# columns short of their tiles
@pytest.mark.parametrize("fmt", ["q4s", "q8", "q40"])
@pytest.mark.parametrize("tile,M,N,K", [("m128_n64", 64, 70, 96), ("m128_n64", 200, 130, 1056),
                                        ("m128_n128", 200, 16400, 32), ("m256_n128", 100, 25700, 32),
                                        ("m256_n256", 257, 18, 32), ("m256_n256", 257, 520, 1056),
                                        ("m256_n256", 513, 96, 2080), ("m256_n256", 300, 300, 4128)])
def test_register_staged(fmt, tile, M, N, K):
    wa, wd, bufs = weights(fmt, K, N, 727)
    a = prng.randn((M, K), 728)
    at = S.tensor(a)
    with launched("smith_gemm_%s_%s" % (fmt, tile)):
        out = matmul(fmt, at, wa, M, N, K)
    assert rel2(out.data, a.astype(np.float64) @ wd) <= BAR
    for b in bufs:
        device.release_buffer(b)


@pytest.mark.parametrize("t", [O.GGML_Q4_0, O.GGML_Q4_1, O.GGML_Q5_0])
@pytest.mark.parametrize("tile,M,N,K", [("m128_n64", 65, 48, 96), ("m128_n64", 129, 272, 1056),
                                        ("m256_n256", 300, 272, 1056)])
def test_register_staged_tiles(t, tile, M, N, K):
    tag = {O.GGML_Q4_0: "q40t", O.GGML_Q4_1: "q41t", O.GGML_Q5_0: "q50t"}[t]
    w = Tiles(t, N, K, 729)
    a = prng.randn((M, K), 730)
    at = S.tensor(a)
    with launched("smith_gemm_%s_%s" % (tag, tile)):
        out = w.run(at, M)
    assert rel2(out.data, a.astype(np.float64) @ w.w.T) <= BAR
    w.close()


@pytest.mark.parametrize("t", [O.GGML_Q4_0, O.GGML_Q4_1, O.GGML_Q5_0, O.GGML_Q4_K, O.GGML_Q6_K])
@pytest.mark.parametrize("M", [66, 130])
def test_planes_off_a_dword(t, M):
    """Planes that start two bytes past a dword take the register-staged
    kernel (the DMA needs dwords)."""
    N, K = 48, 512
    tag = {O.GGML_Q4_0: "q40t", O.GGML_Q4_1: "q41t", O.GGML_Q5_0: "q50t", O.GGML_Q4_K: "q4kt", O.GGML_Q6_K: "q6kt"}[t]
    w = Tiles(t, N, K, 733)
    raw = device.download(w.planes, int(device.lib.smith_gguf_tiles_bytes(t, N, K)), np.uint8)
    base = device.alloc(raw.size + 64)
    device.upload(base, np.concatenate([np.zeros(2, np.uint8), raw, np.zeros(62, np.uint8)]))
    a = prng.randn((M, K), 734)
    at, out = S.tensor(a), S.create([M, N])
    with launched("smith_gemm_%s_m128_n64" % tag):
        device.check(device.lib.smith_linear_gguf_tiles(device.ops_ctx(), t, at.buffer, base + 2, out.buffer, M, N, K,
                                                        None, 0.0, None, 0))
    assert rel2(out.data, a.astype(np.float64) @ w.w.T) <= BAR
    device.release_buffer(base)
    w.close()


@pytest.mark.parametrize("fmt", ["q8", "q40"])
@pytest.mark.parametrize("epi", [1, 2])
@pytest.mark.parametrize("M,N,K", [(300, 320, 1056), (300, 322, 480), (130, 66, 1056)])
def test_register_staged_epilogues(fmt, epi, M, N, K):
    """Residual and SwiGLU with a fused RMSNorm at K % 64 == 32, by the K-split
    reduce and (K = 480) by the kernel itself."""
    check_epilogue(fmt, epi, M, N, K, "smith_gemm_%s_m" % fmt)


# either side of the rule that leaves 65 .. 128 rows of small Q4_K / Q6_K
# matrices to smith_gemm2_*: rows, columns, and N * K at 24 Mi (Q4_K)
@pytest.mark.parametrize("t,M,N,K,v", [(t, M, N, K, v) for t in (O.GGML_Q4_K, O.GGML_Q6_K)
                                       for M, N, K, v in ((64, 528, 768, 3), (65, 528, 768, 2), (66, 16, 256, 2),
                                                          (97, 1040, 2048, 2), (128, 272, 512, 2), (129, 272, 512, 3),
                                                          (100, 8176, 256, 2), (100, 8192, 256, 3))] + [
    (O.GGML_Q4_K, 70, 4080, 6144, 2), (O.GGML_Q4_K, 70, 4096, 6144, 3), (O.GGML_Q6_K, 70, 4096, 6144, 2)])
def test_gemm2_rule(t, M, N, K, v):
    w = Tiles(t, N, K, 731)
    a = prng.randn((M, K), 732)
    at = S.tensor(a)
    with launched("smith_gemm%d_%s_m" % (v, "q4kt" if t == O.GGML_Q4_K else "q6kt")):
        out = w.run(at, M)
    assert rel2(out.data, a.astype(np.float64) @ w.w.T) <= BAR
    w.close()


# tile planes: row tiles from 32 rows, tiles past the last column, one to a few
# stages, rows on either side of the 65 .. 128 that Q4_K / Q6_K may leave to gemm2
@pytest.mark.parametrize("t", [O.GGML_Q4_0, O.GGML_Q4_1, O.GGML_Q5_0, O.GGML_Q4_K, O.GGML_Q6_K])
@pytest.mark.parametrize("M,N,K", [(2, 16, 256), (33, 272, 512), (64, 528, 768), (129, 48, 2048), (200, 1040, 256),
                                   (257, 8208, 256)])
def test_gemm3_tiles(t, M, N, K):
    if t == O.GGML_Q4_0 and M < 64:
        M = 64  # fewer rows of Q4_0 tiles run the GEMVs
    w = Tiles(t, N, K, 711)
    x = prng.randn((M, K), 712)
    xt = S.tensor(x)
    with launched("smith_gemm3_"):
        out = w.run(xt, M)
    assert rel2(out.data, x.astype(np.float64) @ w.w.T) <= BAR
    w.close()
