"""Workloads of the quantized-weight path, as a user's program calls them.

  op        matmulQ4 / matmulQ8 as Python calls them: a new output tensor per
            call, released when the program drops it (the reference's own
            bench shape 32x512 @ 512x512 and its neighbours)
  matmul    smith_matmul_q4 / smith_matmul_q8 of the C ABI on buffers that the
            program keeps: decode GEMVs (M = 1), batched decode (M = 2 .. 63),
            prefill GEMMs (M >= 64)
  quantize  smith_quantize_q4 of a weight matrix
  prefill   loadGGUF(...).forwardPrefill on a prompt: logits of every row
  decode    loadGGUF(...).forwardDecode of one token behind a filled cache

Inputs come from the seed alone.  Weights are N(0, 0.02) quantized by the
formulas below (or random GGUF blocks of that size), activations N(0, 1).
"""
import ctypes
import math
import os
import tempfile

import numpy as np
import torch

import smith_amd as S
from smith_amd import device
from smith_amd import gguf as G
from smith_amd.gguf_loader import loadGGUF

DEV = "cuda"


def listed():
    return [
        # the smallest call: the reference's bench shape through the Python op
        {"name": "q4_op_32x512x512", "kind": "op", "fmt": "q4", "M": 32, "N": 512, "K": 512},
        # one decode projection at M = 1 (the headline GEMV shape)
        {"name": "q4_m1_4096x4096", "kind": "matmul", "fmt": "q4", "M": 1, "N": 4096, "K": 4096},
        # Q8 weights at M = 1: an FFN up projection
        {"name": "q8_m1_14336x4096", "kind": "matmul", "fmt": "q8", "M": 1, "N": 14336, "K": 4096},
        # batched decode, FFN up projection, 8 sequences
        {"name": "q4_m8_14336x4096", "kind": "matmul", "fmt": "q4", "M": 8, "N": 14336, "K": 4096},
        # batched decode with a ragged batch, FFN down projection (long K)
        {"name": "q4_m27_4096x14336", "kind": "matmul", "fmt": "q4", "M": 27, "N": 4096, "K": 14336},
        # more sequences than one GEMV pass takes, Q8 weights
        {"name": "q8_m48_4096x4096", "kind": "matmul", "fmt": "q8", "M": 48, "N": 4096, "K": 4096},
        # prompt of 512 tokens through the FFN up projection
        {"name": "q4_m512_14336x4096", "kind": "matmul", "fmt": "q4", "M": 512, "N": 14336, "K": 4096},
        # several prompts at once through the FFN down projection: the largest
        {"name": "q4_m2048_4096x14336", "kind": "matmul", "fmt": "q4", "M": 2048, "N": 4096, "K": 14336},
        # a prompt of odd length on Q8 weights
        {"name": "q8_m301_14336x4096", "kind": "matmul", "fmt": "q8", "M": 301, "N": 14336, "K": 4096},
        # packing a weight matrix
        {"name": "quantize_q4_4096x14336", "kind": "quantize", "N": 14336, "K": 4096},
        # a prompt through a Llama-shaped GGUF (Q4_K_M type mix), logits of every row
        {"name": "prefill_q4km_128", "kind": "prefill", "mix": "q4_k_m", "dim": 3072, "heads": 24, "kv": 8,
         "ffn": 9216, "vocab": 32000, "layers": 6, "tokens": 128},
        # one decode step of a Llama-shaped GGUF (Q4_0) behind a cache of 200 tokens
        {"name": "decode_q40_200", "kind": "decode", "mix": "q4_0", "dim": 3072, "heads": 24, "kv": 8,
         "ffn": 9216, "vocab": 32000, "layers": 6, "tokens": 200},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    r = rng.random()
    if r < 0.1:
        return {"kind": "op", "fmt": rng.choice(["q4", "q8"]), "M": _log_int(rng, 1, 64), "N": _log_int(rng, 256, 1024),
                "K": 32 * _log_int(rng, 8, 32)}
    if r < 0.68:
        fmt = rng.choice(["q4", "q8"])
        band = rng.random()
        M = 1 if band < 0.15 else (_log_int(rng, 2, 63) if band < 0.55 else _log_int(rng, 64, 2048))
        N, K = _log_int(rng, 512, 14336), 32 * _log_int(rng, 16, 448)
        if rng.random() < 0.5:
            N = (N + 63) // 64 * 64
        if rng.random() < 0.15:  # a last group that is not whole
            K, M = K - rng.randint(1, 31), min(M, 256)
        most = 2048 * 4096 * 14336
        if M * N * K > most:
            M = max(64, most // (N * K))
        return {"kind": "matmul", "fmt": fmt, "M": M, "N": N, "K": K}
    if r < 0.76:
        return {"kind": "quantize", "N": _log_int(rng, 512, 14336), "K": _log_int(rng, 512, 4096)}
    dim, heads, kv, ffn = rng.choice([(1024, 16, 4, 2816), (2048, 32, 4, 5632), (2048, 16, 16, 5632),
                                      (3072, 24, 8, 9216), (4096, 32, 8, 14336)])
    case = {"mix": rng.choice(["q4_0", "q4_k_m"]), "dim": dim, "heads": heads, "kv": kv, "ffn": ffn,
            "vocab": 256 * rng.randint(32, 125), "layers": rng.randint(1, 4)}
    if r < 0.88:
        return {"kind": "prefill", **case, "tokens": _log_int(rng, 2, 250)}
    return {"kind": "decode", **case, "tokens": _log_int(rng, 2, 250)}


# --------------------------------------------------------------------------
# device buffers of the library as torch tensors
# --------------------------------------------------------------------------
class _Buffer:
    """A library allocation seen through the CUDA array interface; released
    when the last torch tensor on it goes."""

    def __init__(self, ptr, shape, typestr, owned=True):
        self.ptr, self.owned = ptr, owned
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (ptr, False), "version": 2}

    def __del__(self):
        if self.owned:
            device.release_buffer(self.ptr)


def _view(ptr, shape, typestr="<f4", owned=False):
    return torch.as_tensor(_Buffer(ptr, shape, typestr, owned), device=DEV)


def _alloc(shape, typestr="<f4"):
    n = int(np.prod(shape)) * int(typestr[2:])
    return _view(device.alloc(n), shape, typestr, True)


# The library looks a kernel up in one code object after another, and a miss
# leaves its status for whoever asks next: a program that also uses torch takes
# it out after the call, or torch's next call reports it as its own.
_hip = ctypes.CDLL("libamdhip64.so.7")


def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 7919 + salt)
    return g


# --------------------------------------------------------------------------
# quantized records
# --------------------------------------------------------------------------
def _groups(w):
    """[K, N] -> [groups, 32, N], the last group padded with its own last row."""
    K, N = w.shape
    pad = -K % 32
    return torch.cat([w, w[-1:].expand(pad, N)]).view(-1, 32, N) if pad else w.view(-1, 32, N)


def _q4_fields(w):
    """quantizeQ4: (nibbles [G, 32, N], scale, zero as f64 [G, N]), in f64 with
    round-half-up; rows past K count as weight 0 and not for the range."""
    K, N = w.shape
    g = _groups(w).double()
    mn, mx = g.amin(1), g.amax(1)
    rng = mx - mn
    scale = torch.where(rng > 0, rng / 15.0, torch.ones_like(rng))
    zero = torch.where(rng > 0, -mn / scale, torch.full_like(rng, 8.0))
    if K % 32:
        g[-1, K % 32:] = 0.0
    t = (g / scale[:, None] + zero[:, None]).clamp(0.0, 15.0)
    del g
    q = t.floor()
    q += (t - q >= 0.5).double()
    return q.to(torch.uint8), scale.float(), zero.float()


def _q4_records(w):
    q, scale, zero = _q4_fields(w)
    out = torch.empty(q.shape[0], q.shape[2], 24, dtype=torch.uint8, device=DEV)
    out[..., :16] = (q[:, 0::2] | (q[:, 1::2] << 4)).permute(0, 2, 1)
    out[..., 16:20] = scale[..., None].contiguous().view(torch.uint8)
    out[..., 20:24] = zero[..., None].contiguous().view(torch.uint8)
    return out


def _q4_weight(w):
    """The f64 weights [K, N] that the records of w stand for."""
    q, scale, zero = _q4_fields(w)
    return ((q.double() - zero.double()[:, None]) * scale.double()[:, None]).view(-1, w.shape[1])[:w.shape[0]]


def _q8_fields(w):
    K, N = w.shape
    g = _groups(w).clone()
    if K % 32:
        g[-1, K % 32:] = 0.0
    d = g.abs().amax(1) / 127.0
    q = torch.round(g / torch.where(d > 0, d, torch.ones_like(d))[:, None]).clamp(-127, 127)
    return q.to(torch.int8), d.half()


def _q8_records(w):
    q, d = _q8_fields(w)
    out = torch.empty(q.shape[0], q.shape[2], 34, dtype=torch.uint8, device=DEV)
    out[..., :2] = d[..., None].contiguous().view(torch.uint8)
    out[..., 2:] = q.permute(0, 2, 1).contiguous().view(torch.uint8)
    return out


def _q8_weight(w):
    q, d = _q8_fields(w)
    return (q.double() * d.double()[:, None]).view(-1, w.shape[1])[:w.shape[0]]


def _matrix(case, seed):
    return torch.randn(case["K"], case["N"], generator=_gen(seed, 1), device=DEV) * 0.02


def _activations(case, seed):
    return torch.randn(case["M"], case["K"], generator=_gen(seed, 2), device=DEV)


def _prepare_matmul(case, seed):
    rec = (_q4_records if case["fmt"] == "q4" else _q8_records)(_matrix(case, seed))
    wq = _alloc(rec.shape, "|u1")
    wq.copy_(rec)
    a = _alloc((case["M"], case["K"]))
    a.copy_(_activations(case, seed))
    return {"case": case, "ctx": device.ops_ctx(), "a": a, "wq": wq, "out": _alloc((case["M"], case["N"]))}


def _run_matmul(st):
    c = st["case"]
    entry = device.lib.smith_matmul_q4 if c["fmt"] == "q4" else device.lib.smith_matmul_q8
    device.check(entry(st["ctx"], st["a"].data_ptr(), st["wq"].data_ptr(), st["out"].data_ptr(), c["M"], c["N"],
                       c["K"], (c["K"] + 31) // 32), "matmul")
    if c["M"] >= 64:
        _hip.hipGetLastError()
    return st["out"]


def _prepare_op(case, seed):
    st = _prepare_matmul(case, seed)
    G32 = (case["K"] + 31) // 32
    st["ta"] = S.Tensor([case["M"], case["K"]], "f32", buffer=st["a"].data_ptr())
    st["tq"] = S.QuantizedWeight(buffer=st["wq"].data_ptr(), K=case["K"], N=case["N"], groups=G32,
                                 totalBytes=st["wq"].numel())
    return st


def _run_op(st):
    c = st["case"]
    y = (S.matmulQ4 if c["fmt"] == "q4" else S.matmulQ8)(st["ta"], st["tq"])
    return _view(y.buffer, y.shape, owned=True)  # released with the returned tensor


def _prepare_quantize(case, seed):
    w = _alloc((case["K"], case["N"]))
    w.copy_(_matrix(case, seed))
    return {"case": case, "ctx": device.ops_ctx(), "w": w, "out": _alloc(((case["K"] + 31) // 32, case["N"], 24), "|u1")}


def _run_quantize(st):
    c = st["case"]
    device.check(device.lib.smith_quantize_q4(st["ctx"], st["w"].data_ptr(), st["out"].data_ptr(), c["K"], c["N"]),
                 "quantizeQ4")
    return st["out"]


# --------------------------------------------------------------------------
# Llama-shaped GGUF models of random blocks
# --------------------------------------------------------------------------
_BYTES = {"Q4_0": (32, 18), "Q4_K": (256, 144), "Q6_K": (256, 210)}


def _blocks(kind, n, seed, salt):
    """n elements of random blocks, weights of about N(0, 0.02): uint8 on the GPU."""
    g = _gen(seed, salt)
    per, size = _BYTES[kind]
    nb = n // per
    b = torch.randint(0, 256, (nb, size), generator=g, device=DEV, dtype=torch.uint8)
    u = torch.rand(nb, 1, generator=g, device=DEV) + 0.5
    if kind == "Q4_0":
        b[:, 0:2] = (u * 0.0043).half().view(torch.uint8)
    elif kind == "Q4_K":
        # every sub-block's min is its scale and dmin = 7.5 d: weights of zero mean
        d = (u * 1.0e-4).half()
        b[:, 0:2] = d.view(torch.uint8)
        b[:, 2:4] = (d.float() * 7.5).half().view(torch.uint8)
        b[:, 8:12] = b[:, 4:8]
        lo = b[:, 12:16] & 0x0F
        b[:, 12:16] = lo | (lo << 4)
    else:
        b[:, 208:210] = (u * 1.5e-5).half().view(torch.uint8)
    return b


def _f16(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).double()


def _nibbles(b):
    return torch.stack([b & 0x0F, b >> 4], -1).view(b.shape[0], -1)


def _dequant(kind, b):
    """The blocks' weights in f64, flat."""
    if kind == "Q4_0":
        return ((_nibbles(b[:, 2:18]).double() - 8.0) * _f16(b, 0)).view(-1)
    if kind == "Q4_K":
        s = b[:, 4:16].int()
        lo_s, lo_m = s[:, 0:4] & 63, s[:, 4:8] & 63
        hi_s = (s[:, 0:4] >> 6) | ((s[:, 8:12] & 15) << 2)
        hi_m = (s[:, 4:8] >> 6) | ((s[:, 8:12] >> 4) << 2)
        sc = (_f16(b, 0) * torch.cat([lo_s, hi_s], 1).double()).float().double()
        mn = (_f16(b, 2) * torch.cat([lo_m, hi_m], 1).double()).float().double()
        q = _nibbles(b[:, 16:144]).view(-1, 8, 32).double()
        return (q * sc[..., None] - mn[..., None]).view(-1)
    ql = _nibbles(b[:, 0:128]).int()
    qh = b[:, 128:192].int()
    qh = torch.stack([(qh >> (2 * i)) & 3 for i in range(4)], -1).view(-1, 256)
    sc = b[:, 192:208].contiguous().view(torch.int8).double() * _f16(b, 208)
    return ((ql | (qh << 4)).view(-1, 16, 16) - 32).double().mul(sc[..., None]).view(-1)


def _tensors(case):
    """[(name, listed shape, block type, salt)] of the model's quantized tensors."""
    km = case["mix"] == "q4_k_m"
    low, high = ("Q4_K", "Q6_K") if km else ("Q4_0", "Q4_0")
    dim, ffn, kvd, vocab = case["dim"], case["ffn"], case["dim"] // case["heads"] * case["kv"], case["vocab"]
    out = [("token_embd.weight", [vocab, dim], low, 11), ("output.weight", [dim, vocab], high, 12)]
    for L in range(case["layers"]):
        p = "blk.%d." % L
        for i, (name, n, k, kind) in enumerate((
                ("attn_q", dim, dim, low), ("attn_k", kvd, dim, low), ("attn_v", kvd, dim, high),
                ("attn_output", dim, dim, low), ("ffn_gate", ffn, dim, low), ("ffn_up", ffn, dim, low),
                ("ffn_down", dim, ffn, high))):
            out.append((p + name + ".weight", [n, k], kind, 100 + 10 * L + i))
    return out


def _norms(case, seed):
    g = _gen(seed, 13)
    names = ["output_norm.weight"] + ["blk.%d.%s.weight" % (L, n) for L in range(case["layers"])
                                      for n in ("attn_norm", "ffn_norm")]
    return {n: 1.0 + 0.02 * torch.randn(case["dim"], generator=g, device=DEV) for n in names}


def _context(case):
    # rotary tables as long as the reference's row indexing needs, 8192 as the usual file says
    return max(8192, (case["tokens"] + 1) * case["heads"])


def _tokens(case, seed):
    n = case["tokens"] + (1 if case["kind"] == "decode" else 0)
    return torch.randint(0, case["vocab"], (n,), generator=_gen(seed, 14), device=DEV).tolist()


def _load(case, seed):
    T = G.GGUF_TYPE
    meta = {"general.architecture": (T["STRING"], "llama"), "general.alignment": (T["UINT32"], 32)}
    for k, v in (("embedding_length", case["dim"]), ("block_count", case["layers"]),
                 ("attention.head_count", case["heads"]), ("attention.head_count_kv", case["kv"]),
                 ("context_length", _context(case)), ("feed_forward_length", case["ffn"]),
                 ("vocab_size", case["vocab"])):
        meta["llama." + k] = (T["UINT32"], v)
    meta["llama.rope.freq_base"] = (T["FLOAT32"], 10000.0)
    meta["llama.attention.layer_norm_rms_epsilon"] = (T["FLOAT32"], 1e-5)
    tensors = []
    for name, shape, kind, salt in _tensors(case):
        n = shape[0] * shape[1]
        per, size = _BYTES[kind]
        tensors.append((name, shape, G.GGML_TYPE[kind], n // per * size,
                        lambda kind=kind, n=n, salt=salt: _blocks(kind, n, seed, salt).cpu().numpy().ravel()))
    for name, g in _norms(case, seed).items():
        tensors.append((name, [case["dim"]], G.GGML_TYPE["F32"], case["dim"] * 4, lambda g=g: g.cpu().numpy()))
    fd, path = tempfile.mkstemp(suffix=".gguf")
    os.close(fd)
    try:
        G.write_gguf(path, meta, tensors)
        return loadGGUF(path)
    finally:
        os.unlink(path)


def _prepare_model(case, seed):
    m = _load(case, seed)
    _hip.hipGetLastError()
    caches = m.createCache()
    tokens = _tokens(case, seed)
    n = case["tokens"]
    shape = (case["kv"], _context(case), case["dim"] // case["heads"])
    kv = []
    for c in caches:
        pair = [_view(c[x].ptr, shape) for x in ("k", "v")]
        for t in pair:
            t.zero_()
        kv.append([t[:, :n] if case["kind"] == "prefill" else t[:, n:n + 1] for t in pair])
    torch.cuda.synchronize()
    if case["kind"] == "decode":
        m.forwardPrefill(tokens[:n], caches)
    _hip.hipGetLastError()
    return {"case": case, "model": m, "caches": caches, "tokens": tokens, "kv": kv}


def _run_model(st):
    c, m = st["case"], st["model"]
    if c["kind"] == "prefill":
        r = m.forwardPrefill(st["tokens"], st["caches"])
    else:
        r = m.forwardDecode(st["tokens"][-1], c["tokens"], st["caches"])
    _hip.hipGetLastError()
    return {"logits": r["logits"], "kv": st["kv"]}


def _rope64(x, case):
    """Whole-row rotation of rows at positions 0 ..: element i pairs with
    i + W/2 and takes entry pos * (W/2) + i of the flat tables."""
    n, W = x.shape
    hd = case["dim"] // case["heads"]
    f = (1.0 / np.power(10000.0, 2.0 * np.arange(hd // 2) / hd)).astype(np.float32).astype(np.float64)
    ang = torch.arange(_context(case), dtype=torch.float64)[:, None] * torch.from_numpy(f)[None]
    rows = n * (W // 2)
    cos, sin = (t.float().double().reshape(-1)[:rows].view(n, W // 2).to(DEV) for t in (ang.cos(), ang.sin()))
    a, b = x[:, :W // 2], x[:, W // 2:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], 1)


def _exact_model(case, seed):
    dim, nh, nkv, vocab = case["dim"], case["heads"], case["kv"], case["vocab"]
    hd = dim // nh
    where = {t[0]: t for t in _tensors(case)}
    norms = {k: v.double() for k, v in _norms(case, seed).items()}

    def weight(name):
        _, shape, kind, salt = where[name]
        return _dequant(kind, _blocks(kind, shape[0] * shape[1], seed, salt)).view(shape)

    def norm(x, name):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * norms[name]

    tokens = torch.tensor(_tokens(case, seed), device=DEV)
    n = len(tokens)
    x = weight("token_embd.weight").float().double()[tokens]
    mask = torch.full((n, n), -math.inf, dtype=torch.float64, device=DEV).triu(1)
    kv = []
    for L in range(case["layers"]):
        p = "blk.%d." % L
        h = norm(x, p + "attn_norm.weight")
        q, k, v = (h @ weight(p + "attn_%s.weight" % s).t() for s in "qkv")
        q, k = _rope64(q, case), _rope64(k, case)
        k, v = (t.view(n, nkv, hd).permute(1, 0, 2).contiguous() for t in (k, v))
        kv.append([t[:, :n] if case["kind"] == "prefill" else t[:, n - 1:] for t in (k, v)])
        out = torch.empty(n, dim, dtype=torch.float64, device=DEV)
        for i in range(nh):
            s = q[:, i * hd:(i + 1) * hd] @ k[i // (nh // nkv)].t().contiguous() / math.sqrt(hd) + mask
            out[:, i * hd:(i + 1) * hd] = torch.softmax(s, -1) @ v[i // (nh // nkv)]
        x = x + out @ weight(p + "attn_output.weight").t()
        h = norm(x, p + "ffn_norm.weight")
        g = h @ weight(p + "ffn_gate.weight").t()
        u = h @ weight(p + "ffn_up.weight").t()
        x = x + (g / (1.0 + torch.exp(-g)) * u) @ weight(p + "ffn_down.weight").t()
    if case["kind"] == "decode":
        x = x[-1:]
    # output.weight's flat data is read as [dim, vocab]
    return {"logits": norm(x, "output_norm.weight") @ weight("output.weight").view(dim, vocab), "kv": kv}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        st = _prepare_model(case, seed)
    else:
        st = {"op": _prepare_op, "matmul": _prepare_matmul, "quantize": _prepare_quantize}[kind](case, seed)
    torch.cuda.synchronize()  # the library works on a stream of its own
    return st


def run(state):
    kind = state["case"]["kind"]
    if kind == "matmul":
        return _run_matmul(state)
    if kind == "op":
        return _run_op(state)
    if kind == "quantize":
        return _run_quantize(state)
    return _run_model(state)


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize":
        return _q4_records(_matrix(case, seed))
    if kind in ("op", "matmul"):
        w = (_q4_weight if case["fmt"] == "q4" else _q8_weight)(_matrix(case, seed))
        return _activations(case, seed).double() @ w
    return _exact_model(case, seed)


def work(case):
    kind = case["kind"]
    if kind in ("op", "matmul"):
        M, N, K = case["M"], case["N"], case["K"]
        rec = (K + 31) // 32 * N * (24 if case["fmt"] == "q4" else 34)
        return {"bytes": rec + 4 * M * (K + N), "flops": 2 * M * N * K}
    if kind == "quantize":
        N, K = case["N"], case["K"]
        return {"bytes": 4 * N * K + (K + 31) // 32 * N * 24, "flops": 0}
    rows = case["tokens"] if kind == "prefill" else 1
    dim, vocab, kvd = case["dim"], case["vocab"], case["dim"] // case["heads"] * case["kv"]
    bytes_, flops = 0, 0
    for name, shape, block, _ in _tensors(case):
        per, size = _BYTES[block]
        if name == "token_embd.weight":
            bytes_ += rows * dim * 4  # the rows looked up, f32 on the device
            continue
        bytes_ += shape[0] * shape[1] // per * size
        flops += 2 * rows * shape[0] * shape[1]
    past = case["tokens"]
    seen = past * (past + 1) / 2 if kind == "prefill" else past + 1
    flops += case["layers"] * 4 * dim * seen
    bytes_ += case["layers"] * 2 * kvd * 4 * (past + (1 if kind == "decode" else 0))
    return {"bytes": bytes_ + rows * vocab * 4, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind in ("op", "matmul"):
        # up to 8 rows: f32 activations (as two f16 parts), exact weights, f32
        # sums; one or two rows take the slot offsets off the f32 sums
        if case["M"] <= 2:
            return {"rel": 1e-4, "max": 1e-3}
        if case["M"] <= 8:
            return {"rel": 1e-5, "max": 1e-4}
        # f16 activations on exact weights; 64 rows up f16 weights as well
        return {"rel": 2e-3, "max": 2e-2}
    # a whole model: the f16 operands of the prompt's GEMMs through every layer
    return {"rel": 2e-2, "max": 2e-1}
