"""The framework's work, as measurable cases through its public entry points.

What a user has the library do, from a tiny model's few tokens to an 8B-shaped
prompt: whole calls of the runner (a prompt and its logits, a prompt and
forced decode steps), and the single layers a program calls through the
dispatch entry points (GEMV, FFN, paged attention, prefill GEMM, routed
experts, sampler).  Shapes are the Llama-3.1-8B-shaped, Mixtral-8x7B-shaped
and tiny configurations of the benchmark and the tests.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

PKG = Path(__file__).resolve().parent.parent / "nexus-inference-engine-_amd"
if str(PKG) not in sys.path:
    sys.path.insert(0, str(PKG))

import nexus_amd  # noqa: E402

TINY = dict(d_model=256, n_heads=4, n_kv_heads=2, head_dim=64, ffn=688, vocab=4096, n_experts=0, top_k=0,
            rope_theta=10000.0)
LLAMA = dict(d_model=4096, n_heads=32, n_kv_heads=8, head_dim=128, ffn=14336, vocab=128256, n_experts=0, top_k=0,
             rope_theta=500000.0)
MIXTRAL = dict(LLAMA, vocab=32000, n_experts=8, top_k=2, rope_theta=1000000.0)
SHAPES = {"tiny": TINY, "llama": LLAMA, "mixtral": MIXTRAL}
EPS = 1e-5
KV_FP16, KV_TQ = 0, 1


# ------------------------------------------------------------------- cases --
def listed():
    return [
        # a tiny model answers a short prompt: every launch is latency
        dict(name="tiny_generate", kind="model", model="tiny", layers=2, kv=KV_FP16, batch=1, prompt=16, steps=32),
        # one user's request on the 8B shape (8 of its 32 layers): a chat
        # prompt, then tokens one by one
        dict(name="llama_generate", kind="model", model="llama", layers=8, kv=KV_FP16, batch=1, prompt=300, steps=24),
        # a long document read at once (4 layers): time to the first token
        dict(name="llama_prompt", kind="model", model="llama", layers=4, kv=KV_FP16, batch=1, prompt=2048, steps=0),
        # the QKV projection of one sequence: the smallest call
        dict(name="gemv_qkv", kind="gemv", N=6144, K=4096, batch=1, out="f16"),
        # the FFN of a decode step, one sequence and a full batch
        dict(name="ffn_b1", kind="ffn", d=4096, F=14336, batch=1),
        dict(name="ffn_b8", kind="ffn", d=4096, F=14336, batch=8),
        # decode attention of a full batch with ragged 4K contexts, fp16 pages
        dict(name="attn_f16_b8", kind="attn_f16", batch=8, hq=32, hkv=8, hd=128, ctx=4096, alloc=True),
        # decode attention of one long conversation, TurboQuant pages
        dict(name="attn_tq_32k", kind="attn_tq", batch=1, hq=32, hkv=8, ctx=32768),
        # a prompt chunk's gate/up projection
        dict(name="gemm_chunk", kind="gemm", M=2048, N=28672, K=4096),
        # a short prompt's down projection (and a routed expert's share of a chunk)
        dict(name="gemm_short", kind="gemm", M=100, N=4096, K=14336),
        # routed experts of a decode step, full batch
        dict(name="moe_ffn_b8", kind="moe_ffn", d=4096, F=14336, E=8, k=2, batch=8),
        # sampling the next token of a full batch
        dict(name="sample_b8", kind="sample", V=128256, batch=8, temperature=0.7, top_k=40, top_p=0.9),
    ]


def _log(rng, lo, hi):
    """A whole number, its logarithm uniform over [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _k_of(rng, lo, hi):
    """A contraction length: whole groups of 32 mostly, sometimes a ragged last group."""
    k = _log(rng, lo, hi)
    return k // 8 * 8 if rng.random() < 0.3 else max(lo, k // 32 * 32)


def draw(rng):
    kind = rng.choice(["model", "model", "gemv", "ffn", "attn_f16", "attn_tq", "gemm", "gemm", "moe_ffn", "sample"])
    if kind == "model":
        name = rng.choice(["tiny", "llama", "llama", "mixtral"])
        batch = rng.choice([1, 1, 2, 3, 8]) if name == "tiny" else rng.choice([1, 1, 2, 4])
        layers = {"tiny": 2, "llama": rng.choice([1, 2, 3]), "mixtral": 1}[name]
        steps = rng.choice([0, 0, _log(rng, 1, 16)])
        prompt = _log(rng, 4, 2048 // batch) if name != "tiny" else _log(rng, 4, 512)
        kv = rng.choice([KV_FP16, KV_FP16, KV_TQ]) if name == "llama" else KV_FP16
        return dict(kind=kind, model=name, layers=layers, kv=kv, batch=batch, prompt=prompt, steps=steps)
    if kind == "gemv":
        K = _k_of(rng, 256, 14336)
        return dict(kind=kind, N=_log(rng, 256, min(131072, 530_000_000 // K)), K=K, batch=rng.randint(1, 8),
                    out=rng.choice(["f16", "f32"]))
    if kind == "ffn":
        d = _k_of(rng, 256, 8192)
        return dict(kind=kind, d=d, F=_k_of(rng, 688, min(28672, 90_000_000 // d)), batch=rng.randint(1, 8))
    if kind == "attn_f16":
        hkv, batch, hd = rng.choice([1, 2, 4, 8]), rng.randint(1, 8), rng.choice([64, 128, 128, 256])
        return dict(kind=kind, batch=batch, hq=hkv * rng.choice([1, 2, 4, 4, 8]), hkv=hkv, hd=hd,
                    ctx=_log(rng, 64, min(32768, 8 * 4096 * 8 * 128 // (batch * hkv * hd))), alloc=rng.random() < 0.5)
    if kind == "attn_tq":
        hkv, batch = rng.choice([1, 2, 4, 8]), rng.randint(1, 8)
        return dict(kind=kind, batch=batch, hq=hkv * rng.choice([1, 2, 4, 4, 8]), hkv=hkv,
                    ctx=_log(rng, 64, 32768 * 8 // max(8, batch * hkv)))
    if kind == "gemm":
        M, K = _log(rng, 9, 2048), _k_of(rng, 256, 14336)
        return dict(kind=kind, M=M, N=_log(rng, 256, min(28672, 117_000_000 // K)), K=K)
    if kind == "moe_ffn":
        d, E = _k_of(rng, 512, 4096), rng.choice([4, 8, 16])
        return dict(kind=kind, d=d, F=_k_of(rng, 512, min(14336, 470_000_000 // (E * d))), E=E, k=rng.randint(1, 4),
                    batch=rng.randint(1, 8))
    T = rng.choice([0.0, 0.7, 0.7, 1.0])
    return dict(kind=kind, V=_log(rng, 4096, 256000), batch=rng.randint(1, 8), temperature=T,
                top_k=rng.choice([0, 20, 40, 40, 200]), top_p=rng.choice([0.9, 0.95, 1.0]))


# ------------------------------------------------------- buffers and inputs --
_CTX = None


def context():
    """The process's one context, as a program keeps it."""
    global _CTX
    if _CTX is None:
        _CTX = nexus_amd.Context(0)
    return _CTX


class Buffer:
    """A library buffer given back with its last user; t is a torch view of it."""

    _TYPES = {torch.float32: "<f4", torch.float16: "<f2", torch.uint8: "|u1", torch.int32: "<i4"}

    def __init__(self, shape, dtype, value=None):
        self.ctx = context()
        n = math.prod(shape) * torch.empty((), dtype=dtype).element_size()
        self.id = self.ctx.alloc(n)
        self.ctx.sync()
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=self._TYPES[dtype], data=(self.id, False),
                                             version=2)
        t = self.t
        if value is not None:
            t.copy_(value.reshape(shape))
            torch.cuda.synchronize()

    @property
    def t(self):
        return torch.as_tensor(self, device="cuda")  # holds a reference to this buffer

    def __del__(self):
        try:
            self.ctx.free(self.id)
        except Exception:
            pass


def _put(value):
    return Buffer(value.shape, value.dtype, value)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 17)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _quantize(w):
    """Symmetric int4 group-32 of w [N][K]: codes 0..15 [N][G*32] and fp16 scales [N][G]."""
    N, K = w.shape
    G = (K + 31) // 32
    w = torch.nn.functional.pad(w, (0, 32 * G - K)).view(N, G, 32)
    s = (w.abs().amax(-1) / 7.0).half()
    sf = s.float().unsqueeze(-1)
    q = torch.where(sf > 0, w / sf, torch.zeros_like(w))
    q = (torch.sign(q) * torch.floor(q.abs() + 0.5)).clamp(-8, 7) + 8
    return q.to(torch.uint8).view(N, 32 * G), s


def _weights(g, N, K, sigma=0.02):
    """N(0, sigma) weights, quantized: codes packed low nibble first, scales."""
    codes, scales = [], []
    step = max(1, (1 << 27) // K)
    for n0 in range(0, N, step):
        q, s = _quantize(_randn(g, min(step, N - n0), K) * sigma)
        codes.append(q[:, 0::2] | (q[:, 1::2] << 4))
        scales.append(s)
    return torch.cat(codes), torch.cat(scales)


def _dequant(codes, scales, K):
    """[N][K] in 64 bits."""
    N = codes.shape[0]
    q = torch.stack((codes & 15, codes >> 4), -1).view(N, -1, 32).double() - 8
    return (q * scales.double().unsqueeze(-1)).view(N, -1)[:, :K]


def _matmul64(x, codes, scales, K):
    """x [M][K] times the weights' transpose in 64 bits, a slab of rows at a time."""
    step = max(1, (1 << 27) // K)
    return torch.cat([x @ _dequant(codes[n:n + step], scales[n:n + step], K).t() for n in range(0, codes.shape[0], step)], 1)


# TurboQuant: Lloyd-Max codebooks for N(0, 1/128), 4 bits on the first 64
# rotated coordinates and 3 on the rest.
def _codebook(bits):
    s, n = 1 / math.sqrt(128), 1 << bits
    c = [-3 * s + 6 * s * (i + 0.5) / n for i in range(n)]
    pdf = lambda x: math.exp(-0.5 * (x / s) ** 2) / (s * math.sqrt(2 * math.pi))  # noqa: E731
    cdf = lambda x: 0.5 * math.erfc(-x / s / math.sqrt(2))  # noqa: E731
    for _ in range(100):
        e = [-10 * s] + [(a + b) / 2 for a, b in zip(c, c[1:])] + [10 * s]
        new = [s * s * (pdf(a) - pdf(b)) / (cdf(b) - cdf(a)) for a, b in zip(e, e[1:])]
        moved = max(abs(a - b) for a, b in zip(new, c))
        c = new
        if moved < 1e-7 * s:
            break
    return torch.tensor(c, dtype=torch.float64, device="cuda")


def _tq_codes(g, n):
    """Codes of n random rotated vectors: [n][128]."""
    y = _randn(g, n, 128).double() / math.sqrt(128)
    out = []
    for part, bits in ((y[:, :64], 4), (y[:, 64:], 3)):
        c = _codebook(bits)
        out.append(torch.bucketize(part.contiguous(), (c[1:] + c[:-1]) / 2))
    return torch.cat(out, 1).to(torch.uint8)


def _tq_pack(q):
    c4 = q[:, 0:64:2] | (q[:, 1:64:2] << 4)
    b = (q[:, 64:].view(-1, 8, 8).int() << (3 * torch.arange(8, device="cuda", dtype=torch.int32))).sum(-1)
    c3 = torch.stack([(b >> (8 * i)) & 255 for i in range(3)], -1).to(torch.uint8).view(-1, 24)
    return c4, c3


def _tq_decode(q, norm, sign):
    """The vectors [n][128] that codes, norms and the rotation's signs stand for, in 64 bits."""
    h = torch.ones(1, 1, dtype=torch.float64, device="cuda")
    for _ in range(7):
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    q = q.long()
    y = torch.cat((_codebook(4)[q[:, :64]], _codebook(3)[q[:, 64:]]), 1)
    return (y @ h) / math.sqrt(128) * sign.double() * norm.double().unsqueeze(1)


def _attn64(q, k, v):
    """softmax(q k^T / sqrt(hd)) v in 64 bits: q [hq][hd], k and v [T][hkv][hd]."""
    hq, hd = q.shape
    hkv = k.shape[1]
    q = q.double().view(hkv, hq // hkv, hd)
    s = q @ k.permute(1, 2, 0).contiguous() / math.sqrt(hd)
    return (torch.softmax(s, -1) @ v.permute(1, 0, 2).contiguous()).view(hq, hd)


def _lens(case):
    """Context lengths of a batch: the longest has ctx positions, the others
    end at different points of the last quarter."""
    c = case["ctx"]
    return [max(1, c - (c * b) // (4 * case["batch"]) - (3 * b) % 16) for b in range(case["batch"])]


# ------------------------------------------------------------------- inputs --
def _inputs(case, seed):
    """The case's inputs as plain tensors, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        M = case["batch"] if kind == "gemv" else case["M"]
        w, s = _weights(g, case["N"], case["K"])
        return dict(x=_randn(g, M, case["K"]).half(), w=w, s=s)
    if kind in ("ffn", "moe_ffn"):
        d, F, B, E = case["d"], case["F"], case["batch"], case.get("E", 1)
        w13, s13 = _weights(g, E * 2 * F, d)
        w2, s2 = _weights(g, E * d, F)
        t = dict(x=_randn(g, B, d).half(), w13=w13, s13=s13, w2=w2, s2=s2)
        if kind == "moe_ffn":
            # a routing of the batch's tokens: the k experts of the largest
            # router logits and their softmax, renormalized
            v, ids = torch.topk(_randn(g, B, E), case["k"], -1)
            t.update(ids=ids.int(), weights=torch.softmax(v, -1))
        return t
    if kind in ("attn_f16", "attn_tq"):
        B, hq, hkv, hd = case["batch"], case["hq"], case["hkv"], case.get("hd", 128)
        mb = (case["ctx"] + 15) // 16
        nb = B * mb
        t = dict(q=_randn(g, B, hq, hd), table=torch.randperm(nb, generator=g, device="cuda").int().view(B, mb),
                 lens=torch.tensor(_lens(case), dtype=torch.int32, device="cuda"))
        if kind == "attn_f16":
            t.update(k=_randn(g, nb, hkv, 16, hd).half(), v=_randn(g, nb, hkv, hd, 16).half())
        else:
            for n in "kv":
                t[n + "q"] = _tq_codes(g, nb * hkv * 16)
                t[n + "c4"], t[n + "c3"] = _tq_pack(t[n + "q"])
                t[n + "n"] = (math.sqrt(128) * (1 + 0.06 * _randn(g, nb * hkv * 16))).half()
                t[n + "s"] = torch.where(_randn(g, 128) < 0, -1.0, 1.0)
        return t
    if kind == "sample":
        # a peaked distribution over the vocabulary, as a model's head gives
        return dict(logits=3.0 * _randn(g, case["batch"], case["V"]))
    r = np.random.default_rng(seed)
    V = SHAPES[case["model"]]["vocab"]
    return dict(prompt=r.integers(0, V, (case["batch"], case["prompt"]), dtype=np.int32),
                tokens=r.integers(0, V, (case["batch"], max(1, case["steps"])), dtype=np.int32))


class State:
    pass


def prepare(case, seed):
    s = State()
    s.case, s.ctx = case, context()
    kind = case["kind"]
    t = _inputs(case, seed)
    if kind == "model":
        cfg = dict(SHAPES[case["model"]], n_layers=case["layers"], batch=case["batch"], kv_kind=case["kv"], eps=EPS,
                   max_seq=(case["prompt"] + case["steps"] + 32) // 16 * 16, seed=int(seed) + 0x5EED)
        s.model = nexus_amd.Model(s.ctx, **cfg)
        s.prompt, s.tokens = t["prompt"], t["tokens"]
        return s
    if kind == "attn_tq":
        t.pop("kq"), t.pop("vq")
    s.buf = {n: _put(v) for n, v in t.items()}
    out = {"gemv": lambda: ((case["batch"], case["N"]), torch.float16 if case.get("out") == "f16" else torch.float32),
           "gemm": lambda: ((case["M"], case["N"]), torch.float32),
           "ffn": lambda: ((case["batch"], case["d"]), torch.float32),
           "moe_ffn": lambda: ((case["batch"], case["d"]), torch.float32),
           "attn_f16": lambda: ((case["batch"], case["hq"], case["hd"]), torch.float16),
           "attn_tq": lambda: ((case["batch"], case["hq"], 128), torch.float16),
           "sample": lambda: ((case["batch"],), torch.int32)}[kind]()
    s.out = Buffer(*out)
    s.view = s.out.t
    return s


def run(s):
    c, ctx = s.case, s.ctx
    kind = c["kind"]
    if kind == "model":
        # each sequence's prompt into its slot, then the batch step by step
        for b in range(c["batch"]):
            s.model.admit(b, s.prompt[b])
        if c["steps"] == 0:
            return s.model.logits()
        return s.model.decode_forced(s.tokens)
    b = {n: v.id for n, v in s.buf.items()}
    y = s.out.id
    if kind == "gemv":
        if c["out"] == "f16":
            ctx.gemv(b["x"], b["w"], b["s"], y, c["N"], c["K"], c["batch"])
        else:
            ctx.gemv_f32(b["x"], b["w"], b["s"], y, c["N"], c["K"], c["batch"])
    elif kind == "gemm":
        ctx.gemm(b["x"], b["w"], b["s"], y, c["M"], c["N"], c["K"])
    elif kind == "ffn":
        ctx.check(ctx.L.nx_ffn_int4_g32(ctx.h, b["x"], b["w13"], b["s13"], b["w2"], b["s2"], y, c["d"], c["F"],
                                        c["batch"], 0), "nx_ffn_int4_g32")
    elif kind == "moe_ffn":
        ctx.check(ctx.L.nx_moe_expert_ffn(ctx.h, b["x"], b["w13"], b["s13"], b["w2"], b["s2"], b["ids"], b["weights"],
                                          y, c["d"], c["F"], c["E"], c["k"], c["batch"], 0), "nx_moe_expert_ffn")
    elif kind == "attn_f16":
        f = ctx.L.nx_attn_decode_paged_f16 if c["alloc"] else ctx.L.nx_attn_decode_paged_f16_noalloc
        mb = (c["ctx"] + 15) // 16
        ctx.check(f(ctx.h, b["q"], b["k"], b["v"], b["table"], b["lens"], y, c["batch"], c["hq"], c["hkv"], c["hd"],
                    mb, c["batch"] * mb), "nx_attn_decode_paged_f16")
    elif kind == "attn_tq":
        mb = (c["ctx"] + 15) // 16
        ctx.check(ctx.L.nx_attn_decode_paged_tq(ctx.h, b["q"], b["kc4"], b["kc3"], b["kn"], b["vc4"], b["vc3"], b["vn"],
                                                b["ks"], b["vs"], b["table"], b["lens"], y, c["batch"], c["hq"],
                                                c["hkv"], mb, c["batch"] * mb), "nx_attn_decode_paged_tq")
    else:
        ctx.sample(b["logits"], y, c["V"], c["batch"], c["temperature"], c["top_k"], c["top_p"], 42)
    return s.view


# --------------------------------------------------------------------- work --
def _w4(N, K):
    """Bytes of an int4 group-32 matrix with its scales."""
    return N * ((K + 31) // 32) * 18


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        M, N, K = case["batch"] if kind == "gemv" else case["M"], case["N"], case["K"]
        return dict(bytes=_w4(N, K) + 2 * M * K + (2 if case.get("out") == "f16" else 4) * M * N, flops=2 * M * N * K)
    if kind == "ffn":
        d, F, B = case["d"], case["F"], case["batch"]
        return dict(bytes=_w4(2 * F, d) + _w4(d, F) + 6 * B * d, flops=6 * B * d * F)
    if kind == "moe_ffn":
        d, F, B, k, E = case["d"], case["F"], case["batch"], case["k"], case["E"]
        active = E * (1 - (1 - k / E) ** B)  # experts that a routing of B tokens reaches
        return dict(bytes=active * (_w4(2 * F, d) + _w4(d, F)) + 6 * B * d, flops=6 * B * k * d * F)
    if kind in ("attn_f16", "attn_tq"):
        n, hd = sum(_lens(case)), case.get("hd", 128)
        per = 4 * hd if kind == "attn_f16" else 116
        return dict(bytes=n * case["hkv"] * per + 6 * case["batch"] * case["hq"] * hd, flops=4 * n * case["hq"] * hd)
    if kind == "sample":
        return dict(bytes=4 * case["V"] * case["batch"], flops=4 * case["V"] * case["batch"])
    c = SHAPES[case["model"]]
    d, F, L, B, P, T, E, k = (c["d_model"], c["ffn"], case["layers"], case["batch"], case["prompt"], case["steps"],
                              c["n_experts"], c["top_k"])
    qd, kvd = c["n_heads"] * c["head_dim"], c["n_kv_heads"] * c["head_dim"]
    attn_w = _w4(qd + 2 * kvd, d) + _w4(d, qd)
    ffn_w = _w4(2 * F, d) + _w4(d, F)
    reach = lambda n: E * (1 - (1 - k / E) ** n) if E else 1  # noqa: E731
    kv = 4 * kvd if case["kv"] == KV_FP16 else 4 * kvd * 58 / 256
    # each prompt reads every weight once and its K and V once, each step
    # the weights and the positions before it
    by = B * (L * (attn_w + reach(P) * ffn_w + P * kv) + _w4(c["vocab"], d))
    by += T * (L * (attn_w + reach(B) * ffn_w + B * (P + T / 2) * kv) + _w4(c["vocab"], d))
    tokens = B * (P + T)
    fl = 2 * tokens * L * ((qd + 2 * kvd) * d + d * qd + 3 * d * F * max(k, 1)) + 2 * B * max(1, T + 1) * c["vocab"] * d
    fl += L * 4 * qd * B * (P * (P + 1) / 2 + T * (P + T / 2))
    return dict(bytes=by, flops=fl)


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "gemm" or (kind == "gemv" and case["out"] == "f32"):
        return dict(rel=2e-6, max=2e-5)  # exact products, 32-bit sums
    if kind == "gemv":
        return dict(rel=2e-4, max=2e-3)  # the result in fp16
    if kind in ("ffn", "moe_ffn"):
        return dict(rel=4e-4, max=4e-3)  # activations in fp16
    if kind == "attn_f16":
        return dict(rel=4e-4, max=4e-3)  # the result in fp16
    if kind == "attn_tq":
        return dict(rel=8e-4, max=8e-3)  # value codebook and result in fp16
    if case["kv"] == KV_TQ:
        return dict(rel=2e-2, max=0.2)   # a K or V code at a boundary may take the next level
    return dict(rel=4e-3, max=4e-2)      # fp16 activations through the layers


# -------------------------------------------------------------------- exact --
def _fmix(z):
    """The splitmix64 finalizer on wrapping 64-bit words."""
    for sh, m in ((30, 0xBF58476D1CE4E5B9), (27, 0x94D049BB133111EB)):
        z = (z ^ ((z >> sh) & ((1 << (64 - sh)) - 1))) * (m - (1 << 64))
    return z ^ ((z >> 31) & ((1 << 33) - 1))


def _signed(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def _normal(seed, tensor, n, sigma, start=0):
    """Elements start..start+n of a synthetic tensor: counter-based draws, the
    sum of four 16-bit fields scaled to sigma."""
    def fmix1(v):
        return int(_fmix(torch.tensor(_signed(v))).item())

    g1, g2 = 0x9E3779B97F4A7C15, 0xD1B54A32D192ED03
    key = fmix1(fmix1(seed + g1) + tensor * g2)
    i = torch.arange(start + 1, start + n + 1, dtype=torch.int64, device="cuda")
    r = _fmix(i * _signed(g1) + _signed(key))
    total = sum((r >> sh) & 0xFFFF for sh in (0, 16, 32, 48))
    k = np.float32(sigma / (2.0 * math.sqrt((65536.0 * 65536.0 - 1.0) / 3.0)))
    return (2 * total - 262140).float() * float(k)


def _model64(case, seed):
    """Logits of the synthetic dense model in 64 bits: its weights quantized
    as stored, nothing rounded after that."""
    c, sd = SHAPES[case["model"]], int(seed) + 0x5EED
    d, F, hd, hq, hkv, V = (c["d_model"], c["ffn"], c["head_dim"], c["n_heads"], c["n_kv_heads"], c["vocab"])
    t = _inputs(case, seed)

    def weight(tensor, N, K):
        step = max(1, (1 << 25) // K)
        parts = []
        for n in range(0, N, step):
            m = min(step, N - n)
            q, s = _quantize(_normal(sd, tensor, m * K, 0.02, n * K).view(m, K))
            parts.append((q[:, 0::2] | (q[:, 1::2] << 4), s))
        return torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts]), K

    def norm(x):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)

    prompt = torch.from_numpy(t["prompt"]).cuda().long()
    ids = torch.cat((prompt, torch.from_numpy(t["tokens"]).cuda().long()), 1) if case["steps"] else prompt
    B, S = ids.shape
    embed = torch.empty(V, d, dtype=torch.float16, device="cuda")
    step = max(1, (1 << 25) // d)
    for v in range(0, V, step):
        n = min(step, V - v)
        embed[v:v + n] = _normal(sd, 1, n * d, 0.02, v * d).half().view(n, d)
    h = embed[ids].double().view(B * S, d)
    del embed
    ang = torch.arange(S, device="cuda").double()[:, None] * c["rope_theta"] ** (
        -2.0 * torch.arange(hd // 2, device="cuda").double() / hd)
    cs, sn = ang.cos()[None, :, None, :], ang.sin()[None, :, None, :]

    def rope(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack((a * cs - b * sn, a * sn + b * cs), -1).flatten(-2)

    mask = torch.ones(S, S, dtype=torch.bool, device="cuda").tril()
    for L in range(case["layers"]):
        tid = 0x100 * (L + 1)
        x = norm(h)
        q = rope(_matmul64(x, *weight(tid, hq * hd, d)).view(B, S, hq, hd))
        k = rope(_matmul64(x, *weight(tid + 1, hkv * hd, d)).view(B, S, hkv, hd))
        v = _matmul64(x, *weight(tid + 2, hkv * hd, d)).view(B, S, hkv, hd)
        att = torch.empty_like(q)
        for b in range(B):
            for i in range(hq):
                j = i // (hq // hkv)
                s = (q[b, :, i] @ k[b, :, j].t().contiguous() / math.sqrt(hd)).masked_fill(~mask, -math.inf)
                att[b, :, i] = torch.softmax(s, -1) @ v[b, :, j].contiguous()
        h = h + _matmul64(att.reshape(B * S, hq * hd), *weight(tid + 3, d, hq * hd))
        x = norm(h)
        a = torch.nn.functional.silu(_matmul64(x, *weight(tid + 4, F, d))) * _matmul64(x, *weight(tid + 5, F, d))
        h = h + _matmul64(a, *weight(tid + 6, d, F))
    h = h.view(B, S, d)
    last = h[:, case["prompt"]:] if case["steps"] else h[:, -1:]
    y = _matmul64(norm(last.reshape(-1, d)), *weight(2, V, d)).view(B, -1, V)
    return (y if case["steps"] else y[:, 0]).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None  # whole numbers
    if kind == "model":
        # compressed pages and expert choices are decisions, which have no
        # 64-bit value of their own
        if case["kv"] != KV_FP16 or SHAPES[case["model"]]["n_experts"]:
            return None
        return _model64(case, seed)
    t = _inputs(case, seed)
    if kind in ("gemv", "gemm"):
        return _matmul64(t["x"].double(), t["w"], t["s"], case["K"])
    if kind in ("ffn", "moe_ffn"):
        d, F, B, E = case["d"], case["F"], case["batch"], case.get("E", 1)
        w13, s13, w2, s2 = (t[n].view(E, -1, t[n].shape[1]) for n in ("w13", "s13", "w2", "s2"))
        y = torch.zeros(B, d, dtype=torch.float64, device="cuda")
        for e in range(E):
            z = _matmul64(t["x"].double(), w13[e], s13[e], d)
            z = _matmul64(torch.nn.functional.silu(z[:, 0::2]) * z[:, 1::2], w2[e], s2[e], F)
            y += z if kind == "ffn" else z * (t["weights"].double() * (t["ids"] == e)).sum(1, keepdim=True)
        return y
    B, hkv, hd = case["batch"], case["hkv"], case.get("hd", 128)
    if kind == "attn_tq":
        kv = [_tq_decode(t[n + "q"], t[n + "n"], t[n + "s"]).view(-1, hkv, 16, 128) for n in "kv"]
    else:
        kv = [t["k"].double(), t["v"].double().transpose(2, 3)]
    out = []
    for b, n in enumerate(_lens(case)):
        pages = t["table"][b].long()
        k, v = (p[pages].permute(0, 2, 1, 3).reshape(-1, hkv, hd)[:n] for p in kv)
        out.append(_attn64(t["q"][b], k, v))
    return torch.stack(out)
