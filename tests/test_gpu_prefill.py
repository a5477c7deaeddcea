"""Batched prefill on the GPU: the int4-g32 GEMM on the matrix cores against
the oracle, and the whole batched prefill (GEMMs, RoPE + page writes,
causal attention, last-token lm_head) against the one-token-per-step
prefill of the reference's loop (hybrid_model.cpp:604-644) and the oracle's
greedy tokens."""
import ctypes as C
import re

import numpy as np
import pytest

import nexus_amd
import oracle
from conftest import TQ_DECODE_TIE, TQ_DECODE_TOL, rel_err
from test_gpu_model import TINY, assert_greedy_parity

pytestmark = pytest.mark.gpu


def _gemm_case(ctx, M, N, K, seed, accumulate=False):
    rng = np.random.default_rng(seed)
    codes, scales = oracle.gen_quant_rows(0, N, K, seed, 0x77, 0.02)
    x = rng.standard_normal((M, K)).astype(np.float16)
    y0 = rng.standard_normal((M, N)).astype(np.float32) if accumulate else np.zeros((M, N), np.float32)
    bx, bw, bs = ctx.upload(x.view(np.uint16)), ctx.upload(codes), ctx.upload(scales)
    by = ctx.upload(y0)
    ctx.gemm(bx, bw, bs, by, M, N, K, accumulate)
    got = ctx.download(by, (M, N), np.float32)
    for b in (bx, bw, bs, by):
        ctx.free(b)
    want = oracle.gemv(codes, scales, x.astype(np.float32), N, K) + (y0 if accumulate else 0)
    return got, want


@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (7, 100, 256), (128, 64, 688), (130, 200, 256), (200, 256, 4096),
                                   (64, 1000, 14336)])
def test_gemm_matches_oracle(ctx, M, N, K):
    """Ragged M (tokens), N (rows) and K (a last group of 16 k at 688) against
    the oracle's GEMV of each row (exact int4 x fp16 products, fp32 sums:
    only the summation order differs), relative error bound 1e-3."""
    got, want = _gemm_case(ctx, M, N, K, seed=M * 7 + N)
    e = rel_err(got, want)
    print(f"M={M} N={N} K={K} rel_err={e:.2e}")
    assert e < 1e-3


def test_gemm_accumulates(ctx):
    got, want = _gemm_case(ctx, 33, 96, 512, seed=5, accumulate=True)
    assert rel_err(got, want) < 1e-3


@pytest.mark.parametrize("M,N,K,acc", [(1024, 8192, 512, False), (2048, 4096, 256, True), (1000, 8200, 688, False)])
def test_gemm_wide_tiles_matches_oracle(ctx, M, N, K, acc):
    """Products that fill the chip with one launch of 128 x 256 tiles, and
    of 64 x 256 where K is ragged: exact tiles, ragged M and N, a last group
    of 16 k, the accumulating epilogue."""
    got, want = _gemm_case(ctx, M, N, K, seed=M + N + K, accumulate=acc)
    e = rel_err(got, want)
    print(f"M={M} N={N} K={K} rel_err={e:.2e}")
    assert e < 1e-3


@pytest.mark.parametrize("M,N,K", [(64, 28672, 4096), (64, 4096, 14336)])
def test_gemm_8b_shapes(ctx, M, N, K):
    """The 8B gate/up and down shapes with 64 tokens."""
    got, want = _gemm_case(ctx, M, N, K, seed=N)
    assert rel_err(got, want) < 1e-3


@pytest.mark.parametrize("M,N,K,acc", [
    (300, 28672, 512, False),    # 256 x 256 tiles, a ragged second token tile
    (600, 28929, 1024, True),    # 256 x 256 tiles over whole rounds, the last columns (ragged) as 128 x 256
    (464, 16389, 1024, True),    # 128 x 256 tiles, five last columns with K in parts
    (514, 29064, 640, False),    # 256 x 256 tiles, the last columns as 32 x 256
    (520, 28672, 1024, False),   # 64 x 256 tiles, in two launches
    (33, 258, 256, True),        # 32 x 256 tiles, both edges ragged
    (128, 300, 8192, True),      # K in 16 parts
    (40, 300, 16384, True),      # K in 32 parts
    (300, 8, 4096, False),       # fewer weight rows than a wavefront takes
    (65, 1000, 4104, False),     # a last group of 8 k, an odd number of stages, K in parts
    (1000, 1001, 2056, True),    # the same with scalar part sums
    (200, 260, 136, False),      # one pair of stages, 8 k of the second
    (9, 300, 1000, False),       # 31 whole groups and 8 k
])
def test_gemm_tile_shapes_and_k_parts(ctx, M, N, K, acc):
    """Every tile shape, K split and column cut the launch chooses between,
    at ragged edges, for a sample of the tokens with every tile's first and
    last among them.  Products are exact and sums fp32 on both sides, in
    orders of their own: each is within about sqrt(K) roundings of 2^-24 of
    the sum, at most 1.6e-5 together at K = 16384."""
    rng = np.random.default_rng(M + N + K)
    codes, scales = oracle.gen_quant_rows(0, N, K, 11, 0x77, 0.02)
    x = rng.standard_normal((M, K)).astype(np.float16)
    y0 = rng.standard_normal((M, N)).astype(np.float32)
    bx, bw, bs, by = ctx.upload(x.view(np.uint16)), ctx.upload(codes), ctx.upload(scales), ctx.upload(y0)
    ctx.gemm(bx, bw, bs, by, M, N, K, acc)
    got = ctx.download(by, (M, N), np.float32)
    for b in (bx, bw, bs, by):
        ctx.free(b)
    rows = sorted({r for t in range(0, M, 32) for r in (t, min(t + 31, M - 1))} if N < 4096 else
                  {0, 31, 32, 63, 64, 127, 128, 255, 256, M - 1})
    want = oracle.gemv(codes, scales, x[rows].astype(np.float32), N, K) + (y0[rows] if acc else 0)
    assert rel_err(got[rows], want) < 2e-5
    assert np.isfinite(got).all()


@pytest.mark.parametrize("M,N,K", [(40, 520, 520), (300, 256, 4096)])
def test_gemm_keeps_tokens_apart(ctx, M, N, K):
    """Infinities and NaN in one token's x stay in its row, also where a
    stage reads past K and a tile past the last token."""
    rng = np.random.default_rng(K)
    codes, scales = oracle.gen_quant_rows(0, N, K, 12, 0x77, 0.02)
    x = rng.standard_normal((M, K)).astype(np.float16)
    bw, bs, by = ctx.upload(codes), ctx.upload(scales), ctx.upload(np.zeros((M, N), np.float32))
    res = []
    for bad in (False, True):
        if bad:
            x[17], x[M - 1, 3] = np.inf, np.nan
        bx = ctx.upload(x.view(np.uint16))
        ctx.gemm(bx, bw, bs, by, M, N, K, False)
        res.append(ctx.download(by, (M, N), np.float32))
        ctx.free(bx)
    for b in (bw, bs, by):
        ctx.free(b)
    rest = [r for r in range(M) if r not in (17, M - 1)]
    assert np.array_equal(res[0][rest], res[1][rest])
    assert not np.isfinite(res[1][[17, M - 1]]).any()


def _cus(ctx):
    """Compute units, from nx_device_name's "(gfx950, N CUs)"."""
    return int(re.search(r"(\d+) CUs", ctx.device_name()).group(1))


@pytest.mark.parametrize("hq,hkv,hd,parts", [
    (32, 8, 128, [1.1]), (64, 8, 128, [1.1, 1.05]), (32, 16, 128, [1.1]), (32, 32, 128, [0.1, 1.2]),
    (64, 16, 64, [1.2]), (64, 8, 64, [1.1, 1.1]), (64, 32, 64, [1.05]), (64, 64, 64, [1.1])])
def test_long_prompt_attention_paths_agree(ctx, hq, hkv, hd, parts):
    """Prompts long enough for the attention that takes its pages through
    LDS (1, 2, 4 and 8 heads per kv head of 64 and of 128; ragged last tiles; a
    second prompt that starts inside a page behind the first), against the
    same tokens in prompts of 64, which take the other kernel: the two
    compute the same products in the same order, so logits differ only by what
    the GEMMs' orders of sums make of fp16 activations.  The LDS kernel takes
    a prompt when hq * ceil(tokens / 16) exceeds 4, 6 or 8 wavefronts per
    compute unit (parts: the prompts in multiples of that line, odd)."""
    G = hq // hkv
    per_cu = 8 if hd == 64 or G == 8 else 4 if G == 4 else 6
    line = per_cu * _cus(ctx) // hq * 16
    chunks = [int(p * line) | 1 for p in parts]
    assert max(chunks) <= 2048 and 64 < line < max(chunks)
    cfg = dict(TINY, n_layers=1, d_model=512, n_heads=hq, n_kv_heads=hkv, head_dim=hd, max_seq=4416, batch=1, kv_kind=0)
    toks = np.random.default_rng(hq + hd).integers(0, cfg["vocab"], (1, sum(chunks)), dtype=np.int32)
    res = []
    for sizes in (chunks, [64] * (sum(chunks) // 64) + ([sum(chunks) % 64] if sum(chunks) % 64 else [])):
        m = nexus_amd.Model(ctx, **cfg)
        at = 0
        for n in sizes:
            m.prefill(np.ascontiguousarray(toks[:, at:at + n]))
            at += n
        res.append(m.logits())
        m.close()
    assert rel_err(res[0], res[1]) < 2e-3


def oracle_script(cfg, script):
    """Greedy tokens and top1-top2 margins of the oracle for a script of
    ("prompt", [B][P]) and ("decode", n) entries: a prompt is run token by
    token and yields its last token's successor; decode steps feed back."""
    om = oracle.Model(**cfg)
    toks, margins, pending, plog = [], [], None, []
    for kind, v in script:
        steps = [v[:, i].copy() for i in range(v.shape[1])] if kind == "prompt" else [None] * v
        for j, t in enumerate(steps):
            lg = om.forward(np.ascontiguousarray(pending if t is None else t, np.int32))
            if kind == "prompt" and j < len(steps) - 1:
                continue
            if kind == "prompt":
                plog.append(lg)
            pending = np.argmax(lg, axis=1).astype(np.int32)
            part = np.sort(lg, axis=1)
            toks.append(pending.copy())
            margins.append(part[:, -1] - part[:, -2])
    om.close()
    oracle_script.prompt_logits = plog  # logits after each prompt of the last script
    return np.stack(toks, 1), np.stack(margins, 1)


def gpu_script(ctx, cfg, script, batched):
    m = nexus_amd.Model(ctx, **cfg)
    m.set_prefill(batched)
    toks, logits = [], []
    for kind, v in script:
        if kind == "prompt":
            toks.append(m.prefill(v)[:, None])
            logits.append(m.logits())
        else:
            toks.append(m.decode(v))
    pos = m.position(0)
    m.close()
    return np.concatenate(toks, 1), logits, pos


# TurboQuant pages need head_dim 128
TQ = dict(TINY, n_heads=4, n_kv_heads=1, head_dim=128, d_model=512, kv_kind=1)
MOE = dict(TINY, n_experts=4, top_k=2)
# tiered pages with a 16-position window: a page is compressed 31 positions
# after its first, so prompts of 40 tokens and more read TurboQuant pages;
# two kv heads
TIERED = dict(TQ, n_kv_heads=2, kv_kind=2, hot_window=16)
# 256-long heads: the causal attention reads q's operands from LDS
HD256 = dict(TINY, n_heads=4, n_kv_heads=2, head_dim=256, d_model=512)
KINDS = {"fp16": TINY, "turboquant": TQ, "moe": MOE, "tiered": TIERED, "hd256": HD256}
# Logits of the two prefill paths: fp16 pages agree to rounding (1e-3).
# TurboQuant pages quantize K and V, which reach the encoder through GEMM
# (batched) or GEMV (one step per token) summation orders: a value at a
# codebook boundary can take the neighbouring code, moving that element by a
# quantization step and the next layer's input with it.  Such flips add up
# with the prompt: 1-2e-3 on the logits at 17-40 tokens, 7e-3 at 96.  The
# bound is 2e-2: a misplaced position or a wrong vector moves the logits by
# O(1), the stored pages are compared with the oracle's code by code in
# test_batched_prefill_turboquant_pages_match_oracle, and the greedy tokens
# with the oracle's in the tests here.
LOGIT_TOL = {"fp16": 1e-3, "turboquant": 2e-2, "moe": 1e-3, "tiered": 2e-2, "hd256": 1e-3}


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("P", [1, 17, 40])
def test_batched_prefill_matches_token_steps(ctx, P, kind):
    """Batched and one-step-per-token prefill: logits after the prompt within
    1e-3 of each other, and both give the oracle's greedy tokens (ties aside).
    TurboQuant pages: the batched path encodes each chunk into the pages and
    attends over them decoded to fp16.  Tiered pages: each query tile reads
    its pages before its cold boundary decoded from TurboQuant, the rest as
    fp16."""
    cfg = dict(KINDS[kind], seed=0x5EED + P)
    script = [("prompt", oracle.prompt_tokens(cfg["seed"], 1, P, cfg["vocab"])), ("decode", 11)]
    want, margins = oracle_script(cfg, script)
    ta, la, pa = gpu_script(ctx, cfg, script, True)
    tb, lb, pb = gpu_script(ctx, cfg, script, False)
    assert pa == pb == P + 10
    e = rel_err(la[0], lb[0])
    eo = max(rel_err(x[0], oracle_script.prompt_logits[0]) for x in (la, lb))
    print(f"P={P} {kind} logits rel_err={e:.2e}, against the oracle {eo:.2e}")
    assert e < LOGIT_TOL[kind] and eo < LOGIT_TOL[kind]
    assert_greedy_parity(ta, want, margins)
    assert_greedy_parity(tb, want, margins)


def test_batched_prefill_turboquant_8_heads_per_kv(ctx):
    """TurboQuant pages with 8 query heads per kv head (two kv heads; the
    causal attention runs as two blocks of 4 heads per kv head over the same
    decoded pages): batched and one-step prefill logits within the
    TurboQuant bound of each other and of the oracle, and both give the
    oracle's greedy tokens (ties aside)."""
    cfg = dict(TQ, n_heads=16, n_kv_heads=2, seed=0x7A8)
    script = [("prompt", oracle.prompt_tokens(cfg["seed"], 1, 40, cfg["vocab"])), ("decode", 7)]
    want, margins = oracle_script(cfg, script)
    ta, la, pa = gpu_script(ctx, cfg, script, True)
    tb, lb, pb = gpu_script(ctx, cfg, script, False)
    assert pa == pb == 40 + 6
    e = rel_err(la[0], lb[0])
    eo = max(rel_err(x[0], oracle_script.prompt_logits[0]) for x in (la, lb))
    print(f"G=8 turboquant logits rel_err={e:.2e}, against the oracle {eo:.2e}")
    assert e < LOGIT_TOL["turboquant"] and eo < LOGIT_TOL["turboquant"]
    assert_greedy_parity(ta, want, margins)
    assert_greedy_parity(tb, want, margins)


@pytest.mark.parametrize("kind", sorted(KINDS))
def test_batched_prefill_two_chunks_matches_oracle(ctx, kind):
    """A 2100-token prompt (two chunks of the batched path, the second
    attending to pages of the first) and 8 greedy tokens against the
    oracle's token-by-token run; RMSNorm weights not 1."""
    cfg = dict(KINDS[kind], max_seq=2304, seed=0x600, norm_sigma=0.1)
    script = [("prompt", oracle.prompt_tokens(cfg["seed"], 1, 2100, cfg["vocab"])), ("decode", 7)]
    want, margins = oracle_script(cfg, script)
    got, lg, _ = gpu_script(ctx, cfg, script, True)
    e = rel_err(lg[0], oracle_script.prompt_logits[0])
    print(f"{kind} 2100-token prompt: logits rel_err against the oracle {e:.2e}")
    assert e < LOGIT_TOL[kind]
    assert_greedy_parity(got, want, margins)


@pytest.mark.parametrize("kind", sorted(KINDS))
def test_batched_prefill_batch2_and_after_decode(ctx, kind):
    """Two sequences, then a second prompt after decode steps (at positions
    > 0): both prefill modes give the oracle's tokens, and their logits
    after each prompt agree within 1e-3."""
    cfg = dict(KINDS[kind], batch=2, seed=0xB2)
    script = [("prompt", oracle.prompt_tokens(cfg["seed"], 2, 9, cfg["vocab"])), ("decode", 3),
              ("prompt", oracle.prompt_tokens(cfg["seed"] + 1, 2, 21, cfg["vocab"])), ("decode", 6)]
    want, margins = oracle_script(cfg, script)
    ta, la, _ = gpu_script(ctx, cfg, script, True)
    tb, lb, _ = gpu_script(ctx, cfg, script, False)
    assert_greedy_parity(ta, want, margins)
    assert_greedy_parity(tb, want, margins)
    for x, y in zip(la, lb):
        e = rel_err(x, y)
        print(f"{kind} logits rel_err={e:.2e}")
        assert e < LOGIT_TOL[kind]
    # against the oracle: after the first prompt, and after the second where
    # the tokens decoded between them were the oracle's
    plog = oracle_script.prompt_logits
    assert rel_err(la[0], plog[0]) < LOGIT_TOL[kind]
    if np.array_equal(ta[:, :4], want[:, :4]):
        assert rel_err(la[1], plog[1]) < LOGIT_TOL[kind]


@pytest.mark.parametrize("kv_kind", [0, 1, 2])
def test_batched_prefill_8b_layer_shape(ctx, kv_kind):
    """Two layers of the 8B shape (d 4096, 32/8 heads of 128, FFN 14336,
    vocab 128256), a 96-token prompt: batched and one-step prefill agree on
    the logits within 1e-3 (fp16 pages; TurboQuant pages: 2e-2) and on the
    next token unless it is a tie.  Tiered pages (32-position window): each
    run compresses its own positions, whose K and V reach the encoder through
    GEMM (batched) or GEMV (one step) sums, so code flips add up on both
    sides (measured against the oracle: one step 1.7-2.2e-2, batched
    0.25-1.1e-2, windows 16-64); the batched logits are held to the oracle's
    within TQ_DECODE_TOL, its token to the oracle's beyond TQ_DECODE_TIE."""
    cfg = dict(n_layers=2, d_model=4096, n_heads=32, n_kv_heads=8, head_dim=128, ffn=14336, vocab=128256,
               n_experts=0, top_k=0, max_seq=256, batch=1, kv_kind=kv_kind, rope_theta=500000.0, eps=1e-5, seed=0x8B)
    if kv_kind == 2:
        cfg["hot_window"] = 32
    script = [("prompt", oracle.prompt_tokens(cfg["seed"], 1, 96, cfg["vocab"])), ("decode", 1)]
    ta, la, _ = gpu_script(ctx, cfg, script, True)
    tb, lb, _ = gpu_script(ctx, cfg, script, False)
    e = rel_err(la[0], lb[0])
    print(f"8B-shape kv_kind {kv_kind} logits rel_err={e:.2e}")
    if kv_kind == 2:
        want, margins = oracle_script(cfg, script)
        eo = rel_err(la[0], oracle_script.prompt_logits[0])
        print(f"8B-shape tiered batched logits against the oracle {eo:.2e}")
        assert eo < TQ_DECODE_TOL and e < 2 * TQ_DECODE_TOL
        if margins[0, 0] > TQ_DECODE_TIE:
            assert ta[0, 0] == want[0, 0]
        return
    assert e < LOGIT_TOL["turboquant" if kv_kind else "fp16"]
    part = np.sort(lb[0], axis=1)
    if part[0, -1] - part[0, -2] > 1e-3:
        assert ta[0, 0] == tb[0, 0]


def test_batched_prefill_turboquant_pages_match_oracle(ctx):
    """The TurboQuant pages the batched prefill writes against the oracle's
    after its token-by-token run of the same prompt: the K and V values
    reach the encoder through different (GEMM vs GEMV) summation orders, so
    a code at a quantization boundary may differ; at least 97% of the code
    bytes of every layer match, and the fp16 norms agree within 1e-3."""
    cfg = dict(TQ, seed=0x7A1)
    P = 57
    prompt = oracle.prompt_tokens(cfg["seed"], 1, P, cfg["vocab"])
    gm = nexus_amd.Model(ctx, **cfg)
    gm.prefill(prompt)
    om = oracle.Model(**cfg)
    for i in range(P):
        om.forward(np.ascontiguousarray(prompt[:, i], np.int32))
    for L in range(cfg["n_layers"]):
        same = total = 0
        for p in range(P):
            for kv in (0, 1):
                form, g = gm.kv_read(L, 0, p, kv)
                w = om.kv_read(L, 0, p, kv, 1)
                assert form == 1 and g.size == w.size == 58
                same += int(np.sum(g[:56] == w[:56]))
                total += 56
                gn, wn = g[56:58].view(np.float16)[0], w[56:58].view(np.float16)[0]
                assert abs(float(gn) - float(wn)) <= 1e-3 * abs(float(wn)), (L, p, kv)
        print(f"layer {L}: {same}/{total} code bytes equal")
        assert same >= 0.97 * total
    gm.close()
    om.close()


def test_batched_prefill_tiered_pages_match_oracle(ctx):
    """The tiered pages the batched prefill leaves (57 prompt tokens, a
    16-position window, prompts at 0 and then at 57 after three decode
    steps): the positions the decode steps would have compressed read back as
    TurboQuant (at least 97% of their code bytes equal to the oracle's after
    its token-by-token run, as in the TurboQuant test, norms within 1e-3),
    the window's positions as fp16 from the ring: each position's vector
    within 1e-2 of the oracle's, relative to its largest element (an RMSNorm
    input that rounds one fp16 step apart moves some elements by up to 5e-4
    on either prefill path; a stale or misplaced position differs by O(1))."""
    cfg = dict(TIERED, max_seq=256, seed=0x7A2)
    H = cfg["hot_window"]
    p1 = oracle.prompt_tokens(cfg["seed"], 1, 57, cfg["vocab"])
    p2 = oracle.prompt_tokens(cfg["seed"] + 1, 1, 30, cfg["vocab"])
    gm = nexus_amd.Model(ctx, **cfg)
    om = oracle.Model(**cfg)
    gm.prefill(p1)
    for i in range(p1.shape[1]):
        lg = om.forward(np.ascontiguousarray(p1[:, i], np.int32))
    # three decode steps fed the oracle's tokens on both sides, then a second
    # prompt starting inside a page
    fed = []
    for _ in range(3):
        t = lg.argmax(axis=1).astype(np.int32)
        fed.append(t)
        lg = om.forward(t)
    gm.decode_forced(np.stack(fed, 1))
    gm.prefill(p2)
    for i in range(p2.shape[1]):
        om.forward(np.ascontiguousarray(p2[:, i], np.int32))
    end = 57 + 3 + 30
    cold = 16 * ((end - H) // 16)  # TurboQuant below, the window's ring from here
    for L in range(cfg["n_layers"]):
        same = total = 0
        for p in range(end):
            for kv in (0, 1):
                form, g = gm.kv_read(L, 0, p, kv)
                if p < cold:
                    w = om.kv_read(L, 0, p, kv, 1)
                    assert form == 1 and g.size == w.size, (L, p, kv, form)
                    for h in range(cfg["n_kv_heads"]):
                        gh, wh = g[58 * h:58 * h + 58], w[58 * h:58 * h + 58]
                        same += int(np.sum(gh[:56] == wh[:56]))
                        total += 56
                        gn, wn = float(gh[56:58].view(np.float16)[0]), float(wh[56:58].view(np.float16)[0])
                        assert abs(gn - wn) <= 1e-3 * abs(wn), (L, p, kv, h)
                else:
                    w = om.kv_read(L, 0, p, kv, 0)
                    assert form == 0 and g.size == w.size, (L, p, kv, form)
                    gv, wv = g.view(np.float16).astype(np.float32), w.view(np.float16).astype(np.float32)
                    assert rel_err(gv, wv) < 1e-2, (L, p, kv)
        print(f"layer {L}: {same}/{total} TurboQuant code bytes equal")
        assert same >= 0.97 * total
    gm.close()
    om.close()


def test_batched_prefill_mixtral_layer_shape(ctx):
    """Two layers of the Mixtral shape (d 4096, 32/8 heads of 128, 8 experts
    of FFN 14336, top-2, vocab 32000), a 96-token prompt: the batched prefill
    (router GEMM, routing, per-expert GEMMs over the gathered token rows,
    combine) and the one-step prefill agree on the logits within 1e-3 and on
    the next token unless it is a tie."""
    cfg = dict(n_layers=2, d_model=4096, n_heads=32, n_kv_heads=8, head_dim=128, ffn=14336, vocab=32000,
               n_experts=8, top_k=2, max_seq=256, batch=1, kv_kind=0, rope_theta=1000000.0, eps=1e-5, seed=0x8E)
    script = [("prompt", oracle.prompt_tokens(cfg["seed"], 1, 96, cfg["vocab"])), ("decode", 1)]
    ta, la, _ = gpu_script(ctx, cfg, script, True)
    tb, lb, _ = gpu_script(ctx, cfg, script, False)
    e = rel_err(la[0], lb[0])
    print(f"Mixtral-shape logits rel_err={e:.2e}")
    assert e < 1e-3
    part = np.sort(lb[0], axis=1)
    if part[0, -1] - part[0, -2] > 1e-3:
        assert ta[0, 0] == tb[0, 0]


@pytest.mark.parametrize("M,N,K", [(100, 4096, 14336), (600, 28929, 1024)])
def test_gemm_without_memory_for_part_sums(poor, M, N, K):
    """A product whose K split finds no workspace, with and without an older,
    smaller one, is computed all the same: no error, one accumulation, the
    same sums up to their order (as in test_gemm_tile_shapes_and_k_parts).  A
    failed allocation is reported by its own call alone."""
    ctx = poor
    rng = np.random.default_rng(M)
    codes, scales = oracle.gen_quant_rows(0, N, K, 14, 0x77, 0.02)
    x = rng.standard_normal((M, K)).astype(np.float16)
    y0 = rng.standard_normal((M, N)).astype(np.float32)
    bx, bw, bs, by = ctx.upload(x.view(np.uint16)), ctx.upload(codes), ctx.upload(scales), ctx.upload(y0)
    rows = sorted({0, 31, 32, M // 2, M - 1})
    want = oracle.gemv(codes, scales, x[rows].astype(np.float32), N, K) + y0[rows]
    for first in (True, False):
        if not first:  # a workspace for a small product
            ctx.limit(0)
            ctx.gemm(bx, bw, bs, ctx.alloc(32 * 256 * 4), 32, 256, K, False)
        ctx.limit(4096)
        with pytest.raises(nexus_amd.NxError) as e:
            ctx.alloc(1 << 20)
        assert e.value.code == 3
        ctx.upload(y0, by)
        ctx.gemm(bx, bw, bs, by, M, N, K, True)
        got = ctx.download(by, (M, N), np.float32)
        assert rel_err(got[rows], want) < 2e-5 and np.isfinite(got).all()


@pytest.mark.parametrize("M,N,K,acc", [(100, 4096, 14336, False), (64, 512, 4096, True), (300, 28672, 512, False)])
def test_gemm_in_a_token_batch_is_the_eager_one(poor, M, N, K, acc):
    """A captured product takes the same tiles and K split as an eager one,
    so the same order of sums and the same bits, on every replay, with eager
    products of another size between them (which may replace the workspace),
    in a context that has none yet when the first is captured."""
    ctx = poor
    rng = np.random.default_rng(M + N)
    codes, scales = oracle.gen_quant_rows(0, N, K, 13, 0x77, 0.02)
    bw, bs = ctx.upload(codes), ctx.upload(scales)
    y0 = rng.standard_normal((M, N)).astype(np.float32)
    by, bt = ctx.upload(y0), ctx.alloc(16 * 256 * 4)
    for rep in range(3):
        bx = ctx.upload(rng.standard_normal((M, K)).astype(np.float16).view(np.uint16))
        res = []
        for captured in (True, False):
            ctx.upload(y0, by)
            if captured:
                ctx.check(ctx.L.nx_token_begin(ctx.h), "begin")
                ctx.gemm(bx, bw, bs, bt, 16, 256, K, False)  # (a smaller workspace first)
            ctx.gemm(bx, bw, bs, by, M, N, K, acc)
            if captured:
                ctx.check(ctx.L.nx_token_end(ctx.h), "end")
            res.append(ctx.download(by, (M, N), np.float32))
        ctx.free(bx)
        assert np.array_equal(res[0], res[1]), rep
        _gemm_case(ctx, 64, 1024, 4096 + 2048 * rep, seed=rep)
    for b in (bw, bs, by):
        ctx.free(b)


def test_small_gemm_is_not_split_where_one_launch_is_faster(ctx):
    """300 x 4096 x 1024 in one launch takes about 1.5 times as long as half
    the K (in two parts and their sums 2.0 times): part sums and their launch
    cost more there than blocks alone on their CUs."""
    us = []
    for K in (512, 1024):
        M, N, ms, best = 300, 4096, C.c_double(), []
        x, y = ctx.upload(np.zeros((M, K), np.uint16)), ctx.alloc(M * N * 4)
        w, s = ctx.upload(np.full((N, K // 2), 0x7A, np.uint8)), ctx.upload(np.full((N, K // 32), 0x2000, np.uint16))
        for _ in range(7):
            ctx.check(ctx.L.nx_time_gemm(ctx.h, x, w, s, y, M, N, K, 40, C.byref(ms)), "time")
            best.append(1e3 * ms.value)
        us.append(float(np.median(best)))
        for b in (x, y, w, s):
            ctx.free(b)
    print(f"300 x 4096: K 512 {us[0]:.1f} us, K 1024 {us[1]:.1f} us")
    assert us[1] < 1.75 * us[0]
