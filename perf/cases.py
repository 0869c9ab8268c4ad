"""The calls whose speed is measured, as a user's program makes them.

Four families, each through a public entry point:
  attn    one attention layer's paged_attention over a ragged batch: decodes,
          prefill chunks, or both in one call (plan and run)
  verify  speculative verification: the attention of a few query positions
          per sequence, then greedy_verify on the step's logits
  cache   a step's cache maintenance: copy-on-write block copies over all
          layers, then the K/V scatter of the step's tokens into one layer
  runner  one HipRunner.execute of a whole model step: logits on the host

A case holds plain values only. The lengths of its sequences follow from the
case (its "lens" seed), so that work() needs no inputs; tokens, weights, K/V,
queries and block tables come from the seed of prepare().
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-lite_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from vllmlite_amd import ops  # noqa: E402
from vllmlite_amd.config import CacheConfig, ModelConfig  # noqa: E402
from vllmlite_amd.hip_runner import HipRunner  # noqa: E402

# ------------------------------------------------------------------ cases --


def _attn(name, **kw):
    """Defaults: 32 query heads over 8 KV heads, head_dim 128, bf16, blocks of
    16, token-major cache, no decodes and no chunks."""
    case = dict(name=name, kind="attn", dtype="bf16", H=32, Hkv=8, D=128, bs=16, layout="token",
                lens=0, decodes=0, dec_lo=1, dec_hi=1, dec_mid=0, chunks=0, q_lo=1, q_hi=1,
                prior_hi=0, pool=0)
    case.update(kw)
    return case


def _runner(name, **kw):
    """Defaults: the 6-layer d_model 384 decoder of the end-to-end mix, fp32."""
    case = dict(name=name, kind="runner", layers=6, d_model=384, H=8, Hkv=4, d_ff=1024, vocab=261,
                max_len=512, lens=0, decodes=0, dec_lo=1, dec_hi=1, drafts=0, chunks=0, q_lo=1,
                q_hi=1, prior_hi=0)
    case.update(kw)
    return case


def listed():
    return [
        # a lightly loaded server's decode: a few short sequences, where the
        # plan, the launches and the host's call count
        _attn("decode_4", decodes=4, dec_lo=100, dec_hi=900, lens=1),
        # the headline decode batch: 256 sequences, contexts around 1024
        # (64..8192), blocks scattered over a 2^17-block pool
        _attn("decode_256", decodes=256, dec_lo=64, dec_hi=8192, dec_mid=1024, pool=1 << 17,
              lens=2),
        # chunked prefill beside running decodes in one call, a full token
        # budget: 16 chunks of 512 tokens and 200 decodes
        _attn("mixed_8392", decodes=200, dec_lo=128, dec_hi=4096, chunks=16, q_lo=512, q_hi=512,
              prior_hi=2048, pool=1 << 17, lens=3),
        # prefill only, ragged: chunks of odd lengths, some without a prefix
        _attn("prefill_ragged", chunks=12, q_lo=17, q_hi=700, prior_hi=3000, lens=4),
        # head_dim 64 with 8 query heads per KV head, head-major blocks, long
        # and short contexts beside each other
        _attn("decode_d64", H=32, Hkv=4, D=64, layout="head", decodes=160, dec_lo=64, dec_hi=8192,
              dec_mid=1024, lens=5),
        # a head_dim that is no power of two: a chunk or two beside decodes
        _attn("mixed_d80", H=16, Hkv=8, D=80, decodes=24, dec_lo=30, dec_hi=2000, chunks=2, q_lo=50,
              q_hi=200, prior_hi=500, lens=6),
        # fp32, the default model shape (8 heads of 64, no grouping): one
        # scheduler step of the default 2048-token budget
        _attn("mixed_fp32", dtype="f32", H=8, Hkv=8, D=64, decodes=24, dec_lo=20, dec_hi=2000,
              chunks=5, q_lo=300, q_hi=500, prior_hi=1200, lens=7),
        # speculative verification: 64 sequences of 4 drafts + 1, contexts
        # 1024..32768, vocabulary of 32000
        dict(name="verify_64x5", kind="verify", H=32, Hkv=8, D=128, bs=16, lens=8, seqs=64,
             drafts=4, ctx_lo=1024, ctx_hi=32768, vocab=32000, pool=1 << 17),
        # copy-on-write copies of 48 shared tail blocks, then a full token
        # budget's K/V scatter
        dict(name="cache_update", kind="cache", dtype="bf16", Hkv=8, D=128, bs=16, layers=2,
             layout="token", pairs=48, tokens=8392, spare=1.25),
        # one decode step of the end-to-end mix's decoder, 16 sequences
        _runner("step_decode_16", decodes=16, dec_lo=18, dec_hi=440, lens=9),
        # the default ModelConfig and scheduler limits: a decode step of 32
        # sequences
        _runner("step_default_decode_32", d_model=512, Hkv=8, d_ff=2048, max_len=2048, decodes=32,
                dec_lo=20, dec_hi=1200, lens=10),
        # the same model's largest step: prefill chunks beside decodes, close
        # to the 2048-token budget
        _runner("step_default_prefill", d_model=512, Hkv=8, d_ff=2048, max_len=2048, decodes=9,
                dec_lo=20, dec_hi=900, chunks=5, q_lo=380, q_hi=420, prior_hi=300, lens=11),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: sizes spread over their logarithm."""
    lens = rng.randrange(1 << 20)
    pick = rng.random()
    if pick < 0.55:
        D = rng.choice([128, 128, 128, 64, 64, 80, 96, 48, 32])
        rep = rng.choice([1, 2, 4, 4, 8])
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32", "f32_bf16kv", "f32_fp8kv"])
        Hkv = rng.choice([1, 2, 4, 8, 8])
        # head dims without matrix tiles and 32-bit inputs: smaller batches, as
        # such models are
        big = dtype == "bf16" and D in (64, 128)
        if not big:
            rep, Hkv = min(rep, 4), min(Hkv, 4)
        c = _attn("", dtype=dtype, H=rep * Hkv, Hkv=Hkv, D=D, bs=rng.choice([16, 16, 16, 32]),
                  layout=rng.choice(["token", "token", "head"]), lens=lens)
        del c["name"]
        mode = rng.choice(["decode", "prefill", "mixed"])
        if mode != "prefill":
            c["decodes"] = _log_int(rng, 1, 200 if big else 32)
            c["dec_lo"] = _log_int(rng, 1, 300)
            c["dec_hi"] = c["dec_lo"] + _log_int(rng, 10, 4000 if big else 1900)
            if rng.random() < 0.5:
                c["dec_mid"] = _log_int(rng, c["dec_lo"], c["dec_hi"])
        if mode != "decode":
            c["chunks"] = _log_int(rng, 1, 12 if big else 3)
            c["q_lo"] = _log_int(rng, 2, 300 if big else 100)
            c["q_hi"] = c["q_lo"] + _log_int(rng, 1, 400 if big else 100)
            c["prior_hi"] = rng.choice([0, _log_int(rng, 16, 2500 if big else 500)])
        return c
    if pick < 0.65:
        lo = _log_int(rng, 16, 2000)
        return dict(kind="verify", H=32, Hkv=8, D=128, bs=16, lens=lens,
                    seqs=_log_int(rng, 1, 48), drafts=rng.randint(1, 7), ctx_lo=lo,
                    ctx_hi=lo + _log_int(rng, 10, 16000), vocab=rng.choice([261, 5003, 32000]),
                    pool=0)
    if pick < 0.75:
        return dict(kind="cache", dtype=rng.choice(["bf16", "f32", "fp8"]),
                    Hkv=rng.choice([1, 4, 8]), D=rng.choice([48, 64, 80, 128]),
                    bs=16, layers=rng.randint(1, 3), layout=rng.choice(["token", "head"]),
                    pairs=_log_int(rng, 1, 64), tokens=_log_int(rng, 1, 8000), spare=1.5)
    hd, H = rng.choice([(48, 8), (64, 8), (32, 8), (64, 4)])
    c = _runner("", layers=rng.randint(2, 6), d_model=hd * H, H=H, Hkv=rng.choice([H // 2, H]),
                d_ff=16 * _log_int(rng, 16, 128), max_len=rng.choice([512, 1024, 2048]), lens=lens)
    del c["name"]
    if rng.random() < 0.6:
        c["decodes"], c["dec_lo"] = _log_int(rng, 1, 32), _log_int(rng, 2, 100)
        c["dec_hi"] = c["dec_lo"] + _log_int(rng, 10, c["max_len"] - 120)
        c["drafts"] = rng.choice([0, 0, 0, 3])
    else:
        c["decodes"], c["dec_lo"], c["dec_hi"] = _log_int(rng, 1, 12), 10, 300
        c["chunks"], c["q_lo"] = _log_int(rng, 1, 4), _log_int(rng, 2, 300)
        c["q_hi"] = c["q_lo"] + _log_int(rng, 1, 100)
        c["prior_hi"] = rng.choice([0, 100])
    return c


# ---------------------------------------------------------------- lengths --


def _seqs(case):
    """(query tokens, context after the step) per sequence, decodes first."""
    r = np.random.default_rng(case["lens"])
    if case["kind"] == "verify":
        q = case["drafts"] + 1
        return [(q, max(q, int(c))) for c in r.integers(case["ctx_lo"], case["ctx_hi"] + 1,
                                                        size=case["seqs"])]
    out = []
    lo, hi = case["dec_lo"], case["dec_hi"]
    q = 1 + case.get("drafts", 0)
    for _ in range(case["decodes"]):
        if case.get("dec_mid"):  # lognormal around dec_mid, else uniform
            c = int(np.clip(r.lognormal(math.log(case["dec_mid"]), 0.6), lo, hi))
        else:
            c = int(r.integers(lo, hi + 1))
        out.append((q, max(q, c)))
    for _ in range(case["chunks"]):
        n = int(r.integers(case["q_lo"], case["q_hi"] + 1))
        out.append((n, n + int(r.integers(0, case["prior_hi"] + 1))))
    return out


def _pairs(seqs):
    """Unmasked (query, key) pairs."""
    return sum(q * (c - q) + q * (q + 1) // 2 for q, c in seqs)


_KV = {"bf16": torch.bfloat16, "f32": torch.float32, "f32_bf16kv": torch.bfloat16,
       "f32_fp8kv": torch.float8_e4m3fn, "fp8": torch.float8_e4m3fn}


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + 17)
    return g


def _randn(shape, g, dtype):
    """N(0, 1) values of dtype on the GPU (narrow types rounded from fp32)."""
    if dtype == torch.float8_e4m3fn:
        return torch.randn(shape, generator=g, device="cuda").to(dtype)
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


# -------------------------------------------------------- attention layers --


def _attn_state(case, seed, seqs, dtype, layout, pool):
    H, Hkv, D, bs = case["H"], case["Hkv"], case["D"], case["bs"]
    g = _gen(seed)
    nblk = [-(-c // bs) for _, c in seqs]
    pool = max(pool, sum(nblk) + 8)
    perm = np.random.default_rng(seed + 1).permutation(pool)
    W = max(nblk)
    tables = np.zeros((len(seqs), W), np.int32)
    off = 0
    for i, n in enumerate(nblk):
        tables[i, :n] = perm[off:off + n]
        off += n
    shape = (pool, Hkv, bs, D) if layout == "head" else (pool * bs, Hkv, D)
    kv = _KV[dtype]
    T = sum(q for q, _ in seqs)
    qsl = np.zeros(len(seqs) + 1, np.int32)
    qsl[1:] = np.cumsum([q for q, _ in seqs])
    query = _randn((T, H, D), g, torch.bfloat16 if dtype == "bf16" else torch.float32)
    s = dict(kc=_randn(shape, g, kv), vc=_randn(shape, g, kv), q=query,
             out=torch.empty_like(query), bt=torch.from_numpy(tables).cuda(),
             lens=torch.tensor([c for _, c in seqs], dtype=torch.int32, device="cuda"),
             qsl=torch.from_numpy(qsl).cuda(), bs=bs, scale=1.0 / math.sqrt(D),
             max_q=max(q for q, _ in seqs), min_q=min(q for q, _ in seqs),
             max_ctx=max(c for _, c in seqs), tables=tables, qsl_np=qsl, seqs=seqs)
    s["ws"] = ops.AttentionWorkspace().get(
        ops.paged_attention_workspace_size(len(seqs), T, H, D, s["max_ctx"]))
    return s


def _attn_call(s):
    ops.paged_attention(s["out"], s["q"], s["kc"], s["vc"], s["bt"], s["lens"], s["qsl"],
                        s["scale"], s["bs"], s["ws"], max_query_len=s["max_q"],
                        min_query_len=s["min_q"], max_context_len=s["max_ctx"])
    return s["out"]


def _attn_exact(case, s, layout):
    """softmax(scale q k^T) v per sequence in 64 bits, causal within the
    sequence's last q positions."""
    H, Hkv, D, bs = case["H"], case["Hkv"], case["D"], case["bs"]
    rep = H // Hkv
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    for i, (ql, c) in enumerate(s["seqs"]):
        nb = -(-c // bs)
        blocks = torch.from_numpy(s["tables"][i, :nb].astype(np.int64)).cuda()

        def rows(cache):  # [Hkv, c, D] in 64 bits
            if layout == "head":
                x = cache[blocks].to(torch.float64).permute(1, 0, 2, 3).reshape(Hkv, nb * bs, D)
            else:
                x = cache.view(-1, bs, Hkv, D)[blocks].to(torch.float64)
                x = x.permute(2, 0, 1, 3).reshape(Hkv, nb * bs, D)
            return x[:, :c].contiguous()

        k, v = rows(s["kc"]), rows(s["vc"])
        t0 = int(s["qsl_np"][i])
        q = s["q"][t0:t0 + ql].to(torch.float64).view(ql, Hkv, rep, D)
        q = q.permute(1, 0, 2, 3).reshape(Hkv, ql * rep, D).contiguous()
        sc = torch.matmul(q, k.transpose(1, 2).contiguous()) * s["scale"]
        if ql > 1:
            pos = (c - ql + torch.arange(ql, device="cuda")).repeat_interleave(rep)
            sc.masked_fill_(torch.arange(c, device="cuda")[None, None, :] > pos[None, :, None],
                            float("-inf"))
        o = torch.matmul(torch.softmax(sc, dim=-1), v)
        out[t0:t0 + ql] = o.view(Hkv, ql, rep, D).permute(1, 0, 2, 3).reshape(ql, H, D)
    return out


# ---------------------------------------------------------------- verify ---


def _verify_state(case, seed):
    s = _attn_state(case, seed, _seqs(case), "bf16", "token", case["pool"])
    g = _gen(seed + 7)
    S, K, V = case["seqs"], case["drafts"], case["vocab"]
    rows = S * (K + 1)
    s["logits"] = torch.randn((rows, V), generator=g, device="cuda")
    picks = s["logits"].view(S, K + 1, V)[:, :K].argmax(-1).to(torch.int32)
    # n-gram drafts: right about two times in three
    other = torch.randint(0, V, (S, K), generator=g, device="cuda", dtype=torch.int32)
    good = torch.rand((S, K), generator=g, device="cuda") < 0.67
    s["drafts"] = torch.where(good, picks, other).contiguous()
    s["row_start"] = torch.arange(0, rows, K + 1, dtype=torch.int32, device="cuda")
    s["num_drafts"] = torch.full((S,), K, dtype=torch.int32, device="cuda")
    s["tokens"] = torch.zeros((S, K + 1), dtype=torch.int32, device="cuda")
    s["accepted"] = torch.zeros(S, dtype=torch.int32, device="cuda")
    return s


def _verify_exact(case, s):
    S, K, V = case["seqs"], case["drafts"], case["vocab"]
    picks = s["logits"].view(S, K + 1, V).argmax(-1).to(torch.int32)
    ok = (picks[:, :K] == s["drafts"]).to(torch.int32)
    acc = ok.cumprod(1).sum(1).to(torch.int32)
    # the accepted drafts and the model's own next token; the rest unused (-1)
    keep = torch.arange(K + 1, device="cuda")[None, :] <= acc[:, None]
    tokens = torch.where(keep, picks, torch.full_like(picks, -1))
    return [_attn_exact(case, s, "token"), tokens, acc]


# ----------------------------------------------------------------- cache ---


def _cache_state(case, seed):
    Hkv, D, bs, L = case["Hkv"], case["D"], case["bs"], case["layers"]
    g = _gen(seed)
    r = np.random.default_rng(seed + 3)
    dt = _KV[case["dtype"]]
    nblk = int(case["spare"] * -(-case["tokens"] // bs)) + 2 * case["pairs"] + 8
    shape = (L, nblk, Hkv, bs, D) if case["layout"] == "head" else (L, nblk * bs, Hkv, D)
    perm = r.permutation(nblk)
    pairs = perm[:2 * case["pairs"]].reshape(-1, 2).astype(np.int32)
    free = perm[2 * case["pairs"]:]
    slots = (free[:, None] * bs + np.arange(bs)[None, :]).reshape(-1)[:case["tokens"]]
    T = case["tokens"]
    return dict(kc=_randn(shape, g, dt), vc=_randn(shape, g, dt), k=_randn((T, Hkv, D), g, dt),
                v=_randn((T, Hkv, D), g, dt), bs=bs,
                pairs=torch.from_numpy(pairs).cuda(),
                slots=torch.from_numpy(slots.astype(np.int32)).cuda())


def _cache_run(s):
    ops.copy_blocks(s["kc"], s["vc"], s["pairs"], s["bs"])
    ops.reshape_and_cache(s["k"], s["v"], s["kc"][0], s["vc"][0], s["slots"])
    bits = {1: torch.uint8, 2: torch.int16, 4: torch.int32}[s["kc"].element_size()]
    return [s["kc"].view(bits), s["vc"].view(bits)]  # bytes move: nothing is rounded


# ---------------------------------------------------------------- runner ---


class _Table:
    def __init__(self, ids):
        self.block_ids = ids


class _Seq:
    """The fields a runner reads of a scheduled sequence."""

    def __init__(self, rid, tokens, blocks, drafts):
        self.request_id, self.token_ids = rid, tokens
        self.table, self.draft_token_ids = _Table(blocks), drafts


class _Item:
    def __init__(self, seq, start, n):
        self.seq, self.start_pos, self.num_tokens = seq, start, n


class _Step:
    def __init__(self, items):
        self.scheduled, self.cow = items, []


def _weights(case, seed):
    """A trained model's stand-in: N(0, 1 / fan-in) projections, norm weights
    around one, the head tied to the embedding."""
    r = np.random.default_rng(seed + 5)
    d, f, V = case["d_model"], case["d_ff"], case["vocab"]
    hd = d // case["H"]

    def mat(k, n):
        return r.standard_normal((k, n), dtype=np.float32) * np.float32(1.0 / math.sqrt(k))

    def norm():
        return (1.0 + 0.1 * r.standard_normal(d)).astype(np.float32)

    w = {"tok_emb": r.standard_normal((V, d), dtype=np.float32) * np.float32(1 / math.sqrt(d))}
    for i in range(case["layers"]):
        p = f"layers.{i}."
        w[p + "attn_norm"], w[p + "ffn_norm"] = norm(), norm()
        w[p + "wq"], w[p + "wo"] = mat(d, d), mat(d, d)
        w[p + "wk"], w[p + "wv"] = mat(d, case["Hkv"] * hd), mat(d, case["Hkv"] * hd)
        w[p + "w_gate"], w[p + "w_up"], w[p + "w_down"] = mat(d, f), mat(d, f), mat(f, d)
    w["final_norm"] = norm()
    w["lm_head"] = np.ascontiguousarray(w["tok_emb"].T)
    return w


def _runner_seqs(case):
    return [(min(q, case["max_len"]), min(c, case["max_len"])) for q, c in _seqs(case)]


def _runner_state(case, seed):
    bs = 16
    seqs = _runner_seqs(case)
    r = np.random.default_rng(seed + 9)
    nblk = [-(-c // bs) for _, c in seqs]
    pool = sum(nblk) + 8
    mc = ModelConfig(n_layers=case["layers"], n_heads=case["H"], n_kv_heads=case["Hkv"],
                     d_model=case["d_model"], d_ff=case["d_ff"], vocab_size=case["vocab"],
                     max_seq_len=case["max_len"])
    runner = HipRunner(mc, CacheConfig(block_size=bs, num_blocks=pool),
                       weights=_weights(case, seed))
    perm = [int(b) for b in r.permutation(pool)]
    items, prior, off = [], [], 0
    for i, (q, c) in enumerate(seqs):
        toks = [int(t) for t in r.integers(0, case["vocab"], size=c)]
        drafts = toks[c - q + 1:] if case["drafts"] and i < case["decodes"] else []
        seq = _Seq(f"r{i}", toks, perm[off:off + nblk[i]], drafts)
        off += nblk[i]
        items.append(_Item(seq, c - q, q))
        if c > q:
            prior.append(_Item(seq, 0, c - q))
    # the cached context, as earlier prefill steps left it
    step, n = [], 0
    for it in prior:
        while it.num_tokens > 0:
            take = min(it.num_tokens, 1024 - n)
            step.append(_Item(it.seq, it.start_pos, take))
            it.start_pos, it.num_tokens, n = it.start_pos + take, it.num_tokens - take, n + take
            if n == 1024:
                runner.execute(_Step(step))
                step, n = [], 0
    if step:
        runner.execute(_Step(step))
    out = _Step(items)
    runner.execute(out)  # a serving process has met the step's shape before
    return dict(runner=runner, step=out, seqs=seqs)


def _runner_exact(case, s, seed):
    """The decoder over every sequence's tokens in 64 bits: RMSNorm, rotary
    position embedding by interleaved pairs (the model's table is fp32),
    causal grouped attention, SwiGLU, tied head. Returns the logits and the
    K and V caches (zero where no sequence owns the slot)."""
    w = {k: torch.from_numpy(v).cuda().double() for k, v in _weights(case, seed).items()}
    d, H, Hkv = case["d_model"], case["H"], case["Hkv"]
    hd, rep = d // H, H // Hkv
    inv = 1.0 / (10000.0 ** (np.arange(0, hd, 2, dtype=np.float32) / hd))
    ang = np.arange(case["max_len"], dtype=np.float32)[:, None] * inv[None, :].astype(np.float32)
    cos = torch.from_numpy(np.cos(ang).astype(np.float32)).cuda().double()
    sin = torch.from_numpy(np.sin(ang).astype(np.float32)).cuda().double()

    def norm(x, g):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * g

    def rope(x):  # [c, heads, hd]
        co, si = cos[:x.shape[0], None, :], sin[:x.shape[0], None, :]
        e, o = x[..., 0::2], x[..., 1::2]
        return torch.stack([e * co - o * si, e * si + o * co], -1).reshape(x.shape)

    cache = [torch.zeros(s["runner"].cache_k.shape, dtype=torch.float64, device="cuda")
             for _ in range(2)]
    rows = []
    for it in s["step"].scheduled:
        c = it.start_pos + it.num_tokens
        x = w["tok_emb"][torch.tensor(it.seq.token_ids[:c], device="cuda")]
        mask = torch.ones((c, c), dtype=torch.bool, device="cuda").triu(1)
        blocks = torch.tensor(it.seq.table.block_ids, device="cuda")
        slots = (blocks[:, None] * 16 + torch.arange(16, device="cuda")).reshape(-1)[:c]
        for i in range(case["layers"]):
            p = f"layers.{i}."
            h = norm(x, w[p + "attn_norm"])
            q = rope((h @ w[p + "wq"]).view(c, H, hd)).transpose(0, 1)
            k = rope((h @ w[p + "wk"]).view(c, Hkv, hd)).transpose(0, 1)
            v = (h @ w[p + "wv"]).view(c, Hkv, hd).transpose(0, 1)
            cache[0][i, slots], cache[1][i, slots] = k.transpose(0, 1), v.transpose(0, 1)
            k, v = k.repeat_interleave(rep, 0), v.repeat_interleave(rep, 0)
            sc = torch.matmul(q.contiguous(), k.transpose(1, 2).contiguous()) / math.sqrt(hd)
            o = torch.matmul(torch.softmax(sc.masked_fill(mask, float("-inf")), -1), v.contiguous())
            x = x + o.transpose(0, 1).reshape(c, d) @ w[p + "wo"]
            h = norm(x, w[p + "ffn_norm"])
            gate = h @ w[p + "w_gate"]
            x = x + (gate * torch.sigmoid(gate) * (h @ w[p + "w_up"])) @ w[p + "w_down"]
        n = min(1 + len(it.seq.draft_token_ids), it.num_tokens)
        rows.append(norm(x[c - n:], w["final_norm"]) @ w["lm_head"])
    return [torch.cat(rows).cpu().numpy()] + cache


# -------------------------------------------------------------- interface --


def prepare(case, seed):
    kind = case["kind"]
    if kind == "attn":
        s = _attn_state(case, seed, _seqs(case), case["dtype"], case["layout"], case["pool"])
    elif kind == "verify":
        s = _verify_state(case, seed)
    elif kind == "cache":
        s = _cache_state(case, seed)
    else:
        s = _runner_state(case, seed)
    s["kind"] = kind
    return s


def run(state):
    kind = state["kind"]
    if kind == "attn":
        return _attn_call(state)
    if kind == "verify":
        _attn_call(state)
        ops.greedy_verify(state["logits"], state["row_start"], state["num_drafts"],
                          state["drafts"], state["tokens"], state["accepted"])
        return [state["out"], state["tokens"], state["accepted"]]
    if kind == "cache":
        return _cache_run(state)
    runner = state["runner"]
    return [runner.execute(state["step"])[0], runner.cache_k, runner.cache_v]


def work(case):
    kind = case["kind"]
    if kind == "cache":
        es = {"bf16": 2, "f32": 4, "fp8": 1}[case["dtype"]]
        row = case["Hkv"] * case["D"] * es
        copies = 2 * 2 * case["pairs"] * case["layers"] * case["bs"] * row
        return {"bytes": copies + 8 * case["pairs"] + case["tokens"] * (4 * row + 4), "flops": 0}
    if kind in ("attn", "verify"):
        seqs = _seqs(case)
        dtype = case.get("dtype", "bf16")
        qe, ke = 2 if dtype == "bf16" else 4, _KV[dtype].itemsize
        T = sum(q for q, _ in seqs)
        b = sum(c for _, c in seqs) * 2 * case["Hkv"] * case["D"] * ke
        b += 2 * T * case["H"] * case["D"] * qe
        b += sum(4 * -(-c // case["bs"]) + 8 for _, c in seqs)
        if kind == "verify":
            b += T * case["vocab"] * 4 + T * 8
        return {"bytes": b, "flops": 4 * case["D"] * case["H"] * _pairs(seqs)}
    seqs = _runner_seqs(case)
    d, f, V, L = case["d_model"], case["d_ff"], case["vocab"], case["layers"]
    kvd = case["Hkv"] * (d // case["H"])
    T = sum(q for q, _ in seqs)
    R = sum(min(q, 1 + case["drafts"]) if i < case["decodes"] else 1
            for i, (q, _) in enumerate(seqs))
    per = d * (d + 2 * kvd) + d * d + 3 * d * f
    kv = sum(c for _, c in seqs) * 2 * kvd * 4
    return {"bytes": L * (per * 4 + kv) + V * d * 4 + R * V * 4 + T * d * 4,
            "flops": L * (2 * T * per + 4 * d * _pairs(seqs)) + 2 * R * V * d}


def tolerance(case):
    kind = case["kind"]
    if kind == "cache":
        return "exact"
    if kind == "runner":
        # fp32 sums in another order, carried through the layers
        return {"rel": 1e-5}
    if kind == "verify":
        return {"rel": 1e-2, "differ": 0.0}
    # bf16: the output's and the weights' rounding; fp32: sums in another order
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 4e-6}


def exact(case, seed):
    kind = case["kind"]
    if kind == "cache":
        return None  # bytes, compared as they are
    if kind == "runner":
        s = _runner_state(case, seed)
        return _runner_exact(case, s, seed)
    s = prepare(case, seed)
    if kind == "verify":
        return _verify_exact(case, s)
    return _attn_exact(case, s, case["layout"])
