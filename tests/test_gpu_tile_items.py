"""The tile kernel's work items at the edges of their rules, against the oracle:
fp32 query chunks cut over the context, head dims widened to fp32 products,
values and lengths at the limits, plans over many sequences."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from batches import make_batch, oracle_attention  # noqa: E402
from test_gpu_kernels import check, dev, expected, ops, run_attention, to_np  # noqa: E402

pytestmark = pytest.mark.gpu

# chunks just above the splittable short queries, at and around a 64-row
# block, contexts around the smallest part (256 keys) and its multiples, a
# chunk that is its whole context (early row blocks see only the first
# parts), short queries and decodes between
CHUNKS = [[(17, 256), (17, 257), (64, 512)], [(65, 513), (1, 300), (63, 1100)],
          [(300, 300), (5, 700), (129, 900), (1, 64)], [(400, 1500)]]


@pytest.mark.parametrize("seqs", CHUNKS)
@pytest.mark.parametrize("H,Hkv,D", [(2, 1, 64), (2, 2, 48), (4, 2, 128)])
@pytest.mark.parametrize("small_ws", [False, True])
def test_fp32_chunks_split_over_the_context(seqs, H, Hkv, D, small_ws):
    """Few heads, so that the plan cuts every chunk into parts of about 256
    keys; with the smallest workspace the parts do not fit and the chunks stay
    whole. The tolerance is the fp32 one of every attention test."""
    b = make_batch(seqs, H, Hkv, D, 16, seed=D + len(seqs))
    ws = ops().lib().vl_paged_attention_min_workspace(len(seqs)) if small_ws else None
    check(run_attention(b, "f32", ws_bytes=ws), expected(b, "f32"), "f32")


def test_fp32_chunk_parts_leave_their_counters_clear():
    """One plan, several runs over fresh inputs: the parts' arrival counters are
    back at zero after each."""
    o = ops()
    b0 = make_batch([(200, 1200), (1, 500), (16, 900)], 4, 4, 64, 16, seed=5)
    ws = o.AttentionWorkspace().get(o.paged_attention_workspace_size(3, 217, 4, 64, 1200))
    bt, sl, qsl = dev(b0["block_tables"]), dev(b0["seq_lens"]), dev(b0["qsl"])
    for run in range(4):
        rng = np.random.default_rng(run)
        b = dict(b0, q=rng.standard_normal(b0["q"].shape).astype(np.float32))
        q, kc, vc = dev(b["q"]), dev(b["k_cache"]), dev(b["v_cache"])
        if run == 0:
            o.paged_attention_plan(q, kc, sl, qsl, 16, ws)
        out = torch.empty_like(q)
        o.paged_attention_run(out, q, kc, vc, bt, sl, qsl, b["scale"], 16, ws, max_query_len=200)
        check(to_np(out), oracle_attention(b), "f32")


# every head dim whose tiles came with no alignment rule: idle staging threads
# (80, 96, 112: units of 8 keys on 160 .. 224 threads), d tiles as quads +
# single, quads + pair, quads + pair + single; bf16 16 / 32 / 48 widened
@pytest.mark.parametrize("dtype,D", [("bf16", 16), ("bf16", 32), ("bf16", 48), ("bf16", 80),
                                     ("bf16", 96), ("bf16", 112), ("f32", 80), ("f32", 96),
                                     ("f32", 112)])
@pytest.mark.parametrize("bs", [4, 16, 32])
@pytest.mark.parametrize("layout", ["token", "head"])
def test_widened_head_dims(dtype, D, bs, layout):
    seqs = [(37, 37), (1, 2000), (70, 133), (1, 1), (5, 700), (0, 9), (17, 500)]
    b = make_batch(seqs, 6, 3, D, bs, seed=D + bs)
    check(run_attention(b, dtype, layout=layout), expected(b, dtype), dtype)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_widened_head_dim_takes_any_alignment(dtype):
    """Query rows, outputs and caches at odd element offsets and strides."""
    o = ops()
    tdt = torch.float32 if dtype == "f32" else torch.bfloat16
    b = make_batch([(40, 90), (1, 700), (3, 3)], 4, 2, 80, 16, seed=9)
    S, T = len(b["seq_lens"]), b["q"].shape[0]

    def odd(x):  # a contiguous copy one element into its storage
        t = dev(x, tdt)
        flat = torch.empty(t.numel() + 1, dtype=tdt, device="cuda")
        v = flat[1:].view(t.shape)
        v.copy_(t)
        return v

    wide = torch.zeros(T, 4 * 80 + 3, dtype=tdt, device="cuda")
    q = wide[:, 1:1 + 320].view(T, 4, 80) if T == 1 else wide[:, 1:321].unflatten(1, (4, 80))
    q.copy_(dev(b["q"], tdt))
    out = odd(np.zeros_like(b["q"]))
    ws = o.AttentionWorkspace().get(o.paged_attention_workspace_size(S, T, 4, 80, 700))
    o.paged_attention(out, q, odd(b["k_cache"]), odd(b["v_cache"]), dev(b["block_tables"]),
                      dev(b["seq_lens"]), dev(b["qsl"]), b["scale"], 16, ws, max_query_len=40)
    check(to_np(out), expected(b, dtype), dtype)


@pytest.mark.parametrize("D", [80, 112])
def test_widened_head_dims_over_an_fp8_cache(D):
    from oracle.attention import fp8_e4m3_decode, fp8_e4m3_encode
    o = ops()
    b = make_batch([(30, 300), (1, 900), (2, 2)], 4, 2, D, 16, seed=D)
    enc = {n: fp8_e4m3_encode(b[n]) for n in ("k_cache", "v_cache")}
    kc, vc = (dev(enc[n]).view(torch.float8_e4m3fn) for n in ("k_cache", "v_cache"))
    q = dev(b["q"])
    out = torch.empty_like(q)
    ws = o.AttentionWorkspace().get(o.paged_attention_workspace_size(3, 33, 4, D, 900))
    o.paged_attention(out, q, kc, vc, dev(b["block_tables"]), dev(b["seq_lens"]), dev(b["qsl"]),
                      b["scale"], 16, ws, max_query_len=30)
    want = oracle_attention(dict(b, k_cache=fp8_e4m3_decode(enc["k_cache"]),
                                 v_cache=fp8_e4m3_decode(enc["v_cache"])))
    check(to_np(out), want, "f32")


@pytest.mark.parametrize("seqs", [[(1, 1)], [(1, 127), (1, 128), (1, 129)], [(1, 8192)],
                                  [(1, 255 + 64 * i) for i in range(24)]])
@pytest.mark.parametrize("small_ws", [False, True])
def test_short_decode_batches_of_the_bandwidth_kernel(seqs, small_ws):
    """Few items, the shortest ranges; contexts around a range's end."""
    b = make_batch(seqs, 32, 8, 128, 16, seed=len(seqs))
    ws = ops().lib().vl_paged_attention_min_workspace(len(seqs)) if small_ws else None
    check(run_attention(b, "bf16", ws_bytes=ws), expected(b, "bf16"), "bf16")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("seqs", [[(17, 17), (400, 900)], [(16, 900), (17, 300)], [(5, 100)],
                                  [(2, 3000 + 100 * i) for i in range(12)]])
def test_bf16_tile_launches_by_query_bounds(D, seqs):
    """All sequences above 16 queries (the 32-row kernel alone), none, or both."""
    b = make_batch(seqs, 8, 4, D, 16, seed=D + len(seqs))
    check(run_attention(b, "bf16"), expected(b, "bf16"), "bf16")


@pytest.mark.parametrize("H,Hkv,D", [(2, 1, 64), (4, 2, 80)])
def test_split_chunk_with_rows_before_the_first_position(H, Hkv, D):
    """More queries than context: queries at negative positions see no key, and
    their rows are written as zeros also where the chunk's context is cut (the
    first row blocks then reach no part). The others match the oracle."""
    o = ops()
    q_len, ctx = 700, 300
    b = make_batch([(q_len, ctx)], H, Hkv, D, 16, seed=D)
    q = dev(b["q"])
    out = torch.full_like(q, float("nan"))
    ws = o.AttentionWorkspace().get(o.paged_attention_workspace_size(1, q_len, H, D, ctx))
    o.paged_attention(out, q, dev(b["k_cache"]), dev(b["v_cache"]), dev(b["block_tables"]),
                      dev(b["seq_lens"]), dev(b["qsl"]), b["scale"], 16, ws, max_query_len=q_len)
    got = to_np(out)
    assert np.array_equal(got[:q_len - ctx], np.zeros_like(got[:q_len - ctx]))
    seen = dict(b, q=b["q"][q_len - ctx:], qsl=np.array([0, ctx], np.int32))
    check(got[q_len - ctx:], oracle_attention(seen), "f32")


@pytest.mark.parametrize("dtype,D", [("f32", 80), ("bf16", 96), ("bf16", 32), ("f32", 48)])
@pytest.mark.parametrize("seqs", [[(2, 0), (40, 300), (1, 0), (5, 700), (40, 0), (1, 1)], [(3, 0)],
                                  [(30, 0), (1, 0)]])
def test_queries_without_context_are_written_as_zeros(dtype, D, seqs):
    """At the head dims whose items run fp32 products, as the generic kernel
    does at its own, beside other sequences and alone."""
    o = ops()
    tdt = torch.float32 if dtype == "f32" else torch.bfloat16
    b = make_batch(seqs, 4, 2, D, 16, seed=D)
    q = dev(b["q"], tdt)
    out = torch.full_like(q, float("nan"))
    S, T = len(seqs), q.shape[0]
    ws = o.AttentionWorkspace().get(o.paged_attention_workspace_size(S, T, 4, D, 700))
    o.paged_attention(out, q, dev(b["k_cache"], tdt), dev(b["v_cache"], tdt),
                      dev(b["block_tables"]), dev(b["seq_lens"]), dev(b["qsl"]), b["scale"], 16, ws)
    got = to_np(out)
    for i, (q_len, ctx) in enumerate(seqs):
        rows = slice(b["qsl"][i], b["qsl"][i + 1])
        if ctx == 0:
            assert np.array_equal(got[rows], np.zeros_like(got[rows]))
        else:
            one = dict(b, q=b["q"][rows], qsl=np.array([0, q_len], np.int32),
                       tables=b["tables"][i:i + 1], seq_lens=b["seq_lens"][i:i + 1])
            check(got[rows], expected(one, dtype), dtype)


@pytest.mark.parametrize("scale", [0.0, -0.11])
@pytest.mark.parametrize("dtype,D", [("f32", 80), ("f32", 48), ("bf16", 112), ("bf16", 32)])
def test_fp32_tiles_take_any_sign_of_scale(dtype, D, scale):
    """A scale of 0 (every visible key weighs the same) and a negative one: a
    masked score is -inf whatever the scale. Narrow items, several row blocks,
    a cut context."""
    seqs = [(37, 37), (70, 300), (1, 700), (3, 90), (17, 500)]
    b = dict(make_batch(seqs, 4, 2, D, 16, seed=D), scale=scale)
    check(run_attention(b, dtype), expected(b, dtype), dtype)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("dtype,D", [("f32", 80), ("f32", 96), ("f32", 112), ("bf16", 16),
                                     ("bf16", 48), ("bf16", 80)])
def test_a_value_row_that_is_not_finite_reaches_only_queries_that_see_it(dtype, D, value):
    """One element of a V row that later queries of the chunk see and earlier
    ones do not, at the head dims without an alignment rule: the earlier rows
    are what they are with the element finite, the others are not finite at
    that dim of that KV head, and every other element is unchanged. Chunks of
    several row blocks, of one, of at most 16 rows, a cut context; the element
    in a full tile, on the diagonal and in the last tile's last key."""
    H, Hkv, bs, d0, g0 = 4, 2, 16, D - 3, 1
    seqs = [(130, 130), (40, 321), (3, 90), (8, 64), (300, 1100)]
    at = [70, 300, 88, 63, 900]  # the key whose V element is not finite
    b = make_batch(seqs, H, Hkv, D, bs, seed=D)
    want = expected(b, dtype)
    v = b["v_cache"].copy()
    sees = np.zeros(want.shape[0], bool)
    for i, ((q_len, ctx), key) in enumerate(zip(seqs, at)):
        v[b["tables"][i][key // bs] * bs + key % bs, g0, d0] = value
        sees[b["qsl"][i]:b["qsl"][i + 1]] = ctx - q_len + np.arange(q_len) >= key
    assert sees.any() and not sees.all()
    got = run_attention(dict(b, v_cache=v), dtype)
    heads = slice(g0 * (H // Hkv), (g0 + 1) * (H // Hkv))
    assert not np.isfinite(got[sees, heads, d0]).any()
    got[sees, heads, d0] = want[sees, heads, d0]
    check(got, want, dtype)


def test_a_tight_workspace_cuts_chunks_into_fewer_parts():
    """Room for about half of the parts the plan aims for: the chunk is cut into
    longer ones (its sums run in another order than uncut), not left whole."""
    H, Hkv, D = 2, 1, 64
    b = make_batch([(64, 4096)], H, Hkv, D, 16, seed=7)
    fixed = ops().lib().vl_paged_attention_min_workspace(1)
    row = (D + 2) * 4 + 16  # a partial row: D floats, its max and sum, a range descriptor
    parts = 4096 // 256
    full, half, one = (run_attention(b, "f32", ws_bytes=fixed + n * (64 * H + 16) * row)
                       for n in (parts, parts // 2, 0))
    for got in (full, half, one):
        check(got, expected(b, "f32"), "f32")
    assert not np.array_equal(full, half) and not np.array_equal(half, one)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_more_sequences_than_the_plan_keeps_in_lds(dtype):
    """Over 2048 sequences the plan recomputes item counts instead of keeping
    them: decodes, short verifies and chunks in one longest-first list."""
    S = 2100
    seqs = [((1, 1 + i % 97) if i % 7 else (5, 5 + i % 140)) for i in range(S)]
    seqs[1000] = (40, 700)
    seqs[2099] = (20, 333)
    b = make_batch(seqs, 2, 1, 80, 16, seed=11)
    check(run_attention(b, dtype), expected(b, dtype), dtype)
