"""The tile kernel's work items at the edges of their rules, against the
oracle: fp32 query chunks cut over the context."""

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
