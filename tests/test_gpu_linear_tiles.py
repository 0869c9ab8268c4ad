"""The projections of many rows (linear_tile_kernel, chosen by how its 32-row
workgroups fill the compute units) and the deep down projection, against
float64 NumPy, and a model that needs both against the oracle runner."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import small_cfg  # noqa: E402
from test_gpu_linear import _close, _ops, _rms, _silu  # noqa: E402
from test_gpu_runner import PROMPTS, _logit_trace  # noqa: E402

pytestmark = pytest.mark.gpu


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _rows_per_workgroup(rows, n, k, mode="store", norm=False):
    """What the dispatch takes for this many rows and columns (linear.hip:
    takes_tiles, launch_tiles): 64- or 32-row workgroups of
    linear_tile_kernel, or 0 (linear_rows_kernel)."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    ntile, row_tiles = -(-n // 16), -(-rows // 16)
    cb = -(-ntile // 4)
    grid, swiglu = cb * -(-rows // 32), mode == "swiglu"
    rounds = -(-grid // cus)
    nsub = 1
    while nsub < 4 and ntile * -(-row_tiles // (2 * nsub)) >= 2 * cus:
        nsub *= 2
    groups = -(-row_tiles // nsub)
    wgs = ntile * groups
    whole = -(-wgs // cus) - 1
    load = whole * nsub + (row_tiles - (groups - 1) * nsub if wgs - whole * cus <= ntile else nsub)
    if grid < cus:
        return 0
    if swiglu and 320 < k <= 384:
        tiles = rounds > 3 or (rounds > 1 and load > 7 * rounds)
    else:
        close = 256 < k <= 512 if swiglu else not norm and k <= 1024
        tiles = rounds != 2 or not close or load >= 12
    return 0 if not tiles else 64 if cb * -(-rows // 64) >= 2 * cus else 32


@pytest.mark.parametrize("rows,k,n,mode,wg_rows",
                         [(512, 384, 1024, "swiglu", 0), (800, 384, 1024, "swiglu", 0),
                          (896, 384, 1024, "swiglu", 32), (1280, 336, 1024, "swiglu", 0),
                          (512, 320, 1024, "swiglu", 32), (544, 320, 1024, "swiglu", 0),
                          (544, 256, 1024, "swiglu", 32), (576, 512, 1024, "swiglu", 32),
                          (288, 512, 2048, "swiglu", 0), (289, 512, 2048, "swiglu", 0),
                          (305, 512, 2048, "swiglu", 32), (1000, 512, 512, "store", 32),
                          (1056, 512, 512, "store", 0), (1056, 512, 512, "norm", 32),
                          (768, 384, 768, "store", 32), (1376, 384, 384, "accumulate", 0),
                          (1376, 1024, 384, "accumulate", 0),
                          (1400, 1024, 384, "accumulate", 32), (1400, 384, 768, "accumulate", 32)])
def test_which_kernel_many_rows_take(rows, k, n, mode, wg_rows):
    """The sizes on both sides of the rule's lines. Row-major weights always run
    linear_rows_kernel, so a tiled weight that gives its bits ran it too."""
    norm, mode = mode == "norm", "store" if mode == "norm" else mode
    assert _rows_per_workgroup(rows, n, k, mode, norm) == wg_rows
    o = _ops()
    rng = np.random.default_rng(rows + k)
    halves = 2 if mode == "swiglu" else 1
    x, w = _dev(rng.standard_normal((rows, k)).astype(np.float32)), _dev(
        (0.05 * rng.standard_normal((k, halves * n))).astype(np.float32))
    g = torch.ones(k, device="cuda") if norm else None
    kind = {"store": o.LINEAR_STORE, "accumulate": o.LINEAR_ACCUMULATE,
            "swiglu": o.LINEAR_SWIGLU}[mode]
    tiled, plain = (torch.zeros(rows, n, device="cuda") for _ in range(2))
    o.linear_rows(tiled, x, o.tile16(w, halves), g, mode=kind)
    o.linear_rows(plain, x, w, g, mode=kind)
    assert torch.equal(tiled, plain) == (wg_rows == 0)
    _close(tiled.cpu().numpy(), plain.cpu().numpy())


# 32- and 64-row workgroups, a last row block and a last column block that are
# not full, K below a chunk of 64, a multiple of it and not
@pytest.mark.parametrize("rows,k,n,mode,wg_rows",
                         [(1400, 1024, 384, "accumulate", 32), (1000, 496, 1100, "store", 32),
                          (1030, 384, 1152, "store", 32), (700, 64, 1030, "swiglu", 32),
                          (260, 512, 2048, "swiglu", 0), (2050, 16, 520, "store", 32),
                          (1024, 512, 2048, "swiglu", 64), (1000, 400, 2041, "swiglu", 64),
                          (2050, 16, 1030, "store", 64), (2050, 336, 1100, "store", 64),
                          (4111, 1024, 512, "accumulate", 64)])
@pytest.mark.parametrize("norm", [False, True])
def test_many_rows_over_tiled_weights(rows, k, n, mode, wg_rows, norm):
    assert _rows_per_workgroup(rows, n, k, mode, norm) == wg_rows
    o = _ops()
    rng = np.random.default_rng(rows + k + norm)
    halves = 2 if mode == "swiglu" else 1
    x = rng.standard_normal((rows, k)).astype(np.float32)
    w = (0.05 * rng.standard_normal((k, halves * n))).astype(np.float32)
    g = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    res = rng.standard_normal((rows, n)).astype(np.float32)
    y = (_rms(x.astype(np.float64), g.astype(np.float64)) if norm else x.astype(np.float64)) @ w
    want = {"store": y[:, :n], "accumulate": res + y[:, :n],
            "swiglu": _silu(y[:, :n]) * y[:, n:] if halves == 2 else None}[mode]
    out = _dev(res)
    o.linear_rows(out, _dev(x), o.tile16(_dev(w), halves), _dev(g) if norm else None,
                  mode={"store": o.LINEAR_STORE, "accumulate": o.LINEAR_ACCUMULATE,
                        "swiglu": o.LINEAR_SWIGLU}[mode])
    torch.cuda.synchronize()
    _close(out.cpu().numpy(), want)


@pytest.mark.parametrize("rows", [1, 16, 33, 1100, 4111])
@pytest.mark.parametrize("k,n", [(16, 512), (1040, 40), (2048, 512)])
def test_deep_projection(rows, k, n):
    assert _rows_per_workgroup(rows, n, k) == (0 if rows < 1100 or n < 512 else
                                               32 if rows == 1100 else 64)
    o = _ops()
    rng = np.random.default_rng(rows + k)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    w = (0.02 * rng.standard_normal((k, n))).astype(np.float32)
    res = rng.standard_normal((rows, n)).astype(np.float32)
    wt = o.tile16(_dev(w))
    out, acc = torch.full((rows, n), float("nan"), device="cuda"), _dev(res)
    o.linear_rows_deep(out, _dev(x), wt)
    o.linear_rows_deep(acc, _dev(x), wt, mode=o.LINEAR_ACCUMULATE)
    torch.cuda.synchronize()
    want = x.astype(np.float64) @ w.astype(np.float64)
    _close(out.cpu().numpy(), want)
    _close(acc.cpu().numpy(), res + want)
    with pytest.raises(RuntimeError):  # deeper than the kernel
        o.linear_rows_deep(out, torch.zeros(rows, 2064, device="cuda"),
                           torch.zeros(-(-n // 16), 2064, 16, device="cuda"))


@pytest.mark.parametrize("layout", ["token", "head"])
@pytest.mark.parametrize("cache", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,wg_rows", [(1000, 32), (2741, 64)])
def test_many_rows_qkv_equals_projection_then_rope(layout, cache, rows, wg_rows):
    """Rows gathered by index with placeholders, copied to x_out, the record
    copied too: the same bits as the projection of the gathered rows followed
    by vl_rope_and_cache."""
    o = _ops()
    H, Hkv, D, k = 8, 4, 48, 384
    n = (H + 2 * Hkv) * D
    assert _rows_per_workgroup(rows, n, k, norm=True) == wg_rows
    blocks = -(-rows // 16)
    rng = np.random.default_rng(3)
    table = _dev(rng.standard_normal((261, k)).astype(np.float32))
    prev = _dev(rng.integers(0, 261, 12).astype(np.int32))
    ids_np = rng.integers(0, 261, rows).astype(np.int32)
    ids_np[[0, 500, rows - 1]] = [-1, -12, -13]  # -13: past num_prev -> id 0
    ids = _dev(ids_np)
    w = o.tile16(_dev((0.05 * rng.standard_normal((k, n))).astype(np.float32)))
    g = _dev((1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32))
    pos = _dev(rng.integers(0, 64, rows).astype(np.int32))
    slots = rng.permutation(16 * blocks)[:rows].astype(np.int32)
    slots[::7] = -1
    slot = _dev(slots)
    ang = rng.standard_normal((64, D // 2)).astype(np.float32)
    cos, sin = _dev(np.cos(ang)), _dev(np.sin(ang))
    shape = (blocks, Hkv, 16, D) if layout == "head" else (16 * blocks, Hkv, D)
    kc1, vc1, kc2, vc2 = (torch.zeros(shape, device="cuda", dtype=cache) for _ in range(4))
    q1, q2 = torch.empty((rows, H, D), device="cuda"), torch.empty((rows, H * D), device="cuda")
    x_out = torch.full((rows, k), float("nan"), device="cuda")
    rec = torch.arange(200001, dtype=torch.int32).pin_memory()
    rec_dst = torch.zeros(200001, dtype=torch.int32, device="cuda")
    o.qkv_rope_cache(q2, kc2, vc2, table, w, g, pos, slot, cos, sin, H, Hkv, D, row_index=ids,
                     x_out=x_out, prev_ids=prev, record=(rec, rec_dst))
    o.resolve_tokens(ids, prev)
    x = table[ids.long()].contiguous()
    qkv = torch.empty((rows, n), device="cuda")
    o.linear_rows(qkv, x, w, g, mode=o.LINEAR_STORE)
    o.rope_and_cache(qkv, q1, kc1, vc1, pos, slot, cos, sin, H, Hkv, D)
    torch.cuda.synchronize()
    assert torch.equal(q1.view(rows, -1), q2) and torch.equal(x_out, x)
    assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
    assert torch.equal(rec_dst.cpu(), rec)


@pytest.mark.parametrize("shape", [dict(n_heads=4, n_kv_heads=4, d_model=128, d_ff=1040),
                                   dict(n_heads=8, n_kv_heads=8, d_model=512, d_ff=2048),
                                   dict(n_heads=8, n_kv_heads=4, d_model=512, d_ff=512)])
def test_deeper_models_match_the_oracle_runner(shape):
    """Every step's logits of models whose down projection is deeper than
    vl_linear_rows takes, or whose decode steps keep wo out of the attention
    launch: within 2e-4 of each row's largest logit, as the other shapes."""
    from oracle.runner import NumpyRunner
    from vllmlite_amd.hip_runner import HipRunner
    cfg = small_cfg(layers=2)
    for f, v in shape.items():
        setattr(cfg.model, f, v)
    got = _logit_trace(HipRunner, cfg, PROMPTS, 6)
    want = _logit_trace(NumpyRunner, cfg, PROMPTS, 6)
    assert len(got) == len(want)
    for (g, dec), (w, _) in zip(got, want):
        scale = np.abs(w).max(axis=-1, keepdims=True)
        assert np.all(np.abs(g - w) <= 2e-4 * scale), f"decode step {dec}"


@pytest.mark.parametrize("lens,bucket", [((211, 300, 169), 1024), ((120, 99), 256)])
def test_long_prompts_through_the_runner(lens, bucket):
    """Prefill steps of a model with d_ff 2048 large enough that its
    projections take linear_tile_kernel (layer 0's gather, residual copy and
    record among them), with rows past the step's tokens in the bucket: the
    logits of that step and of the decodes after it, and every layer's cached
    K and V, against the oracle runner, within 2e-4 of the largest."""
    from oracle.runner import NumpyRunner
    from vllmlite_amd.hip_runner import HipRunner
    cfg = small_cfg(layers=2)
    for f, v in dict(n_heads=8, n_kv_heads=8, d_model=512, d_ff=2048).items():
        setattr(cfg.model, f, v)
    assert bucket // 2 < sum(n + 1 for n in lens) < bucket
    assert _rows_per_workgroup(bucket, 2048, 512, "swiglu", True) == (64 if bucket == 1024 else 32)
    rng = np.random.default_rng(bucket)
    prompts = ["".join(chr(c) for c in rng.integers(32, 127, n)) for n in lens]
    runners = []

    def made(cls):
        return lambda m, c: runners.append(cls(m, c)) or runners[-1]

    got = _logit_trace(made(HipRunner), cfg, prompts, 3)
    want = _logit_trace(made(NumpyRunner), cfg, prompts, 3)
    assert len(got) == len(want)
    for (g, dec), (w, _) in zip(got, want):
        assert np.all(np.abs(g - w) <= 2e-4 * np.abs(w).max(axis=-1, keepdims=True)), dec
    for name in ("cache_k", "cache_v"):
        g, w = getattr(runners[0], name).cpu().numpy(), getattr(runners[1], name)
        assert np.abs(g - w).max() <= 2e-4 * np.abs(w).max(), name
