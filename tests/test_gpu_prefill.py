"""Varlen prefill ops vs the CPU oracle: packed new-token attention (the reference's op) and
causal prefill over paged, optionally quantized KV with a cached context (this build's extension)."""

import ctypes

import pytest
import torch

from areno_amd import workloads
from areno_amd.accel import attention as ops
from areno_amd.accel import cabi
from oracle import attention_ref as ar
from tests.gpu_util import DEV, assert_close, compact_pages, dequant_cpu, gpu_quantize, tolerances

pytestmark = pytest.mark.gpu


def _packed(lens, hq, hkv, d, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    t = sum(lens)
    q, k, v = (torch.randn(t, h, d, generator=g).to(dtype) for h in (hq, hkv, hkv))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    return q, k, v, cu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("window_left", [None, 0, 7])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 64), (28, 4, 128), (4, 4, 80), (8, 2, 256), (6, 6, 192), (8, 2, 512), (40, 2, 128)])
def test_varlen_new_tokens_only(dtype, window_left, hq, hkv, d):
    q, k, v, cu = _packed([5, 1, 130, 0, 67], hq, hkv, d, dtype)
    out = ops.areno_varlen_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), window_left=window_left)
    want = ar.ref_varlen(q, k, v, cu, ar.window_left_arg(window_left), d**-0.5)
    assert out.dtype == dtype and out.shape == q.shape
    assert_close(out, want, *tolerances("bf16"), what="varlen")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128, 192, 256, 512])
@pytest.mark.parametrize("profile", ["climb", "jump", "fall", "wide"])
def test_varlen_score_ranges_that_move_along_the_keys(dtype, d, profile):
    """The matrix-core kernel keeps a softmax reference value per row that it raises only when a key tile exceeds it
    by a margin, so rows whose scores climb slowly (the reference lags), jump far (a late raise rescales everything
    before it), fall (the first tile dominates) or spread over a wide range all have to come out like the oracle's
    exact-maximum softmax."""
    lens = [300, 33, 1, 150]
    q, k, v, cu = _packed(lens, 4, 2, d, torch.float32, seed=d)
    pos = torch.cat([torch.arange(n, dtype=torch.float32) for n in lens])
    if profile == "climb":  # a shared direction whose weight grows by a little per key
        gain = 0.02 * pos
    elif profile == "jump":  # every 97th key scores far above its neighbours
        gain = torch.where(pos % 97 == 96, 9.0, 0.0)
    elif profile == "fall":
        gain = 6.0 - 0.03 * pos
    else:
        gain = torch.zeros_like(pos)
        q, k = 5.0 * q, 5.0 * k
    direction = torch.ones(d) * (d**-0.5)
    q = q + 2.0 * (d**0.25) * direction  # every query has a component along the shared direction
    k = k + gain[:, None, None] * (d**0.25) * direction
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    out = ops.areno_varlen_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV))
    want = ar.ref_varlen(q, k, v, cu, ar.window_left_arg(None), d**-0.5)
    assert_close(out, want, *tolerances("bf16"), what=f"varlen {profile}")


def _expected_prefill(w, window_left=None):
    kc, vc = dequant_cpu(w.k_cache, w.k_scale), dequant_cpu(w.v_cache, w.v_scale)
    return ar.ref_paged_varlen_prefill(w.q.cpu().float(), kc, vc, w.block_table.cpu(), w.cu_seqlens_q.cpu(),
                                       w.context_lens.cpu(), ar.window_left_arg(window_left), w.softmax_scale)  # fmt: skip


def _run_prefill(w, window_left=None):
    return ops.areno_paged_varlen_causal_attention(
        w.q, w.k_cache, w.v_cache, w.block_table, w.cu_seqlens_q, w.context_lens,
        window_left=window_left, softmax_scale=w.softmax_scale, k_scale=w.k_scale, v_scale=w.v_scale,
    )  # fmt: skip


@pytest.mark.parametrize("kv", ["bf16", "fp16", "int8", "fp8"])
@pytest.mark.parametrize("window_left", [None, 33])
def test_paged_prefill_small(kv, window_left):
    w = workloads.cfg4_prefill(kv, device=DEV, seqs=5, new_hi=70, ctx_hi=300, quantize_fn=gpu_quantize, seed=5)
    out = _run_prefill(w, window_left)
    assert_close(out, _expected_prefill(w, window_left), *tolerances(kv), what=f"paged prefill {kv}")


@pytest.mark.parametrize("hq,hkv,d,bs", [
    (28, 4, 128, 16), (8, 8, 64, 32), (6, 2, 128, 256), (4, 1, 96, 16),
    # more than 16 q heads per kv head: several workgroup rows per kv head, 16 q heads each (16 + 16, 16 + 4, 16 + 8 at
    # head dim 256, 16 + 16 + 1)
    (32, 1, 128, 16), (40, 2, 64, 32), (24, 1, 256, 16), (33, 1, 128, 16),
    # page sizes that are no power of two: the key's page by a multiplication and a shift
    (28, 4, 128, 12), (8, 2, 64, 48), (16, 8, 512, 80), (8, 8, 128, 1000),
])  # fmt: skip
def test_paged_prefill_shapes(hq, hkv, d, bs):
    g = torch.Generator().manual_seed(d + hq)
    new = torch.tensor([1, 64, 17, 129])
    ctx = torch.tensor([0, 5, 200, 63])
    w = workloads.make_prefill_workload("shapes", seed=3, new_lens=new, ctx_lens=ctx, hq=hq, hkv=hkv, d=d, bs=bs,
                                        kv="bf16", device=DEV)  # fmt: skip
    assert_close(_run_prefill(w), _expected_prefill(w), *tolerances("bf16"), what="prefill shapes")


@pytest.mark.parametrize("kv", ["bf16", "fp16", "int8", "fp8"])
@pytest.mark.parametrize("d", [256, 192, 512])
@pytest.mark.parametrize("hq,hkv,window_left", [(16, 8, None), (8, 1, 40), (12, 4, None)])
def test_paged_prefill_head_dims_192_256_512(kv, d, hq, hkv, window_left):
    """Head dims 256 (the sliding-attention layers of the Gemma family, Qwen3.5), 192 (128 + 64 rotary channels of
    the MLA-style layers) and 512 (the Gemma family's full-attention layers) on the matrix-core kernel: one 16-row
    tile per wave, at 512 shared by two waves with half of the head each; a query block cut by many shares goes
    through the merge of the wide partials."""
    new = torch.tensor([3, 150, 64, 1, 33])
    ctx = torch.tensor([900, 0, 77, 2500, 310])
    w = workloads.make_prefill_workload("wide", seed=11 + hq, new_lens=new, ctx_lens=ctx, hq=hq, hkv=hkv, d=d, bs=16,
                                        kv=kv, device=DEV, quantize_fn=gpu_quantize)  # fmt: skip
    assert_close(_run_prefill(w, window_left), _expected_prefill(w, window_left), *tolerances(kv),
                 what=f"prefill D={d} {kv}")  # fmt: skip


@pytest.mark.parametrize("kv", ["bf16", "fp16", "int8", "fp8"])
@pytest.mark.parametrize("d,bs", [(64, 16), (64, 64), (128, 8), (128, 128), (64, 24), (128, 5), (128, 100)])
def test_paged_prefill_staging_schemes(kv, d, bs):
    """The staging of a key tile has two schemes: one K and one V chunk per thread and round, or, when a tile has at
    most one chunk per thread (8-bit tiles up to head dim 128, 16-bit tiles at 64), K staged by the first half of
    the workgroup and V by the second.  8-bit tiles at head dim 64 leave half of each half without a live chunk.
    Page sizes below, at and above the 32-key tile, powers of two and others."""
    new = torch.tensor([70, 1, 200, 33])
    ctx = torch.tensor([0, 1300, 95, 640])
    w = workloads.make_prefill_workload("staging", seed=d + bs, new_lens=new, ctx_lens=ctx, hq=8, hkv=2, d=d, bs=bs,
                                        kv=kv, device=DEV, quantize_fn=gpu_quantize)  # fmt: skip
    assert_close(_run_prefill(w), _expected_prefill(w), *tolerances(kv), what=f"prefill staging D={d} {kv} page {bs}")


@pytest.mark.parametrize("seed", range(32))
def test_random_draws_of_prefill_shape_length_window_and_cache_type(seed):
    """Seeded random configurations through the paged prefill op: cache type, head counts (up to 33 q heads per kv
    head: several workgroup rows per kv head), head dim (one tile or two per wave, the head split over two waves at
    512, 96 on the one-wave-per-row kernel), page size (12 and 48: no power of two), number of sequences, new and
    cached lengths (sequences without new tokens, single tokens, blocks cut by many shares) and window."""
    import random

    rng = random.Random(7000 + seed)
    kv = rng.choice(["bf16", "fp16", "int8", "fp8"])
    group = rng.choice([1, 2, 4, 7, 8, 16, 20, 33])
    hkv = rng.choice([h for h in (1, 2, 4, 8) if h * group <= 64])
    d = rng.choice([64, 128, 128, 192, 256, 512, 96])
    bs = rng.choice([8, 16, 32, 64, 256, 12, 48])
    slow = d == 96  # one wave per (token, head): keep the work small
    seqs = rng.choice([1, 3, 9] if slow else [1, 3, 9, 40])
    g = torch.Generator().manual_seed(seed)
    new_profile = rng.choice(["ones", "short", "mixed", "long"])
    if new_profile == "ones":
        new = torch.randint(0, 2, (seqs,), generator=g)
    elif new_profile == "short":
        new = torch.randint(0, 20, (seqs,), generator=g)
    elif new_profile == "mixed":
        new = torch.where(torch.rand(seqs, generator=g) < 0.6, torch.randint(0, 9, (seqs,), generator=g),
                          torch.randint(60, 300, (seqs,), generator=g))  # fmt: skip
    else:
        new = torch.randint(100, 140 if slow else 400, (seqs,), generator=g)
    if int(new.sum()) == 0:
        new[0] = 1
    ctx_hi = 300 if slow else rng.choice([1, 90, 700, 4000])
    ctx = torch.where(torch.rand(seqs, generator=g) < 0.3, torch.zeros(seqs, dtype=torch.int64),
                      torch.randint(0, ctx_hi, (seqs,), generator=g))  # fmt: skip
    window = rng.choice([None, None, 0, 33, 700])
    w = workloads.make_prefill_workload(f"draw-{seed}", seed=900 + seed, new_lens=new, ctx_lens=ctx, hq=hkv * group,
                                        hkv=hkv, d=d, bs=bs, kv=kv, device=DEV, quantize_fn=gpu_quantize,
                                        act_dtype=torch.float16 if kv == "fp16" else torch.bfloat16)  # fmt: skip
    what = f"draw {seed}: {kv} {hkv * group}/{hkv} d={d} bs={bs} seqs={seqs} new={new_profile} ctx<{ctx_hi} window={window}"
    assert_close(_run_prefill(w, window), _expected_prefill(w, window), *tolerances(kv), what=what)


def test_prefill_with_a_full_sequence_list():
    """1024 sequences, the most one launch of the matrix-core kernel indexes: the prefix sum over the sequences must
    also produce its last entry, the total."""
    g = torch.Generator().manual_seed(3)
    new = torch.randint(1, 4, (1024,), generator=g)
    ctx = torch.randint(0, 40, (1024,), generator=g)
    w = workloads.make_prefill_workload("full-list", seed=31, new_lens=new, ctx_lens=ctx, hq=4, hkv=2, d=64, bs=16,
                                        kv="bf16", device=DEV)  # fmt: skip
    assert_close(_run_prefill(w), _expected_prefill(w), *tolerances("bf16"), what="1024 sequences")


def test_write_then_prefill_then_decode_are_consistent():
    """The three ops agree with each other: cache write of the new tokens, prefill with ctx,
    and n = 1 prefill == decode without append."""
    w = workloads.cfg4_prefill("fp8", device=DEV, seqs=6, new_hi=40, ctx_hi=200, quantize_fn=gpu_quantize, seed=9)
    ops.areno_paged_cache_write(w.k_new, w.v_new, w.k_cache, w.v_cache, w.cache_block_ids, w.cache_block_offsets,
                                k_scale=w.k_scale, v_scale=w.v_scale)  # fmt: skip
    out = _run_prefill(w)
    assert_close(out, _expected_prefill(w), *tolerances("fp8"), what="after write")
    # last query of each sequence == a decode row whose token is already cached: compare through the oracle
    cu = w.cu_seqlens_q.cpu().long()
    last = cu[1:] - 1
    lens = (w.context_lens.cpu().long() + (cu[1:] - cu[:-1]) - 1).int()
    kc, vc = dequant_cpu(w.k_cache, w.k_scale), dequant_cpu(w.v_cache, w.v_scale)
    dec = ar.ref_paged_decode(w.q.cpu().float()[last], kc, vc, w.block_table.cpu(), lens, -1, w.softmax_scale)
    assert_close(out[last.to(DEV)], dec, *tolerances("fp8"), what="prefill last row vs decode oracle")


def test_cfg4_reduced():
    """cfg 4 shape (32/8 heads, D=128, fp8) with the full range of new lengths and a reduced context range."""
    w = workloads.cfg4_prefill("fp8", device=DEV, seqs=6, new_hi=512, ctx_hi=3000, quantize_fn=gpu_quantize)
    assert_close(_run_prefill(w), _expected_prefill(w), *tolerances("fp8"), what="cfg4 reduced")


def test_cfg4_full_size():
    """cfg 4 at its stated size: 16 sequences, 1..512 new tokens on 0..16 384 cached ones, 32 / 8 heads, fp8 pages.  The new
    tokens go through the quantizing cache write first, as in the op sequence the benchmark times.  Every sequence is checked
    against the oracle on its first and last query row and 16 random ones in between (a row sees all of its sequence's keys
    up to its own position, so the long contexts are covered by every sampled row)."""
    w = workloads.cfg4_prefill("fp8", device=DEV, quantize_fn=gpu_quantize)
    assert w.context_lens.shape == (16,)
    ops.areno_paged_cache_write(w.k_new, w.v_new, w.k_cache, w.v_cache, w.cache_block_ids, w.cache_block_offsets,
                                k_scale=w.k_scale, v_scale=w.v_scale)  # fmt: skip
    out = _run_prefill(w)
    torch.cuda.synchronize()
    got = out.cpu().float()
    assert torch.isfinite(got).all()
    cu = w.cu_seqlens_q.cpu().tolist()
    ctx = w.context_lens.cpu().tolist()
    print(f"cfg4 full: new {[cu[i + 1] - cu[i] for i in range(16)]} ctx {ctx}")
    g = torch.Generator().manual_seed(4)
    hq, hkv = w.q.shape[1], w.k_cache.shape[2]
    worst = 0.0
    for s in range(16):
        n = cu[s + 1] - cu[s]
        picks = sorted({0, n - 1} | set(torch.randint(0, n, (16,), generator=g).tolist()))
        bs = w.k_cache.shape[1]
        cols = (ctx[s] + n + bs - 1) // bs
        table = w.block_table[s : s + 1, :cols].cpu()
        kc, compact = compact_pages(w.k_cache, w.k_scale, table)
        vc, _ = compact_pages(w.v_cache, w.v_scale, table)
        k = ar.gather_paged(kc, compact[0], ctx[s] + n).repeat_interleave(hq // hkv, dim=1).transpose(0, 1).unsqueeze(0)
        v = ar.gather_paged(vc, compact[0], ctx[s] + n).repeat_interleave(hq // hkv, dim=1).transpose(0, 1).unsqueeze(0)
        for i in picks:
            upto = ctx[s] + i + 1
            q1 = w.q[cu[s] + i].cpu().float().view(1, hq, 1, -1)
            want = ar.ref_attention(q1, k[:, :, :upto], v[:, :, :upto], ctx[s] + i, -1, w.softmax_scale).view(hq, -1)
            err = (got[cu[s] + i] - want).abs().max().item()
            worst = max(worst, err)
            assert err <= tolerances("fp8")[0], f"cfg4 full: sequence {s} (ctx {ctx[s]}, new {n}) row {i}: max-abs {err:.4g}"
    print(f"cfg4 full: max-abs {worst:.3e} over the sampled rows")


@pytest.mark.parametrize("kv", ["bf16", "int8"])
def test_prefill_one_query_block_cut_by_many_shares(kv):
    """A single short chunk on a long context: every workgroup owns a slice of the same query block's keys, so the
    result only exists after the merge of all their partials."""
    w = workloads.make_prefill_workload("long-ctx", seed=21, new_lens=torch.tensor([9]), ctx_lens=torch.tensor([6000]),
                                        hq=8, hkv=2, d=128, bs=16, kv=kv, device=DEV, quantize_fn=gpu_quantize)  # fmt: skip
    assert_close(_run_prefill(w), _expected_prefill(w), *tolerances(kv), what="one block, many shares")


@pytest.mark.parametrize("hq,hkv", [(4, 1), (8, 2), (16, 8), (40, 2)])
@pytest.mark.parametrize("lens,ctxs", [([5], [1600]), ([40], [1600]), ([3, 70], [0, 900]), ([1, 0, 2, 90], [700, 5, 350, 0]), ([200] * 9, [40] * 9)])
def test_prefill_few_items_over_many_shares(hq, hkv, lens, ctxs):
    """The merge looks its items up among the units (256 of a lone kv head) when the tokens allow fewer items than units:
    one item in dozens of pieces (and batches), items in units far apart, units without steps, as many items as units.
    The bar is the file's."""
    w = workloads.make_prefill_workload("few items", seed=hq, new_lens=torch.tensor(lens), ctx_lens=torch.tensor(ctxs), hq=hq, hkv=hkv,
                                        d=64, bs=16, kv="bf16", device=DEV, quantize_fn=gpu_quantize)  # fmt: skip
    assert_close(_run_prefill(w), _expected_prefill(w), *tolerances("bf16"), what=f"{hq}/{hkv} {lens[:4]}")


def test_prefill_sequences_without_new_tokens_and_single_tokens():
    """Empty chunks (cu_seqlens repeats) between chunks of 1, 33 and 200 tokens; contexts 0, tile-aligned and odd."""
    new = torch.tensor([0, 1, 0, 33, 1, 0, 200, 0])
    ctx = torch.tensor([50, 0, 0, 64, 1023, 7, 31, 0])
    w = workloads.make_prefill_workload("ragged", seed=22, new_lens=new, ctx_lens=ctx, hq=12, hkv=4, d=64, bs=32,
                                        kv="fp8", device=DEV, quantize_fn=gpu_quantize)  # fmt: skip
    assert_close(_run_prefill(w), _expected_prefill(w), *tolerances("fp8"), what="ragged chunks")


@pytest.mark.parametrize("window_left", [0, 31, 32, 100, 5000])
def test_prefill_window_moves_the_first_tile(window_left):
    """Sliding windows shorter than, equal to and longer than a key tile, and longer than every context."""
    new = torch.tensor([70, 3, 130])
    ctx = torch.tensor([900, 40, 0])
    w = workloads.make_prefill_workload("window", seed=23, new_lens=new, ctx_lens=ctx, hq=8, hkv=2, d=128, bs=16,
                                        kv="bf16", device=DEV)  # fmt: skip
    assert_close(_run_prefill(w, window_left), _expected_prefill(w, window_left), *tolerances("bf16"),
                 what=f"window {window_left}")  # fmt: skip


def test_prefill_many_sequences():
    """More sequences than workgroup shares per kv head: most shares hold several whole query blocks."""
    g = torch.Generator().manual_seed(24)
    new = torch.randint(1, 40, (300,), generator=g)
    ctx = torch.randint(0, 90, (300,), generator=g)
    w = workloads.make_prefill_workload("many", seed=24, new_lens=new, ctx_lens=ctx, hq=8, hkv=8, d=64, bs=16,
                                        kv="int8", device=DEV, quantize_fn=gpu_quantize)  # fmt: skip
    assert_close(_run_prefill(w), _expected_prefill(w), *tolerances("int8"), what="many sequences")


def test_prefill_c_abi_rejects_a_short_workspace():
    from areno_amd.accel import cabi

    w = workloads.cfg4_prefill("fp8", device=DEV, seqs=2, new_hi=8, ctx_hi=40, quantize_fn=gpu_quantize, seed=5)
    cache = cabi.describe_cache(w.k_cache, w.v_cache, w.k_scale, w.v_scale)
    need = cabi.prefill_workspace_bytes(w.k_cache.shape[2], w.k_cache.shape[3])
    assert need > 0
    out = torch.empty_like(w.q)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)

    def call(nbytes):
        return cabi.paged_varlen_prefill(cache, w.q, out, w.block_table, w.cu_seqlens_q, w.context_lens, ws,
                                         softmax_scale=w.softmax_scale, workspace_bytes=nbytes)  # fmt: skip

    assert call(need - 1) == cabi.ERR_WORKSPACE
    assert b"workspace" in cabi.lib().areno_hip_last_error()
    assert call(need) == 0
    torch.cuda.synchronize()
    assert_close(out, _expected_prefill(w), *tolerances("fp8"), what="c abi prefill")


def test_dense_causal_attention_wrapper():
    g = torch.Generator().manual_seed(1)
    q = torch.randn(2, 4, 9, 64, generator=g).bfloat16()
    k = torch.randn(2, 4, 21, 64, generator=g).bfloat16()
    v = torch.randn(2, 4, 21, 64, generator=g).bfloat16()
    out = ops.areno_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), query_start=12, window_left=6)
    want = ar.ref_attention(q, k, v, 12, 6, 64**-0.5)
    assert_close(out, want, *tolerances("bf16"), what="dense")


def test_varlen_error_behaviour():
    q, k, v, cu = _packed([4, 4], 4, 2, 64, torch.bfloat16)
    with pytest.raises(RuntimeError, match="requires CUDA"):
        ops.areno_varlen_causal_attention(q, k, v, cu)
    q, k, v, cu = (t.to(DEV) for t in (q, k, v, cu))
    with pytest.raises(ValueError, match="int32 1D cu_seqlens"):
        ops.areno_varlen_causal_attention(q, k, v, cu.long())
    with pytest.raises(ValueError, match="token count mismatch"):
        ops.areno_varlen_causal_attention(q, k[:-1], v, cu)
    with pytest.raises(ValueError, match="divisible by kv heads"):
        ops.areno_varlen_causal_attention(q[:, :3], k, v, cu)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,window_left", [
    (28, 4, 128, None), (7, 1, 128, 63), (4, 4, 64, None), (3, 1, 64, 64), (20, 1, 128, None), (4, 2, 256, None),
    (6, 6, 192, 31), (8, 1, 256, 33),
])  # fmt: skip
@pytest.mark.parametrize("lens", [
    [1], [18, 19], [127, 128, 129], [63, 0, 64, 65, 1, 300], [3] * 70, [0] * 64 + [40, 0, 200], [5, 1, 0] * 50,
])  # fmt: skip
def test_varlen_query_blocks_and_key_tiles(dtype, hq, hkv, d, window_left, lens):
    """Packed attention at the edges of its query blocks (128 rows: 128 tokens of one head, 18 of seven, 8 of sixteen),
    of its key tiles (64 keys, 32 at the wide heads) and of its block list (up to 64 sequences in one lane each, more
    in rounds; empty ones between).  Tolerance: that of the file's other 16-bit outputs against the fp32 oracle, and in
    the 2-norm what the type gives: the output is rounded to 8 (bf16) or 11 bits, and so are the probabilities, each
    by at most half a unit."""
    q, k, v, cu = _packed(lens, hq, hkv, d, dtype, seed=d + len(lens))
    out = ops.areno_varlen_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), window_left=window_left)
    want = ar.ref_varlen(q, k, v, cu, ar.window_left_arg(window_left), d**-0.5)
    what = f"varlen {hq}/{hkv} d={d} window={window_left} lens={lens[:6]}"
    assert_close(out, want, *tolerances("bf16"), what=what)
    err = ((out.cpu().float() - want).norm() / want.norm()).item()
    assert err <= (2.0**-8 if dtype == torch.bfloat16 else 2.0**-11), f"{what}: {err:.3g} in the 2-norm"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(129, 1, 64), (320, 2, 128), (136, 1, 256)])
def test_packed_calls_of_the_generic_kernel_stay_there(dtype, hq, hkv, d):
    """More than 128 q heads per kv head have no matrix-core launch: such calls are computed in fp32 like fp32 inputs,
    and rounded once, bit for bit."""
    q, k, v, cu = _packed([40, 0, 1, 90], hq, hkv, d, dtype, seed=hq)
    q, k, v, cu = (x.to(DEV) for x in (q, k, v, cu))
    want = ops.areno_varlen_causal_attention(q.float(), k.float(), v.float(), cu).to(dtype)
    assert torch.equal(ops.areno_varlen_causal_attention(q, k, v, cu), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128, 192, 256, 512])
def test_packed_calls_without_their_workspace_are_refused(dtype, d):
    """The C entry's contract: 16-bit inputs come with the workspace that areno_hip_prefill_workspace_bytes names."""
    q, k, v, cu = (x.to(DEV) for x in _packed([40, 9], 4, 2, d, dtype, seed=d))
    out = torch.full_like(q, float("nan"))
    need = cabi.prefill_workspace_bytes(2, d)
    workspace = torch.empty(need, dtype=torch.uint8, device=DEV)
    for ptr, size in ((None, need), (workspace.data_ptr(), need - 1), (workspace.data_ptr(), need)):
        status = cabi.lib().areno_hip_varlen_attention(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), cabi.dtype_code(q), q.shape[0], 4, 2, d,
            cu.data_ptr(), 2, -1, d**-0.5, ptr, size, cabi.current_stream_ptr())  # fmt: skip
        torch.cuda.synchronize()
        served = ptr is not None and size == need
        assert (status == 0) == served
        assert torch.isfinite(out).all() if served else torch.isnan(out).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens,hq,hkv,d,window_left", [
    ([6143], 1, 1, 128, None), ([6145], 1, 1, 128, None), ([4099], 3, 3, 64, None), ([4100, 4095], 2, 2, 64, None),
    ([4097], 2, 1, 192, None), ([2047], 2, 1, 256, None), ([2049], 2, 1, 256, None), ([4500], 1, 1, 256, 4100),
    ([8300, 40], 1, 1, 64, None),
])  # fmt: skip
def test_packed_calls_of_few_heads_and_long_sequences(dtype, lens, hq, hkv, d, window_left):
    """Launches on either side of the rule that gives few heads over long sequences to the kernel that cuts blocks into
    equal shares.  Tolerance as in the file's other 16-bit outputs against the fp32 oracle."""
    q, k, v, cu = _packed(lens, hq, hkv, d, dtype, seed=sum(lens))
    out = ops.areno_varlen_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), window_left=window_left)
    want = ar.ref_varlen(q, k, v, cu, ar.window_left_arg(window_left), d**-0.5)
    assert_close(out, want, *tolerances("bf16"), what=f"varlen {hq}/{hkv} d={d} window={window_left} lens={lens}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("lens,hq,hkv,d", [
    ([5, 0, 130], 7, 1, 64), ([128, 127], 6, 6, 128), ([1], 4, 2, 128), ([60], 4, 4, 192), ([40, 33], 20, 1, 256),
    ([90, 7], 4, 2, 512), ([30], 4, 2, 96), ([2] * 70, 28, 4, 128), ([0, 0], 3, 1, 64), ([2100], 2, 1, 256),
])  # fmt: skip
@pytest.mark.parametrize("behind", [1, 37, 1500])
def test_rows_behind_the_last_sequence_are_zeros(dtype, lens, hq, hkv, d, behind):
    """A padded pack (``cu_seqlens[-1]`` below the tokens): the output's last rows are written, as zeros, whatever their
    inputs hold, and the others are what they are without the padding."""
    q, k, v, cu = (x.to(DEV) for x in _packed(lens, hq, hkv, d, dtype, seed=d))
    want = ops.areno_varlen_causal_attention(q, k, v, cu) if sum(lens) else q
    pads = [torch.full((behind, *x.shape[1:]), float("nan"), dtype=dtype, device=DEV) for x in (q, k, v)]
    q, k, v = (torch.cat(pair) for pair in zip((q, k, v), pads))
    out = torch.full_like(q, float("nan"))
    workspace = torch.empty(cabi.prefill_workspace_bytes(hkv, d), dtype=torch.uint8, device=DEV)
    cabi.check(cabi.lib().areno_hip_varlen_attention(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), cabi.dtype_code(q), q.shape[0], hq, hkv, d,
        cu.data_ptr(), len(lens), -1, d**-0.5, workspace.data_ptr(), workspace.numel(), cabi.current_stream_ptr()), "varlen")  # fmt: skip
    assert (out[sum(lens) :] == 0).all()
    if sum(lens):
        assert_close(out[: sum(lens)], want.cpu().float(), *tolerances("bf16"), what="rows in front of the padding")


@pytest.mark.parametrize("kv", ["bf16", "int8"])
@pytest.mark.parametrize("d,page", [(128, 16), (256, 24), (512, 16), (96, 16)])
@pytest.mark.parametrize("behind", [1, 600])
def test_paged_rows_behind_the_last_sequence_are_zeros(kv, d, page, behind):
    new, ctx = torch.tensor([3, 150, 0, 33]), torch.tensor([900, 0, 77, 31])
    w = workloads.make_prefill_workload("padded", seed=d, new_lens=new, ctx_lens=ctx, hq=8, hkv=2, d=d, bs=page, kv=kv,
                                        device=DEV, quantize_fn=gpu_quantize)  # fmt: skip
    q = torch.cat([w.q, torch.full((behind, *w.q.shape[1:]), float("nan"), dtype=w.q.dtype, device=DEV)])
    out = torch.full_like(q, float("nan"))
    workspace = torch.empty(cabi.prefill_workspace_bytes(2, d), dtype=torch.uint8, device=DEV)
    cache = cabi.describe_cache(w.k_cache, w.v_cache, w.k_scale, w.v_scale)
    cabi.check(cabi.paged_varlen_prefill(cache, q, out, w.block_table, w.cu_seqlens_q, w.context_lens, workspace), "prefill")
    assert (out[w.q.shape[0] :] == 0).all()
    assert_close(out[: w.q.shape[0]], _run_prefill(w).cpu().float(), *tolerances(kv), what="rows in front of the padding")


def _errors(out, q, k, v, lens, ctx):
    """Relative distance from 64 bits of ``out``, and of attention whose only roundings are those of the probabilities, against
    the row's largest score, and of the result; a row's sum is that of the rounded probabilities, as in the kernels."""
    G, num, rounded, den, a, b = q.shape[1] // k.shape[1], 0.0, 0.0, 0.0, 0, 0
    for n, c in zip(lens, ctx):
        hidden = torch.arange(n + c)[None] > torch.arange(c, c + n)[:, None]
        for h in range(q.shape[1]):
            keys, values = k[b : b + n + c, h // G].double(), v[b : b + n + c, h // G].double()
            s = (q[a : a + n, h].double() @ keys.T * q.shape[2] ** -0.5).masked_fill(hidden, -float("inf"))
            p = (s - s.amax(1, keepdim=True)).exp()
            p16 = p.to(out.dtype).double()
            want, near = p @ values / p.sum(1, keepdim=True), p16 @ values / p16.sum(1, keepdim=True)
            num += (out[a : a + n, h].double() - want).square().sum().item()
            rounded += (near.to(out.dtype).double() - want).square().sum().item()
            den += want.square().sum().item()
        a, b = a + n, b + n + c
    return (num / den) ** 0.5, (rounded / den) ** 0.5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens", [[48] * 60, [64] * 60, list(range(33, 65)) * 2])
def test_short_sequences_are_as_precise_as_their_rounded_probabilities(dtype, lens):
    """Steps of 32 keys (which launches of up to 64 tokens a sequence take) start a row with a reference that a later step may exceed;
    short sequences' probabilities are still rounded as finely as against the row's maximum.  The bound's margin is for the sums' order, some 1e-4 of a rounding."""
    q, k, v, cu = _packed(lens, 8, 2, 128, dtype)
    out = ops.areno_varlen_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV)).cpu()
    error, bound = _errors(out, q, k, v, lens, [0] * len(lens))
    assert error <= bound * 1.0003, (error, bound)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(28, 4, 128), (8, 1, 128), (8, 2, 64), (8, 4, 256)])
@pytest.mark.parametrize("new,ctx", [([64], [600]), ([16], [3000]), ([60, 20, 50, 44], [400, 100, 300, 20])])
def test_paged_prefill_of_few_items_is_as_precise_as_its_rounded_probabilities(dtype, hq, hkv, d, new, ctx):
    """Units of one item have more steps than equal shares; their probabilities are rounded as finely as against the row's
    maximum all the same."""
    g = torch.Generator().manual_seed(d)
    total, bs = [n + c for n, c in zip(new, ctx)], 16
    k, v = (torch.randn(sum(total), hkv, d, generator=g).to(dtype) for _ in range(2))
    q = torch.randn(sum(new), hq, d, generator=g).to(dtype)
    pages = [-(-n // bs) for n in total]
    table, ids, offs, first = torch.zeros(len(new), max(pages), dtype=torch.int32), [], [], 0
    for i, n in enumerate(total):
        table[i, : pages[i]] = torch.arange(first, first + pages[i])
        ids.append(first + torch.arange(n) // bs)
        offs.append(torch.arange(n) % bs)
        first += pages[i]
    k_cache, v_cache = (torch.zeros(first, bs, hkv, d, dtype=dtype, device=DEV) for _ in range(2))
    ops.areno_paged_cache_write(k.to(DEV), v.to(DEV), k_cache, v_cache, torch.cat(ids).to(DEV), torch.cat(offs).to(DEV))
    cu = torch.tensor([0] + new).cumsum(0).to(torch.int32)
    out = ops.areno_paged_varlen_causal_attention(q.to(DEV), k_cache, v_cache, table.to(DEV), cu.to(DEV), torch.tensor(ctx, dtype=torch.int32, device=DEV)).cpu()
    error, bound = _errors(out, q, k, v, new, ctx)
    assert error <= bound * 1.001, (error, bound)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(7, 1, 128), (2, 2, 64), (3, 1, 192)])
@pytest.mark.parametrize("lens", [
    [2] * 256, [2] * 257, [1] * 1000 + [150] * 24, [7, 0] * 512, [0] * 1023 + [300], [40] + [0, 3] * 300, [1] * 1025,
])  # fmt: skip
def test_varlen_of_many_sequences(dtype, hq, hkv, d, lens):
    """Up to 256 and up to 1 024 sequences have their block counts in four and sixteen registers per lane; more take the
    generic kernel.  Tolerance as in the file's other 16-bit outputs against the fp32 oracle."""
    q, k, v, cu = _packed(lens, hq, hkv, d, dtype, seed=len(lens))
    out = ops.areno_varlen_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV))
    want = ar.ref_varlen(q, k, v, cu, -1, d**-0.5)
    assert_close(out, want, *tolerances("bf16"), what=f"varlen of {len(lens)} sequences {hq}/{hkv} d={d}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("window_left", [None, 100])
@pytest.mark.parametrize("lens,hq,hkv", [([701, 390], 28, 4), ([450, 351], 3, 3), ([701, 1, 64], 8, 2), ([129] * 40 + [1], 16, 16)])
def test_varlen_steps_of_either_length(dtype, window_left, lens, hq, hkv):
    """Head dim 128 has kernels with steps of 64 and of 32 keys: few long blocks, and short sequences or many blocks."""
    q, k, v, cu = _packed(lens, hq, hkv, 128, dtype)
    out = ops.areno_varlen_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), window_left=window_left)
    want = ar.ref_varlen(q, k, v, cu, ar.window_left_arg(window_left), 128**-0.5)
    assert_close(out, want, *tolerances("bf16"), what="varlen")


@pytest.mark.parametrize("kv", ["same", "int8", "fp8"])
@pytest.mark.parametrize("act", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(28, 4, 128), (16, 16, 64), (6, 6, 256), (8, 1, 256), (24, 8, 192), (40, 2, 128), (3, 3, 128)])
@pytest.mark.parametrize("lens", [[1, 33, 0, 130, 64, 257, 18], [701, 390]])
def test_prefill_with_its_cache_write(kv, act, hq, hkv, d, lens):
    """One op for the cache write and the packed attention leaves the bits of the two ops: tokens of every place in a block and a
    key tile, empty sequences, tokens in front of the first sequence and behind the last, ids outside the pool, a window."""
    cache_dtype, scale_dtype = {"same": (act, None), "int8": (torch.int8, torch.float16), "fp8": (torch.float8_e4m3fn, torch.float32)}[kv]
    front, behind, bs = 3, 5, 16
    t = front + sum(lens) + behind
    g = torch.Generator().manual_seed(d + hq)
    q, k, v = (torch.randn(t, h, d, generator=g).to(act).to(DEV) for h in (hq, hkv, hkv))
    k[7], v[9] = 0, 1e4
    cu = (front + torch.tensor([0] + lens).cumsum(0)).to(torch.int32).to(DEV)
    blocks = t // bs + 2
    slots = torch.randperm(blocks * bs, generator=g)[:t].to(DEV)
    ids, offs = slots // bs, slots % bs
    ids[11], offs[12], ids[13], offs[14] = -1, bs, blocks, -1  # not stored

    def pools():
        shape = (blocks, bs, hkv, d)
        made = [torch.full(shape, 3.0, device=DEV).to(cache_dtype) for _ in range(2)]
        scales = [None, None] if scale_dtype is None else [torch.full(shape[:3], 7, device=DEV, dtype=scale_dtype) for _ in range(2)]
        return made, dict(zip(("k_scale", "v_scale"), scales))

    bits = lambda x: x.view(torch.uint8)  # noqa: E731
    for window in (None, 40):
        (k1, v1), s1 = pools()
        ops.areno_paged_cache_write(k, v, k1, v1, ids, offs, **s1)
        want = ops.areno_varlen_causal_attention(q, k, v, cu, window_left=window)
        (k2, v2), s2 = pools()
        out = ops.areno_varlen_causal_attention_cache_write(q, k, v, cu, k2, v2, ids, offs, window_left=window, **s2)
        assert torch.equal(bits(out[front:]), bits(want[front:]))  # (no sequence's rows in front: not defined)
        for a, b in [(k1, k2), (v1, v2), (s1["k_scale"], s2["k_scale"]), (s1["v_scale"], s2["v_scale"])]:
            assert a is None or torch.equal(bits(a), bits(b))


def test_prefill_whose_keys_lie_in_the_pages_it_writes():
    """Keys that lie in the pages, every one in its own place: the store leaves them as they are."""
    t, bs = 64, 16
    g = torch.Generator().manual_seed(3)
    q, v = (torch.randn(t, h, 128, generator=g).to(torch.bfloat16).to(DEV) for h in (8, 2))
    pool = torch.randn(t // bs, bs, 2, 128, generator=g).to(torch.bfloat16)
    slots = torch.arange(t, device=DEV)  # every row is its own place, so that the store leaves the keys as they are
    cu = torch.tensor([0, t], dtype=torch.int32, device=DEV)
    ids, offs = slots // bs, slots % bs
    want_pool, pool = pool.to(DEV).clone(), pool.to(DEV)
    other = torch.zeros_like(pool)
    want = ops.areno_varlen_causal_attention(q, want_pool.view(t, 2, 128), v, cu)
    out = ops.areno_varlen_causal_attention_cache_write(q, pool.view(t, 2, 128), v, cu, pool, other, ids, offs)
    assert torch.equal(out, want) and torch.equal(pool, want_pool) and torch.equal(other.view(t, 2, 128), v)


@pytest.mark.parametrize("kv", ["same", "int8"])
@pytest.mark.parametrize("first_row", [0, 40, 63])
def test_prefill_whose_queries_lie_in_the_pages_it_writes(kv, first_row):
    """What the attention reads must not be pages that its launch writes: such a call stores first and attends then, with the stored
    rows as queries.  Queries that are the pages of K, or share their last row (8-bit pages: the last bytes) with them."""
    t, bs, h, d = 64, 16, 2, 128
    _, k, v, cu = (x.to(DEV) for x in _packed([40, 24], h, h, d, torch.bfloat16))
    slots = torch.arange(t, device=DEV)
    dtype, per_row = (torch.bfloat16, h * d) if kv == "same" else (torch.int8, 2 * h * d)  # (elements of a row of queries)
    memory = torch.randint(0, 60, (2 * t * per_row,), device=DEV, dtype=torch.int32).to(dtype)  # K's pool, and queries from first_row on
    pools = [memory[: t * h * d].view(t // bs, bs, h, d), torch.zeros(t // bs, bs, h, d, device=DEV, dtype=dtype)]
    q = memory[first_row * h * d :][: t * per_row].view(torch.bfloat16).view(t, h, d)
    scales = {} if kv == "same" else {n: torch.zeros(t // bs, bs, h, device=DEV) for n in ("k_scale", "v_scale")}
    out = ops.areno_varlen_causal_attention_cache_write(q, k, v, cu, *pools, slots // bs, slots % bs, **scales)
    want = ops.areno_varlen_causal_attention(q.clone(), k, v, cu)  # (the pages are stored: q is what it became)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))  # (codes read as 16-bit numbers may be NaN)
    assert kv != "same" or torch.equal(pools[0].view(t, h, d), k)


@pytest.mark.parametrize("first_row", [0, 40, 63])
def test_prefill_whose_output_lies_in_the_pages_it_writes(first_row):
    """The C entry with ``out`` inside a pool (or behind its last row but one): the pages are stored first, then the output."""
    t, bs, hq, hkv, d = 64, 16, 2, 2, 128
    q, k, v, cu = (x.to(DEV) for x in _packed([40, 24], hq, hkv, d, torch.bfloat16))
    slots = torch.arange(t, device=DEV)
    ids, offs = slots // bs, slots % bs
    memory = torch.zeros(first_row + t, hkv, d, device=DEV, dtype=torch.bfloat16)  # V's pool, and the output from first_row on
    k_pool, v_pool, out = torch.zeros(t // bs, bs, hkv, d, device=DEV, dtype=torch.bfloat16), memory[:t].view(t // bs, bs, hkv, d), memory[first_row:]
    workspace = torch.empty(cabi.prefill_workspace_bytes(hkv, d), dtype=torch.uint8, device=DEV)
    cache = cabi.describe_cache(k_pool, v_pool)
    cabi.check(cabi.lib().areno_hip_varlen_attention_cache_write(
        ctypes.byref(cache), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), cabi.dtype_code(q), t, hq, cu.data_ptr(), 2, -1, d**-0.5,
        ids.data_ptr(), offs.data_ptr(), workspace.data_ptr(), workspace.numel(), cabi.current_stream_ptr()), "prefill")  # fmt: skip
    assert torch.equal(out, ops.areno_varlen_causal_attention(q, k, v, cu))
    assert torch.equal(k_pool.view(t, hkv, d), k) and torch.equal(memory[:first_row], v[:first_row])


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 64), (28, 4, 128), (6, 6, 192), (16, 8, 256)])
@pytest.mark.parametrize("lens", [[5, 130, 33], [2] * 90])
def test_packed_output_of_eight_byte_alignment(hq, hkv, d, lens):
    """The C entry names no alignment for ``out``: from 8 bytes on it goes the way of an aligned one, to the bit."""
    q, k, v, cu = (x.to(DEV) for x in _packed(lens, hq, hkv, d, torch.bfloat16))
    workspace = torch.empty(cabi.prefill_workspace_bytes(hkv, d), dtype=torch.uint8, device=DEV)
    memory = torch.full((q.numel() + 8,), float("nan"), device=DEV, dtype=torch.bfloat16)
    out = memory[4 : 4 + q.numel()].view(q.shape)
    cabi.check(cabi.lib().areno_hip_varlen_attention(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), cabi.dtype_code(q), q.shape[0], hq, hkv, d,
        cu.data_ptr(), len(lens), -1, d**-0.5, workspace.data_ptr(), workspace.numel(), cabi.current_stream_ptr()), "varlen")  # fmt: skip
    assert torch.equal(out, ops.areno_varlen_causal_attention(q, k, v, cu))
    assert memory[:4].isnan().all() and memory[-4:].isnan().all()


def test_prefill_with_its_cache_write_takes_part_in_autograd():
    q, k, v, cu = _packed([40, 9], 8, 2, 128, torch.bfloat16)
    q, k, v = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    slots = torch.arange(49, device=DEV)
    pools = [torch.zeros(4, 16, 2, 128, device=DEV, dtype=torch.bfloat16) for _ in range(2)]
    out = ops.areno_varlen_causal_attention_cache_write(q, k, v, cu.to(DEV), *pools, slots // 16, slots % 16)
    grads = torch.autograd.grad(out, (q, k, v), torch.ones_like(out))
    want = torch.autograd.grad(ops.areno_varlen_causal_attention(q, k, v, cu.to(DEV)), (q, k, v), torch.ones_like(out))
    assert all(torch.equal(a, b) for a, b in zip(grads, want))


@pytest.mark.parametrize("hq,hkv", [(28, 4), (32, 8), (8, 1), (16, 16), (40, 2)])
@pytest.mark.parametrize("window_left", [None, 200])
@pytest.mark.parametrize("new,ctx", [
    ([1], [0]), ([1], [3001]), ([9], [5000]), ([64, 1, 33, 7], [2000, 33, 900, 0]), ([300], [40]), ([1] * 7, [0, 31, 32, 33, 1500, 64, 640]),
    ([40, 0, 3, 0], [700, 50, 2, 0]), ([2] * 15, list(range(0, 600, 40))), ([5] * 70, [64] * 70),
])  # fmt: skip
def test_paged_prefill_of_few_items(hq, hkv, window_left, new, ctx):
    """Where a launch has fewer items (query blocks) than units, every unit belongs to one item; where they are about as
    many, or more, the units are equal shares of all steps.  Items of one step and of a hundred, sequences without new
    tokens, more sequences than lanes, a packed end that no sequence holds."""
    w = workloads.make_prefill_workload("few", seed=hq + len(new), new_lens=torch.tensor(new), ctx_lens=torch.tensor(ctx), hq=hq, hkv=hkv,
                                        d=128, bs=16, kv="int8", device=DEV, quantize_fn=gpu_quantize)  # fmt: skip
    t = w.q.shape[0]
    q = torch.cat([w.q, w.q[:3]])
    out = ops.areno_paged_varlen_causal_attention(q, w.k_cache, w.v_cache, w.block_table, w.cu_seqlens_q, w.context_lens,
                                                  window_left=window_left, softmax_scale=w.softmax_scale, k_scale=w.k_scale,
                                                  v_scale=w.v_scale)  # fmt: skip
    assert_close(out[:t], _expected_prefill(w, window_left), *tolerances("int8"), what="prefill of few items")
    assert not out[t:].any()


@pytest.mark.parametrize("kv,d,page", [("bf16", 64, 16), ("fp8", 128, 64), ("int8", 192, 16), ("bf16", 256, 24), ("int8", 64, 256), ("bf16", 512, 16)])
@pytest.mark.parametrize("hq,hkv", [(14, 2), (16, 16)])
@pytest.mark.parametrize("new,ctx", [([9], [3000]), ([3] * 8, [3000, 2500, 2000, 1500, 1000, 600, 300, 100]), ([40, 0, 3, 0], [700, 50, 2, 0])])
def test_paged_prefill_of_few_items_in_every_type(kv, d, page, hq, hkv, new, ctx):
    """The same over the caches' types, head dims and page sizes; the second pack, at 16 heads, is one that looks for units of one
    item in vain and takes equal shares."""
    w = workloads.make_prefill_workload("few", seed=d + page, new_lens=torch.tensor(new), ctx_lens=torch.tensor(ctx), hq=hq, hkv=hkv, d=d, bs=page,
                                        kv=kv, device=DEV, quantize_fn=gpu_quantize)  # fmt: skip
    assert_close(_run_prefill(w), _expected_prefill(w, None), *tolerances(kv), what="prefill of few items")
