"""What a user of the attention path has it do, as cases that can be timed and compared.

Six kinds of pass, each through the public entry points in the order an engine or a trainer calls them:

* ``decode``   one layer's decode attention of a batch, called eagerly through the inference backend;
* ``step``     a decode step replayed from a captured graph: pages and block table, rotary rows, the step's plan,
               then for every layer norm + rotary and the decode op with its append;
* ``rollout``  a planned decode step of sampled groups whose rows share their prompt's pages, called eagerly;
* ``chunk``    one layer of a chunked prefill over a paged cache: norm + rotary + cache write, then attention of the
               new tokens over the cached context and themselves;
* ``prompts``  one layer of a prefill of fresh prompts through the inference backend: cache write, then attention;
* ``train``    forward and backward of the packed attention op: the output and the gradients of q, k and v.

Lengths belong to the case (``lengths`` is the seed they are drawn from, log-uniform for rollouts' continuations and
uniform elsewhere), values and page assignments to the seed given to ``prepare``.  Caches are filled by the
framework's own cache write, so quantized pages hold what a serving program's hold.
"""

from __future__ import annotations

import math
import random

import torch

from areno_amd.accel import attention as ops
from areno_amd.engine import DeviceBlockTables, HipInferBackend, InferMeta

DEVICE = "cuda"
ACTS = {"bf16": torch.bfloat16, "fp16": torch.float16}
CACHES = {"int8": (torch.int8, torch.float16), "fp8": (torch.float8_e4m3fn, torch.float32)}
ROPE_THETA = 1e6
EPS = 1e-6


def listed():
    return [
        # the latency of a lone request: a chat with one sequence of 4 k tokens, 16-bit pages
        _case("decode", name="decode-1x4096-bf16", batch=1, ctx_lo=4096, ctx_hi=4096),
        # a serving batch in the engine's eager mode, 16-bit pages, lengths all over the range
        _case("decode", name="decode-64x4096-bf16", batch=64, ctx_lo=512, ctx_hi=4096),
        # the same batch with an int8 cache as a captured decode step: a quarter of a 28-layer model
        _case("step", name="step-64x4096-int8", batch=64, ctx_lo=512, ctx_hi=4096, kv="int8", layers=7),
        # a sampling phase: 32 prompts with 8 samples each, fp8 pages, two layers
        _case("rollout", name="rollout-32x8-fp8", seqs=32, batch=256, heads="32/8", ctx_lo=256, ctx_hi=2048, kv="fp8",
              layers=2),
        # chunked prefill of long contexts with an fp8 cache
        _case("chunk", name="chunk-16x512-on-16k-fp8", seqs=16, new_lo=1, new_hi=512, ctx_lo=0, ctx_hi=16384,
              heads="32/8", kv="fp8"),
        # a few short follow-ups to running conversations
        _case("chunk", name="chunk-4x64-on-4k-int8", seqs=4, new_lo=1, new_hi=64, ctx_lo=256, ctx_hi=4096, kv="int8"),
        # admission of a batch of short prompts, 16-bit pages
        _case("prompts", name="prompts-32x512-bf16", seqs=32, new_lo=33, new_hi=512),
        # two long prompts on a sliding-window layer with wide heads, pages of 256 tokens
        _case("prompts", name="prompts-2x6000-d256-w1024-bf16", seqs=2, new_lo=3000, new_hi=6000, heads="16/8", d=256,
              window=1024, page=256),
        # a fine-tuning micro-batch of short ragged samples on a small model (16 heads of 64), fp16
        _case("train", name="train-16x600-d64-fp16", seqs=16, new_lo=20, new_hi=600, heads="16/16", d=64, act="fp16"),
        # the training shape of the benchmark: two sequences of 2 k tokens
        _case("train", name="train-2x2048-bf16", seqs=2, new_lo=2048, new_hi=2048),
        # a full micro-batch of long samples
        _case("train", name="train-4x4096-bf16", seqs=4, new_lo=4096, new_hi=4096, heads="32/8"),
        # a sliding-window layer with wide heads in training, ragged samples
        _case("train", name="train-4x1000-d256-w512-bf16", seqs=4, new_lo=300, new_hi=1000, heads="16/8", d=256,
              window=512),
    ]  # fmt: skip


def _case(kind, *, name=None, seqs=0, batch=0, heads="28/4", d=128, page=16, kv="", act="bf16", new_lo=0, new_hi=0,
          ctx_lo=0, ctx_hi=0, window=-1, layers=1, lengths=1):  # fmt: skip
    """``kv``: the cache's type (empty: the activations').  ``window``: tokens to the left a query sees, -1 for all."""
    c = dict(kind=kind, seqs=seqs, batch=batch, heads=heads, d=d, page=page, kv=kv or act, act=act, new_lo=new_lo,
             new_hi=new_hi, ctx_lo=ctx_lo, ctx_hi=ctx_hi, window=window, layers=layers, lengths=lengths)  # fmt: skip
    return c if name is None else dict(name=name, **c)


def draw(rng):
    """One more case of the listed kinds.  Limits on tokens and on query-key pairs keep it at or below the largest
    listed case."""

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "decode", "step", "rollout", "chunk", "chunk", "prompts", "prompts", "train", "train", "train"])
    lengths = rng.randrange(1, 1 << 20)
    heads = rng.choice(["28/4", "32/8", "16/16", "8/2", "24/8"])
    d = rng.choice([64, 128, 128, 128])
    act = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    kv = rng.choice(["", "int8", "fp8"])
    page = rng.choice([16, 16, 32, 64, 256])
    hq, hkv = map(int, heads.split("/"))
    if kind in ("decode", "step"):
        batch = log_int(1, 128)
        hi = log_int(64, min(16384, 64 * 4096 * 4 * 128 // (batch * hkv * d)))
        layers = rng.randint(2, 7) if kind == "step" else 1
        return _case(kind, batch=batch, heads=heads, d=d, page=page, kv=kv, act=act, ctx_lo=max(1, hi // 8), ctx_hi=hi,
                     layers=layers, window=rng.choice([-1, -1, -1, 1024]) if kind == "decode" else -1, lengths=lengths)  # fmt: skip
    if kind == "rollout":
        seqs, samples = log_int(2, 32), rng.choice([4, 8])
        hi = log_int(128, 2048)
        return _case(kind, seqs=seqs, batch=seqs * samples, heads=rng.choice(["32/8", "28/4", "16/16"]), page=16,
                     kv=kv or "fp8", act=act, ctx_lo=hi // 8, ctx_hi=hi, layers=rng.randint(1, 2), lengths=lengths)  # fmt: skip
    if kind == "chunk":
        seqs = log_int(1, 16)
        new, ctx = log_int(8, 512), log_int(64, 16384)
        return _case(kind, seqs=seqs, heads=heads, d=d, page=page, kv=kv or act, act=act, new_lo=1, new_hi=new, ctx_lo=0,
                     ctx_hi=ctx, lengths=lengths)  # fmt: skip
    wide = rng.random() < 0.25
    if wide:
        heads, d = rng.choice(["16/8", "8/1", "6/6"]), rng.choice([256, 256, 192])
        hq, hkv = map(int, heads.split("/"))
    window = rng.choice([-1, 512, 1024]) if wide else rng.choice([-1, -1, -1, 1024])
    seqs = log_int(1, 32)
    if kind == "prompts":
        hi = log_int(16, min(8192, 24576 // seqs))
        return _case(kind, seqs=seqs, heads=heads, d=d, page=page, kv="" if wide else kv, act=act, new_lo=max(1, hi // 8),
                     new_hi=hi, window=window, lengths=lengths)  # fmt: skip
    # the widest window of the wide training case, and the tokens of the long one, bound what a drawn one costs
    hi = log_int(32, min(1000, 4000 // seqs) if wide else min(4096, 16384 // seqs))
    window = 512 if wide else window
    return _case(kind, seqs=seqs, heads=heads, d=d, act=act, new_lo=max(1, hi // 8), new_hi=hi, window=window, lengths=lengths)


# ---- lengths ---------------------------------------------------------------------------------------------------------
def _uniform(case, salt, n, lo, hi):
    rng = random.Random(case["lengths"] * 8 + salt)
    return [rng.randint(lo, hi) for _ in range(n)]


def _decode_lengths(case):
    """Cached tokens of every row; for rollouts the prompt's length and the row's continuation (median 1 k, at most
    8 k)."""
    if case["kind"] != "rollout":
        return _uniform(case, 0, case["batch"], case["ctx_lo"], case["ctx_hi"])
    prompts = _uniform(case, 0, case["seqs"], case["ctx_lo"], case["ctx_hi"])
    rng = random.Random(case["lengths"] * 8 + 1)
    samples = case["batch"] // case["seqs"]
    median = min(1000, case["ctx_hi"])
    return [p + max(1, min(8192, int(median * math.exp(rng.gauss(0.0, 1.0))))) for p in prompts for _ in range(samples)]


def _shared_blocks(case):
    """Full pages of every prompt of a rollout."""
    return [p // case["page"] for p in _uniform(case, 0, case["seqs"], case["ctx_lo"], case["ctx_hi"])]


def _prefill_lengths(case):
    new = _uniform(case, 0, case["seqs"], case["new_lo"], case["new_hi"])
    ctx = _uniform(case, 1, case["seqs"], case["ctx_lo"], case["ctx_hi"])
    return new, ctx


# ---- inputs ----------------------------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed * 1009 + 17)


def _normal(gen, *shape, dtype):
    return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32).to(dtype)


def _heads(case):
    hq, hkv = map(int, case["heads"].split("/"))
    return hq, hkv, case["d"]


def _caches(case, gen, blocks, layers):
    """Pools ``(layers, blocks, page, kv heads, d)`` full of earlier tokens, quantized by the cache write where the
    cache is (1 % of such values at eight times the spread, as activations have them)."""
    hq, hkv, d = _heads(case)
    act, page = ACTS[case["act"]], case["page"]
    shape = (layers, blocks, page, hkv, d)
    if case["kv"] not in CACHES:
        pools = [torch.empty(shape, device=DEVICE, dtype=act) for _ in range(2)]
        for pool in pools:
            for layer in pool:
                layer.copy_(_normal(gen, *shape[1:], dtype=act))
        return pools[0], pools[1], None, None
    cache_dtype, scale_dtype = CACHES[case["kv"]]
    k, v = (torch.zeros(shape, device=DEVICE, dtype=torch.uint8).view(cache_dtype) for _ in range(2))
    ks, vs = (torch.ones(shape[:4], device=DEVICE, dtype=scale_dtype) for _ in range(2))
    slots = torch.arange(blocks * page, device=DEVICE)
    for layer in range(layers):
        rows = [_normal(gen, blocks * page, hkv, d, dtype=torch.float32) for _ in range(2)]
        for x in rows:
            x.mul_(torch.where(torch.rand(x.shape, generator=gen, device=DEVICE) < 0.01, 8.0, 1.0))
        ops.areno_paged_cache_write(rows[0].to(act), rows[1].to(act), k[layer], v[layer], slots // page, slots % page,
                                    k_scale=ks[layer], v_scale=vs[layer])  # fmt: skip
    return k, v, ks, vs


def _tables(seed, rows, spare=0.1):
    """Block table of rows that own pages by logical number, over a shuffled pool: ``(table, pages in the pool)``."""
    used = 1 + max(max(r) for r in rows)
    pool = used + max(1, int(used * spare))
    perm = torch.randperm(pool, generator=torch.Generator().manual_seed(seed)).to(torch.int32)
    table = torch.empty((len(rows), max(map(len, rows))), dtype=torch.int32)
    for i, row in enumerate(rows):
        ids = perm[torch.tensor(row)]
        table[i, : len(row)] = ids
        table[i, len(row) :] = ids[-1]  # the engine pads with the row's last page
    return table, pool


def _own_pages(tokens, page):
    rows, at = [], 0
    for n in tokens:
        need = max(1, -(-n // page))
        rows.append(list(range(at, at + need)))
        at += need
    return rows


def _rope_tables(d, positions):
    freq = 1.0 / (ROPE_THETA ** (torch.arange(0, d, 2, dtype=torch.float32, device=DEVICE) / d))
    angle = torch.outer(torch.arange(positions, dtype=torch.float32, device=DEVICE), freq)
    angle = torch.cat((angle, angle), dim=-1)
    return angle.cos(), angle.sin()


def _norm_weights(gen, d):
    return tuple(1.0 + 0.1 * torch.randn(d, generator=gen, device=DEVICE) for _ in range(2))


def _cu(lens):
    out = [0]
    for n in lens:
        out.append(out[-1] + n)
    return out


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEVICE)


# ---- prepare ---------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    gen = _generator(seed)
    state = {"case": case, **_PREPARE[case["kind"]](case, seed, gen)}
    return state


def _prepare_decode(case, seed, gen):
    hq, hkv, d = _heads(case)
    act = ACTS[case["act"]]
    lens = _decode_lengths(case)
    table, pool = _tables(seed, _own_pages([n + 1 for n in lens], case["page"]))
    k, v, ks, vs = _caches(case, gen, pool, 1)
    b = case["batch"]
    return {
        "backend": HipInferBackend(),
        "q": _normal(gen, 1, b, hq, d, dtype=act), "k": _normal(gen, 1, b, hkv, d, dtype=act),
        "v": _normal(gen, 1, b, hkv, d, dtype=act), "k_cache": k[0], "v_cache": v[0],
        "k_scale": None if ks is None else ks[0], "v_scale": None if vs is None else vs[0],
        "meta": InferMeta(mode="decode", cache_seqlens=_i32(lens), block_table=table.to(DEVICE)),
        "window": None if case["window"] < 0 else (case["window"], 0),
    }  # fmt: skip


def _prepare_step(case, seed, gen):
    """The captured step of ``case["layers"]`` layers and its static inputs."""
    hq, hkv, d = _heads(case)
    act, page, b, layers = ACTS[case["act"]], case["page"], case["batch"], case["layers"]
    lens = _decode_lengths(case)
    columns = max(lens) // page + 1
    blocks = sum(n // page + 1 for n in lens) + b
    pages = DeviceBlockTables(blocks, b, columns, page, DEVICE)
    # the rows were admitted with part of their tokens and grew side by side since, so their pages interleave
    order = random.Random(seed)
    for part in range(4, 17):
        rows = order.sample(range(b), b)
        pages.reserve(rows, [max(1, n * part // 16) for n in (lens[r] for r in rows)])
    k, v, ks, vs = _caches(case, gen, blocks + 1, layers)  # one page more: the scratch page of padded tables
    cos, sin = _rope_tables(d, max(lens) + 1)
    qw, kw = _norm_weights(gen, d)
    s = {
        "pages": pages, "rows": torch.arange(b, device=DEVICE), "lens": _i32(lens),
        "positions": torch.tensor(lens, device=DEVICE), "cos": cos, "sin": sin, "qw": qw, "kw": kw,
        "table": torch.zeros((b, columns), dtype=torch.int32, device=DEVICE),
        "q": _normal(gen, layers, b, hq, d, dtype=act), "k": _normal(gen, layers, b, hkv, d, dtype=act),
        "v": _normal(gen, layers, b, hkv, d, dtype=act), "k_cache": k, "v_cache": v, "k_scale": ks, "v_scale": vs,
        "plan": torch.empty(1 << 20, dtype=torch.uint8, device=DEVICE), "layers": layers,
    }  # fmt: skip
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _decode_step(s)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _decode_step(s)
    return {**s, "graph": graph, "out": out}


def _decode_step(s):
    scales = s["k_scale"] is not None
    table = s["pages"].decode_step(s["rows"], s["lens"], pad="scratch", out=s["table"])
    rope = ops.areno_rope_rows(s["positions"], s["cos"], s["sin"], s["q"].dtype)
    plan = ops.areno_paged_decode_plan(table, s["lens"], s["k_cache"][0], s["v_cache"][0], q_heads=s["q"].shape[2],
                                       q_dtype=s["q"].dtype, k_scale=s["k_scale"][0] if scales else None,
                                       v_scale=s["v_scale"][0] if scales else None, buffer=s["plan"])  # fmt: skip
    outs = []
    for i in range(s["layers"]):
        q, k = ops.areno_qk_norm_rope_cache_write(s["q"][i], s["k"][i], s["v"][i], s["positions"], s["cos"], s["sin"],
                                                  q_norm_weight=s["qw"], k_norm_weight=s["kw"], eps=EPS,
                                                  rope_rows=rope)  # fmt: skip
        outs.append(ops.areno_paged_causal_attention_decode(
            q, k, s["v"][i], s["k_cache"][i], s["v_cache"][i], table, s["lens"],
            k_scale=s["k_scale"][i] if scales else None, v_scale=s["v_scale"][i] if scales else None, plan=plan))  # fmt: skip
    return outs


def _prepare_rollout(case, seed, gen):
    hq, hkv, d = _heads(case)
    act, page, layers = ACTS[case["act"]], case["page"], case["layers"]
    lens, shared = _decode_lengths(case), _shared_blocks(case)
    samples = case["batch"] // case["seqs"]
    rows, at = [], 0
    for p, count in enumerate(shared):
        common = list(range(at, at + count))
        at += count
        for n in lens[p * samples : (p + 1) * samples]:
            own = n // page + 1 - count
            rows.append(common + list(range(at, at + own)))
            at += own
    table, pool = _tables(seed, rows)
    k, v, ks, vs = _caches(case, gen, pool, layers)
    b = case["batch"]
    return {
        "q": _normal(gen, layers, b, hq, d, dtype=act), "k": _normal(gen, layers, b, hkv, d, dtype=act),
        "v": _normal(gen, layers, b, hkv, d, dtype=act), "k_cache": k, "v_cache": v, "k_scale": ks, "v_scale": vs,
        "lens": _i32(lens), "table": table.to(DEVICE), "shared": _i32([n * page for n in shared]), "samples": samples,
    }  # fmt: skip


def _prepare_chunk(case, seed, gen):
    hq, hkv, d = _heads(case)
    act, page = ACTS[case["act"]], case["page"]
    new, ctx = _prefill_lengths(case)
    table, pool = _tables(seed, _own_pages([a + b for a, b in zip(new, ctx)], page))
    k, v, ks, vs = _caches(case, gen, pool, 1)
    positions, ids = _slots(table, new, ctx, page)
    t = sum(new)
    cos, sin = _rope_tables(d, max(a + b for a, b in zip(new, ctx)))
    qw, kw = _norm_weights(gen, d)
    return {
        "q": _normal(gen, t, hq, d, dtype=act), "k": _normal(gen, t, hkv, d, dtype=act),
        "v": _normal(gen, t, hkv, d, dtype=act), "k_cache": k[0], "v_cache": v[0],
        "k_scale": None if ks is None else ks[0], "v_scale": None if vs is None else vs[0], "positions": positions,
        "ids": ids, "offsets": positions % page, "table": table.to(DEVICE), "cu": _i32(_cu(new)), "ctx": _i32(ctx),
        "cos": cos, "sin": sin, "qw": qw, "kw": kw,
    }  # fmt: skip


def _slots(table, new, ctx, page):
    """Position and page of every new token."""
    positions, ids = [], []
    for i, (n, c) in enumerate(zip(new, ctx)):
        p = torch.arange(c, c + n)
        positions.append(p)
        ids.append(table[i].long()[p // page])
    return torch.cat(positions).to(DEVICE), torch.cat(ids).to(DEVICE)


def _prepare_prompts(case, seed, gen):
    hq, hkv, d = _heads(case)
    act, page = ACTS[case["act"]], case["page"]
    new, _ = _prefill_lengths(case)
    table, pool = _tables(seed, _own_pages(new, page))
    k, v, ks, vs = _caches(case, gen, pool, 1)
    positions, ids = _slots(table, new, [0] * len(new), page)
    t = sum(new)
    return {
        "backend": HipInferBackend(),
        "q": _normal(gen, 1, t, hq, d, dtype=act), "k": _normal(gen, 1, t, hkv, d, dtype=act),
        "v": _normal(gen, 1, t, hkv, d, dtype=act), "k_cache": k[0], "v_cache": v[0],
        "k_scale": None if ks is None else ks[0], "v_scale": None if vs is None else vs[0],
        "meta": InferMeta(mode="prefill", cu_seqlens=_i32(_cu(new)), max_seqlen=max(new), block_table=table.to(DEVICE),
                          cache_block_ids=ids, cache_block_offsets=positions % page),
        "window": None if case["window"] < 0 else (case["window"], 0),
    }  # fmt: skip


def _prepare_train(case, seed, gen):
    hq, hkv, d = _heads(case)
    act = ACTS[case["act"]]
    new, _ = _prefill_lengths(case)
    t = sum(new)
    q, k, v = (_normal(gen, t, h, d, dtype=act).requires_grad_(True) for h in (hq, hkv, hkv))
    return {"q": q, "k": k, "v": v, "cu": _i32(_cu(new)), "grad": _normal(gen, t, hq, d, dtype=act),
            "window": None if case["window"] < 0 else case["window"]}  # fmt: skip


_PREPARE = {"decode": _prepare_decode, "step": _prepare_step, "rollout": _prepare_rollout, "chunk": _prepare_chunk,
            "prompts": _prepare_prompts, "train": _prepare_train}  # fmt: skip


# ---- run -------------------------------------------------------------------------------------------------------------
def run(state):
    return _RUN[state["case"]["kind"]](state)


def _pools(s):
    return [t for t in (s["k_cache"], s["v_cache"], s["k_scale"], s["v_scale"]) if t is not None]


def _run_backend(s):
    out = s["backend"](s["q"], s["k"], s["v"], s["k_cache"], s["v_cache"], s["meta"], window_size=s["window"],
                       k_scale=s["k_scale"], v_scale=s["v_scale"])  # fmt: skip
    return [out, *_pools(s)]


def _run_step(s):
    s["graph"].replay()
    return [*s["out"], s["table"], *_pools(s)]


def _run_rollout(s):
    scales = s["k_scale"] is not None
    plan = ops.areno_paged_decode_plan(s["table"], s["lens"], s["k_cache"][0], s["v_cache"][0], q_heads=s["q"].shape[2],
                                       q_dtype=s["q"].dtype, k_scale=s["k_scale"][0] if scales else None,
                                       v_scale=s["v_scale"][0] if scales else None, prefix_group_rows=s["samples"],
                                       shared_prefix_lens=s["shared"])  # fmt: skip
    outs = []
    for i in range(s["q"].shape[0]):
        outs.append(ops.areno_paged_causal_attention_decode(
            s["q"][i], s["k"][i], s["v"][i], s["k_cache"][i], s["v_cache"][i], s["table"], s["lens"],
            k_scale=s["k_scale"][i] if scales else None, v_scale=s["v_scale"][i] if scales else None,
            prefix_group_rows=s["samples"], shared_prefix_lens=s["shared"], plan=plan))  # fmt: skip
    return [*outs, *_pools(s)]


def _run_chunk(s):
    q, k = ops.areno_qk_norm_rope_cache_write(
        s["q"], s["k"], s["v"], s["positions"], s["cos"], s["sin"], q_norm_weight=s["qw"], k_norm_weight=s["kw"],
        eps=EPS, k_cache=s["k_cache"], v_cache=s["v_cache"], cache_block_ids=s["ids"], cache_block_offsets=s["offsets"],
        k_scale=s["k_scale"], v_scale=s["v_scale"])  # fmt: skip
    out = ops.areno_paged_varlen_causal_attention(q, s["k_cache"], s["v_cache"], s["table"], s["cu"], s["ctx"],
                                                  k_scale=s["k_scale"], v_scale=s["v_scale"])  # fmt: skip
    return [out, q, k, *_pools(s)]


def _run_train(s):
    out = ops.areno_varlen_causal_attention(s["q"], s["k"], s["v"], s["cu"], window_left=s["window"])
    return [out, *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["grad"])]


_RUN = {"decode": _run_backend, "step": _run_step, "rollout": _run_rollout, "chunk": _run_chunk,
        "prompts": _run_backend, "train": _run_train}  # fmt: skip


# ---- work and tolerance ----------------------------------------------------------------------------------------------
def _seen(case, position):
    return position + 1 if case["window"] < 0 else min(position + 1, case["window"] + 1)


def work(case):
    hq, hkv, d = _heads(case)
    e = 2  # activations
    row = hkv * (2 * d * e if case["kv"] not in CACHES else 2 * (d + CACHES[case["kv"]][1].itemsize))  # one cached token
    if case["kind"] in ("decode", "step", "rollout"):
        lens = _decode_lengths(case)
        seen = read = sum(_seen(case, n) for n in lens)
        if case["kind"] == "rollout":  # a prompt's shared pages are read once for its samples
            read -= (case["batch"] // case["seqs"] - 1) * case["page"] * sum(_shared_blocks(case))
        rows = case["batch"]
        columns = sum(-(-(n + 1) // case["page"]) for n in lens)
        layer = read * row + rows * (2 * hq + 2 * hkv) * d * e
        if case["kind"] == "step":  # the norm and rotary step in front: q and k in and out, the token's rotary row
            layer += rows * ((2 * hq + 2 * hkv) * d * e + 2 * d * 4)
        return {"bytes": case["layers"] * layer + 4 * columns + 4 * rows, "flops": case["layers"] * 4 * hq * d * seen}
    new, ctx = _prefill_lengths(case)
    t = sum(new)
    pairs = 0
    for n, c in zip(new, ctx):
        w = case["window"]
        # positions c .. c + n - 1 see position + 1 keys, at most window + 1
        if w < 0 or c + n <= w + 1:
            pairs += n * c + n * (n + 1) // 2
        else:
            ramp = max(0, w + 1 - c)
            pairs += ramp * c + ramp * (ramp + 1) // 2 + (n - ramp) * (w + 1)
    if case["kind"] == "train":
        # two products forward, five backward; q, k, v, the output's gradient in, the output and three gradients out
        return {"bytes": t * (4 * hq + 4 * hkv) * d * e, "flops": 14 * hq * d * pairs}
    if case["kind"] == "prompts":
        return {"bytes": t * ((2 * hq + 2 * hkv) * d * e + row + 16), "flops": 4 * hq * d * pairs}
    read = sum(c + n for n, c in zip(new, ctx))
    return {"bytes": read * row + t * ((3 * hq + 3 * hkv) * d * e + row + 24 + 8 * d), "flops": 4 * hq * d * pairs}


def tolerance(case):
    """Four times what the passes showed against the same attention in 64 bits over the same (dequantized) inputs: the
    outputs' own rounding makes most of it (bf16 2.6e-3, fp16 3.2e-4 relative; gradients 7e-2 and 7e-3 at the worst
    value of a tensor, outputs 2e-2 and 2e-3), and the fp16 rounding of dequantized keys and values 9e-4 where the
    activations are fp16.  Pages hold what the cache write's closed form says and do not differ at all."""
    if case["act"] == "fp16":
        return {"rel": 1.3e-3 if case["kv"] not in CACHES else 3.6e-3, "max": 0.03}
    return {"rel": 1e-2, "max": 0.28 if case["kind"] == "train" else 0.08}
