"""The backend module driven the way the engine drives it: prompt prefill (store + attention), a second prefill
chunk that must see the first, then decode steps, on plain and quantized caches; every output against the CPU oracle
on the (dequantized) cache contents."""

import pytest
import torch

from areno_amd.accel import attention as ops
from areno_amd.engine import InferMeta, allocate_kv_caches, build_infer_attention_backend
from oracle import attention_ref as ar
from tests.gpu_util import DEV, assert_close, dequant_cpu, tolerances

pytestmark = pytest.mark.gpu

BS = 16


def _block_plan(total_lens, num_blocks, gen):
    """Shuffled pages for each sequence, enough for ``total_lens`` tokens; returns the int32 block table."""
    perm = torch.randperm(num_blocks - 1, generator=gen).tolist()  # the last block stays free as the scratch block
    need = [(n + BS - 1) // BS for n in total_lens]
    table = torch.full((len(total_lens), max(need)), num_blocks - 1, dtype=torch.int32)
    for s, n in enumerate(need):
        table[s, :n] = torch.tensor([perm.pop() for _ in range(n)], dtype=torch.int32)
    return table


def _write_plan(table, starts, counts):
    ids, offs = [], []
    for s, (a, n) in enumerate(zip(starts, counts)):
        pos = torch.arange(a, a + n)
        ids.append(table[s].long()[pos // BS])
        offs.append(pos % BS)
    return torch.cat(ids), torch.cat(offs)


@pytest.mark.parametrize("kv,hq,hkv,d,dv", [("auto", 8, 2, 64, 64), ("int8", 28, 4, 128, 128), ("fp8", 8, 8, 128, 96)])
def test_prefill_chunk_decode_loop(kv, hq, hkv, d, dv):
    gen = torch.Generator().manual_seed(41)
    dtype = torch.bfloat16
    prompt, chunk2, steps = [37, 5, 64], [3, 10, 1], 3
    total = [a + b + steps for a, b in zip(prompt, chunk2)]
    num_blocks = sum((n + BS - 1) // BS for n in total) + 4
    layer = allocate_kv_caches(1, num_blocks, BS, hkv, d, DEV, dtype, kv)[0]
    table = _block_plan(total, num_blocks, gen)
    backend = build_infer_attention_backend()
    name = {"auto": "bf16"}.get(kv, kv)
    scale = d**-0.5

    def rand(t, h, w):
        return torch.randn(1, t, h, w, generator=gen).to(dtype)

    def call(q, k, v, meta):
        return backend(q.to(DEV), k.to(DEV), v.to(DEV), layer.k_cache, layer.v_cache, meta, softmax_scale=scale,
                       k_scale=layer.k_scale, v_scale=layer.v_scale)  # fmt: skip

    def cache_cpu():
        return dequant_cpu(layer.k_cache, layer.k_scale), dequant_cpu(layer.v_cache, layer.v_scale)

    # ---- prompt prefill: attention over the fresh (unquantized) K/V, pages written on the side ------------------
    t1 = sum(prompt)
    q, k, v = rand(t1, hq, d), rand(t1, hkv, d), rand(t1, hkv, dv)
    cu = torch.tensor([0] + list(torch.tensor(prompt).cumsum(0)), dtype=torch.int32)
    ids, offs = _write_plan(table, [0, 0, 0], prompt)
    meta = InferMeta(mode="prefill", cu_seqlens=cu.to(DEV), max_seqlen=max(prompt), block_table=table.to(DEV),
                     cache_block_ids=ids.to(DEV), cache_block_offsets=offs.to(DEV))  # fmt: skip
    out = call(q, k, v, meta)
    assert out.shape == (1, t1, hq, dv)
    v_pad = torch.nn.functional.pad(v[0].float(), (0, d - dv))
    want = ar.ref_varlen(q[0].float(), k[0].float(), v_pad, cu, -1, scale)[..., :dv]
    assert_close(out[0], want, *tolerances("bf16"), what="prompt prefill")

    # ---- second chunk: must see the cached prompt through the pages -------------------------------------------------
    t2 = sum(chunk2)
    q, k, v = rand(t2, hq, d), rand(t2, hkv, d), rand(t2, hkv, dv)
    cu2 = torch.tensor([0] + list(torch.tensor(chunk2).cumsum(0)), dtype=torch.int32)
    ids, offs = _write_plan(table, prompt, chunk2)
    ctx = torch.tensor(prompt, dtype=torch.int32)
    meta = InferMeta(mode="prefill", cu_seqlens=cu2.to(DEV), max_seqlen=max(chunk2), block_table=table.to(DEV),
                     cache_block_ids=ids.to(DEV), cache_block_offsets=offs.to(DEV), context_lens=ctx.to(DEV))  # fmt: skip
    out = call(q, k, v, meta)
    kc, vc = cache_cpu()
    want = ar.ref_paged_varlen_prefill(q[0].float(), kc, vc, table, cu2, ctx, -1, scale)[..., :dv]
    assert_close(out[0], want, *tolerances(name), what="chunk over cached context")

    # ---- decode steps ---------------------------------------------------------------------------------------------------
    lens = torch.tensor([a + b for a, b in zip(prompt, chunk2)], dtype=torch.int32)
    for step in range(steps):
        q, k, v = rand(3, hq, d), rand(3, hkv, d), rand(3, hkv, dv)
        meta = InferMeta(mode="decode", cache_seqlens=(lens + step).to(DEV), block_table=table.to(DEV))
        out = call(q, k, v, meta)
        assert out.shape == (1, 3, hq, dv)
        kc, vc = cache_cpu()
        want = ar.ref_paged_decode(q[0].float(), kc, vc, table, lens + step, -1, scale)[..., :dv]
        assert_close(out[0], want, *tolerances(name), what=f"decode step {step}")


def test_loop_driven_by_device_block_tables():
    """Same loop with the page bookkeeping on the device: tables, write slots and positions come from
    DeviceBlockTables (no host-built table is uploaded), decode crosses page borders, one sequence finishes and a
    new one is admitted into the freed pages; outputs against the oracle reading through the device's own table."""
    from areno_amd.engine import DeviceBlockTables
    from oracle.block_table_ref import RefBlockTables

    gen = torch.Generator().manual_seed(43)
    dtype, hq, hkv, d = torch.bfloat16, 8, 2, 64
    scale = d**-0.5
    num_blocks, max_rows, max_blocks = 12, 4, 6
    layer = allocate_kv_caches(1, num_blocks + 1, BS, hkv, d, DEV, dtype, "int8")[0]
    pages = DeviceBlockTables(num_blocks, max_rows, max_blocks, BS, DEV)
    lists = RefBlockTables(num_blocks, max_rows, max_blocks, BS)  # the reference's host lists, kept in step
    backend = build_infer_attention_backend()

    def same_pages():
        for row in range(max_rows):
            assert pages.row_pages(row) == lists.row_pages(row), f"row {row}"
        assert pages.free_list() == lists.free_list() and pages.status() == (0, -1)

    def rand(t, h):
        return torch.randn(1, t, h, d, generator=gen).to(dtype)

    def call(q, k, v, meta):
        return backend(q.to(DEV), k.to(DEV), v.to(DEV), layer.k_cache, layer.v_cache, meta, softmax_scale=scale,
                       k_scale=layer.k_scale, v_scale=layer.v_scale)  # fmt: skip

    def prefill(rows, lens):
        pages.reserve(rows, lens)
        lists.reserve(rows, lens)
        cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
        t = int(cu[-1])
        ids, offs, pos = pages.prefill_slots(rows, [0] * len(rows), cu, t)
        assert pos.cpu().tolist() == [p for n in lens for p in range(n)]
        table = pages.block_table(rows)
        q, k, v = rand(t, hq), rand(t, hkv), rand(t, hkv)
        meta = InferMeta(mode="prefill", cu_seqlens=cu.to(DEV), max_seqlen=max(lens), block_table=table,
                         cache_block_ids=ids, cache_block_offsets=offs)  # fmt: skip
        out = call(q, k, v, meta)
        want = ar.ref_varlen(q[0].float(), k[0].float(), v[0].float(), cu, -1, scale)
        assert_close(out[0], want, *tolerances("bf16"), what="prefill")

    def decode(rows, lens_dev, steps):
        rows_dev = torch.tensor(rows, device=DEV)
        for step in range(steps):
            pages.ensure_decode(rows_dev, lens_dev)
            lists.ensure_decode(rows, lens_dev.cpu().tolist())
            table = pages.block_table(rows_dev)
            assert table.cpu().tolist() == lists.gather(rows, False)
            q, k, v = rand(len(rows), hq), rand(len(rows), hkv), rand(len(rows), hkv)
            meta = InferMeta(mode="decode", cache_seqlens=lens_dev, block_table=table)
            out = call(q, k, v, meta)
            kc, vc = dequant_cpu(layer.k_cache, layer.k_scale), dequant_cpu(layer.v_cache, layer.v_scale)
            want = ar.ref_paged_decode(q[0].float(), kc, vc, table.cpu(), lens_dev.cpu(), -1, scale)
            assert_close(out[0], want, *tolerances("int8"), what=f"decode step {step}")
            lens_dev += 1
        pages.check()

    prefill([2, 0, 3], [30, 16, 5])
    lens_dev = torch.tensor([30, 16, 5], dtype=torch.int32, device=DEV)
    decode([2, 0, 3], lens_dev, 4)  # row 0 opens its second page at position 16, row 2 its third at 32
    assert pages.row_pages(2) == [0, 1, 5] and pages.row_pages(0) == [2, 4] and pages.row_pages(3) == [3]
    same_pages()
    pages.release([0])
    lists.release([0])
    prefill([1], [40])  # takes pages 6 .. 8 from the head of the free list; row 0's pages wait at the tail
    assert pages.row_pages(1) == [6, 7, 8] and pages.free_list() == [9, 10, 11, 2, 4]
    lens_dev = torch.tensor([34, 40, 9], dtype=torch.int32, device=DEV)
    decode([2, 1, 3], lens_dev, 9)  # row 3 reaches position 16 one step before row 1 reaches 48
    assert pages.row_pages(1) == [6, 7, 8, 10] and pages.row_pages(3) == [3, 9]
    same_pages()


@pytest.mark.parametrize("kv", ["auto", "int8"])
def test_a_pass_is_the_same_through_the_extension_and_the_ops(kv):
    """The backend hands most calls to the extension as a whole; a call that wants a gradient, or whose values need padding,
    goes through the ops.  Same output and pages either way; what is refused there is refused here (in which words: below)."""
    gen = torch.Generator().manual_seed(9)
    hq, hkv, d, t = 8, 2, 64, 45
    backend = build_infer_attention_backend()
    q, k, v = (torch.randn(1, t, h, d, generator=gen).to(torch.bfloat16).to(DEV) for h in (hq, hkv, hkv))
    slots = torch.arange(t, device=DEV)
    table = torch.arange(8, dtype=torch.int32, device=DEV).view(2, 4)
    prefill = InferMeta(mode="prefill", cu_seqlens=torch.tensor([0, 40, t], dtype=torch.int32, device=DEV), max_seqlen=40,
                        block_table=table, cache_block_ids=slots // BS, cache_block_offsets=slots % BS)  # fmt: skip
    decode = InferMeta(mode="decode", cache_seqlens=torch.tensor([40, 5], dtype=torch.int32, device=DEV), block_table=table)
    layers = [allocate_kv_caches(1, 8, BS, hkv, d, DEV, torch.bfloat16, kv)[0] for _ in range(2)]
    for layer in layers:
        for pool in (layer.k_cache, layer.v_cache):
            pool.view(torch.uint8).zero_()
    for meta, rows in ((prefill, t), (decode, 2)):
        outs = []
        for layer, wants_grad in zip(layers, (False, True)):
            x = q[:, :rows].detach().requires_grad_(wants_grad)
            outs.append(backend(x, k[:, :rows], v[:, :rows], layer.k_cache, layer.v_cache, meta, window_size=(20, 0),
                                k_scale=layer.k_scale, v_scale=layer.v_scale))  # fmt: skip
            assert outs[-1].requires_grad == wants_grad
        assert torch.equal(outs[0], outs[1])
        for a, b in ((layers[0].k_cache, layers[1].k_cache), (layers[0].v_cache, layers[1].v_cache)):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
        bad = [(dict(q=q[..., :32]), RuntimeError), (dict(k_cache=layers[0].k_cache[0]), ValueError), (dict(q=q.cpu()), RuntimeError)]
        for changed, error in bad:
            args = {**dict(q=q[:, :rows], k=k[:, :rows], v=v[:, :rows], k_cache=layers[0].k_cache), **changed}
            if "q" in changed:
                args["q"] = args["q"][:, :rows]
            with pytest.raises((error, ValueError)):
                backend(args["q"], args["k"], args["v"], args["k_cache"], layers[0].v_cache, meta, k_scale=layers[0].k_scale,
                        v_scale=layers[0].v_scale)  # fmt: skip


def _refusals(kv, mode):
    """Calls of the backend that are refused: what they change of a good one, and of its metadata."""
    scales = [] if kv == "auto" else [
        ({"k_scale": lambda x: x[..., 0].contiguous()}, {}), ({"v_scale": lambda x: x[..., 0].contiguous()}, {}),
        ({"k_scale": lambda x: x[None], "v_scale": lambda x: x[None]}, {}), ({"k_scale": lambda x: x.transpose(1, 2)}, {}),
        ({"k_scale": lambda x: x.cpu()}, {}), ({"k_scale": lambda x: x[:4]}, {}), ({"k_scale": lambda x: None, "v_scale": lambda x: None}, {}),
        ({"v_scale": lambda x: x.bfloat16()}, {}),
    ]  # fmt: skip
    metas = {"prefill": ("cu_seqlens", "cache_block_ids", "cache_block_offsets"), "decode": ("cache_seqlens", "block_table")}[mode]
    return scales + [
        ({"k_cache": lambda x: x[0]}, {}), ({"v_cache": lambda x: x.transpose(1, 2)}, {}), ({"k_cache": lambda x: x[:4]}, {}),
        ({"v_cache": lambda x: x.cpu()}, {}), ({"q": lambda x: torch.cat([x, x], -1)}, {}), ({"q": lambda x: x.cpu()}, {}),
        ({"k": lambda x: x[:, :, :1]}, {}), ({"v": lambda x: torch.cat([x, x], 2)}, {}), ({"k": lambda x: x[:, :1]}, {}), ({"v": lambda x: x[:, :1]}, {}),
        ({"k": lambda x: x[..., :32]}, {}), ({"q": lambda x: x.half()}, {}), ({"k": lambda x: x.half()}, {}), ({"v": lambda x: x.cpu()}, {}), ({"q": lambda x: x[:, :, :3]}, {}),
    ] + [({}, {n: change}) for n in metas for change in (lambda x: x.float(), lambda x: x[None], lambda x: x.cpu())] + [({}, {}, "no number")]  # fmt: skip


@pytest.mark.parametrize("mode", ["prefill", "decode"])
@pytest.mark.parametrize("kv", ["auto", "int8"])
def test_a_refused_pass_is_refused_in_the_words_of_the_ops(kv, mode):
    """Every call that the backend refuses raises what the ops raise that it stands for, type and message."""
    hq, hkv, d, t = 8, 2, 64, 45
    backend, dtype = build_infer_attention_backend(), torch.bfloat16
    slots, table = torch.arange(t, device=DEV), torch.arange(8, dtype=torch.int32, device=DEV).view(2, 4)
    fields, rows = {
        "prefill": (dict(cu_seqlens=torch.tensor([0, 40, t], dtype=torch.int32, device=DEV), max_seqlen=40, block_table=table,
                         cache_block_ids=slots // BS, cache_block_offsets=slots % BS), t),
        "decode": (dict(cache_seqlens=torch.tensor([40, 5], dtype=torch.int32, device=DEV), block_table=table), 2),
    }[mode]  # fmt: skip
    layer = allocate_kv_caches(1, 8, BS, hkv, d, DEV, dtype, kv)[0]
    good = {n: torch.zeros(1, rows, h, d, dtype=dtype, device=DEV) for n, h in (("q", hq), ("k", hkv), ("v", hkv))}
    good["v"].normal_()
    good.update(k_cache=layer.k_cache, v_cache=layer.v_cache, k_scale=layer.k_scale, v_scale=layer.v_scale)
    scale_of = lambda x: dict(softmax_scale=x) if x is not None else {}  # noqa: E731

    def by_the_ops(a, m, scale):
        q, k, v = (a[n].reshape(-1, a[n].shape[-2], a[n].shape[-1]).contiguous() for n in "qkv")
        scales = dict(k_scale=a["k_scale"], v_scale=a["v_scale"])
        if mode == "decode":
            for n in ("cache_seqlens", "block_table"):
                if m[n].dtype != torch.int32:
                    raise ValueError(f"native decode requires int32 {n}")
            return ops.areno_paged_causal_attention_decode(q, k, v, a["k_cache"], a["v_cache"], m["block_table"].contiguous(),
                                                           m["cache_seqlens"].contiguous(), **scales, **scale_of(scale))  # fmt: skip
        ops.areno_paged_cache_write(k, v, a["k_cache"], a["v_cache"], m["cache_block_ids"], m["cache_block_offsets"], **scales)
        return ops.areno_varlen_causal_attention(q, k, v, m["cu_seqlens"].contiguous(), **scale_of(scale))

    for changes, meta_changes, *scale in _refusals(kv, mode):
        scale = scale[0] if scale else None
        a = {n: changes[n](x) if n in changes else x for n, x in good.items()}
        m = {n: meta_changes[n](x) if n in meta_changes else x for n, x in fields.items()}
        raised = []
        for call in (lambda: by_the_ops(a, m, scale),
                     lambda: backend(*(a[n] for n in ("q", "k", "v", "k_cache", "v_cache")), InferMeta(mode=mode, **m),
                                     k_scale=a["k_scale"], v_scale=a["v_scale"], **scale_of(scale))):  # fmt: skip
            with pytest.raises(Exception) as refused:
                call()
            raised.append((refused.type, str(refused.value).split("\n")[0]))
        assert raised[0] == raised[1], (list(changes), list(meta_changes), scale)
    out = [backend(*(good[n] for n in ("q", "k", "v", "k_cache", "v_cache")), InferMeta(mode=mode, **fields), k_scale=good["k_scale"],
                   v_scale=good["v_scale"], softmax_scale=x) for x in (0.25, "0.25")]  # fmt: skip
    assert torch.equal(*out)  # (whatever float() takes)
