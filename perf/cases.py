"""Performance cases of the paged KV-cache path.

Each case is one pass of work that an inference engine has this package do,
through its public entry points, over inputs already on the GPU:

  decode    one layer of a decode step: ``PagedKVCache.append_and_decode``
            (the new token's K/V appended, then paged GQA decode attention)
            after ``prepare_decode_step`` planned the step
  step      a decode step in the engine's FlashInfer / vLLM call shape:
            ``BatchDecodeWithPagedKVCacheWrapper.plan`` and, per layer,
            ``reshape_and_cache_flash`` and ``run``
  prefill   one layer of a continuation-prefill step: ``PagedKVCache.append``
            of the chunks and ``prefill`` over everything cached (causal)
  copy      the append of a chunk of every sequence and the gather of the
            whole sequences into contiguous rows
  evict     the device half of a swap: ``gather_blocks`` of the victims into
            the staging buffer and ``scatter_blocks`` into other blocks (the
            host-link half is the runtime's copy, bound by the link)
  xpacked   one layer of the dense sandbox's mixed step in vLLM's x-packed
            layout: ``reshape_and_cache`` of the prompts' and the decodes' new
            tokens and ``paged_attention_v2`` (or v1) of the decodes

``listed()`` are fixed cases, ``draw(rng)`` gives further ones of the same
ranges.  Pages are always 16 tokens from a seeded permuted pool; K, V and Q
are N(0, 1) (Q N(0, 9) on the longest contexts).
"""
from __future__ import annotations

import math
import random

import torch

from gpu_offloading_amd import ops
from gpu_offloading_amd.decode import BatchDecodeWithPagedKVCacheWrapper
from gpu_offloading_amd.kv_cache import PagedKVCache

PAGE = 16
DEVICE = "cuda"


# ------------------------------------------------------------------- cases
def listed():
    return [
        # The reference's published latency point: one request just past a
        # 128-token prompt, Mixtral attention.
        dict(name="decode_b1_ctx129", kind="decode", batch=1, lo=128, hi=128, hkv=8, group=4,
             dim=128, lse=False, q_std=1.0, lens_seed=0),
        # A small interactive batch with ragged contexts, called the way the
        # engine calls vLLM and FlashInfer: plan, then append + run per layer.
        dict(name="step_b8_ragged", kind="step", layers=4, batch=8, lo=300, hi=2000, hkv=8,
             group=4, dim=128, lens_seed=1),
        # The serving decode step of the benchmark: Mixtral shape, 64 requests.
        dict(name="decode_b64_mixtral", kind="decode", batch=64, lo=512, hi=4096, hkv=8, group=4,
             dim=128, lse=False, q_std=1.0, lens_seed=2),
        # Long-context decode: 16 requests at 32K tokens, logits with std ~3.
        dict(name="decode_b16_32k", kind="decode", batch=16, lo=32767, hi=32767, hkv=8, group=4,
             dim=128, lse=False, q_std=3.0, lens_seed=0),
        # OLMoE shape (multi-head attention, 16 heads), a full batch.
        dict(name="decode_b128_olmoe", kind="decode", batch=128, lo=1024, hi=3072, hkv=16,
             group=1, dim=128, lse=False, q_std=1.0, lens_seed=3),
        # One GPU's shard of Mixtral under tensor parallelism over 8 GPUs:
        # one KV head and its four query heads.
        dict(name="decode_b64_tp8", kind="decode", batch=64, lo=512, hi=4096, hkv=1, group=4,
             dim=128, lse=False, q_std=1.0, lens_seed=4),
        # head_dim 64 with eight query heads per KV head, log-sum-exp returned
        # (partial attention that the caller merges).
        dict(name="decode_b32_d64_g8", kind="decode", batch=32, lo=500, hi=3001, hkv=8, group=8,
             dim=64, lse=True, q_std=1.0, lens_seed=5),
        # Chunked prefill in bulk: the second 2048-token chunk of 8 prompts.
        dict(name="prefill_8x2048", kind="prefill", batch=8, q_lo=2048, q_hi=2048, past_lo=2048,
             past_hi=2048, hkv=8, group=4, dim=128, lens_seed=0),
        # Chunked prefill beside decodes: a few short ragged chunks over long
        # histories (the tail of a prompt, a follow-up turn of a chat).
        dict(name="prefill_ragged_chunks", kind="prefill", batch=3, q_lo=60, q_hi=400,
             past_lo=3000, past_hi=8000, hkv=8, group=4, dim=128, lens_seed=6),
        # Chunk append and gather into contiguous rows, 8 x 2048 tokens.
        dict(name="copy_8x2048", kind="copy", batch=8, new=2048, past_lo=0, past_hi=0, hkv=8,
             dim=128, lens_seed=0),
        # Eviction and restore of 16 2048-token OLMoE sequences (one layer).
        dict(name="evict_2048_blocks", kind="evict", blocks=2048, pool=8192, hkv=16, dim=128),
        # The dense sandbox's mixed step: 32 heads, fp16, 64 decodes and two
        # 512-token prompts.
        dict(name="xpacked_mixed_fp16", kind="xpacked", dtype="float16", v2=True, heads=32,
             group=1, batch=64, lo=512, hi=4096, prefills=2, prefill_len=512, lens_seed=7),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "step", "prefill", "prefill", "copy",
                       "evict", "xpacked"])
    ls = rng.randrange(1 << 20)
    hkv = rng.choice([1, 2, 4, 8, 8, 16])
    if kind == "decode":
        dim, group = rng.choice([64, 128, 128, 128, 256]), rng.choice([1, 2, 4, 4, 8])
        batch = _log(rng, 1, 128)
        most = (1 << 30) // (batch * hkv * dim * 4)          # at most 1 GB of K and V
        hi = _log(rng, 2, max(3, min(32767, most)))
        return dict(kind=kind, batch=batch, lo=max(1, int(hi * rng.uniform(0.1, 1.0))), hi=hi,
                    hkv=hkv, group=group, dim=dim, lse=rng.random() < 0.25,
                    q_std=3.0 if hi > 16000 else 1.0, lens_seed=ls)
    if kind == "step":
        batch, hi = _log(rng, 1, 32), _log(rng, 20, 4000)
        return dict(kind=kind, layers=rng.choice([2, 3, 4]), batch=batch,
                    lo=max(1, int(hi * rng.uniform(0.1, 1.0))), hi=hi, hkv=hkv,
                    group=rng.choice([1, 4, 8]), dim=128, lens_seed=ls)
    if kind == "prefill":
        group, batch = rng.choice([1, 2, 4, 4, 8]), _log(rng, 1, 8)
        hkv = min(hkv, 8)
        q_hi = _log(rng, 9, 2048)
        # at most the pairs of 8 x 2048 queries over 4096 keys with 32 heads
        most = 8 * 2048 * 3072 * 32 // (batch * q_hi * hkv * group) - q_hi
        past_hi = _log(rng, 1, max(2, min(30000, most)))
        return dict(kind=kind, batch=batch, q_lo=max(1, int(q_hi * rng.uniform(0.2, 1.0))),
                    q_hi=q_hi, past_lo=int(past_hi * rng.uniform(0.2, 1.0)), past_hi=past_hi,
                    hkv=hkv, group=group, dim=128, lens_seed=ls)
    if kind == "copy":
        batch, dim = _log(rng, 1, 64), rng.choice([64, 128, 256])
        new = _log(rng, 1, 16384 * 8 * 128 // (batch * 16 * 256))
        past = _log(rng, 1, 2048 * 8 // batch)
        return dict(kind=kind, batch=batch, new=new, past_lo=past // 3, past_hi=past, hkv=hkv,
                    dim=dim, lens_seed=ls)
    if kind == "evict":
        blocks = _log(rng, 8, 2048)
        return dict(kind=kind, blocks=blocks, pool=4 * blocks, hkv=hkv,
                    dim=rng.choice([64, 128]))
    heads, group = rng.choice([(32, 1), (16, 1), (8, 4), (4, 8), (8, 1), (4, 2)])
    batch = _log(rng, 1, 64)
    hi = _log(rng, 30, max(100, 64 * 4096 * 8 // (batch * heads)))
    v2 = rng.random() < 0.8
    return dict(kind=kind, dtype=rng.choice(["float16", "bfloat16"]), v2=v2, heads=heads,
                group=group, batch=batch, lo=max(1, int(hi * rng.uniform(0.1, 1.0))),
                hi=hi if v2 else min(hi, 4096), prefills=rng.choice([0, 1, 2, 4]),
                prefill_len=_log(rng, 16, 512), lens_seed=ls)


# ------------------------------------------------------------------ inputs
def _lens(case, lo, hi, n, salt=0):
    """The case's ragged lengths (part of the case, not of the inputs)."""
    r = random.Random(case["lens_seed"] * 8 + salt)
    return [r.randint(min(lo, hi), hi) for _ in range(n)]


def _pages(n):
    return (n + PAGE - 1) // PAGE


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _randn(shape, g, dtype=torch.bfloat16, std=1.0):
    return torch.empty(shape, dtype=dtype, device=DEVICE).normal_(0.0, std, generator=g)


def _order(n, seed):
    """The pool's free list: a seeded permutation of its pages."""
    order = list(range(n))
    random.Random(seed).shuffle(order)
    return order


def _tables(counts, order):
    """Each sequence's pages, taken from the free list in order."""
    out, at = [], 0
    for n in counts:
        out.append(order[at:at + n])
        at += n
    return out


def _decode_inputs(case, seed):
    """(lens with the new token, pages, free list, per-layer caches, q, k, v)."""
    layers = case.get("layers", 1)
    lens = [n + 1 for n in _lens(case, case["lo"], case["hi"], case["batch"])]
    total = sum(_pages(n) for n in lens) + case["batch"]
    g, hkv, d = _gen(seed), case["hkv"], case["dim"]
    caches = [_randn((total, 2, PAGE, hkv, d), g) for _ in range(layers)]
    q = [_randn((case["batch"], hkv * case["group"], d), g, std=case.get("q_std", 1.0))
         for _ in range(layers)]
    k = [_randn((case["batch"], hkv, d), g) for _ in range(layers)]
    v = [_randn((case["batch"], hkv, d), g) for _ in range(layers)]
    return lens, total, _order(total, seed), caches, q, k, v


def _prefill_inputs(case, seed):
    past = _lens(case, case["past_lo"], case["past_hi"], case["batch"])
    chunk = _lens(case, case["q_lo"], case["q_hi"], case["batch"], 1)
    total = sum(_pages(p + c) for p, c in zip(past, chunk)) + 1
    g, hkv, d = _gen(seed), case["hkv"], case["dim"]
    cache = _randn((total, 2, PAGE, hkv, d), g)
    n = sum(chunk)
    return (past, chunk, total, _order(total, seed), cache,
            _randn((n, hkv * case["group"], d), g), _randn((n, hkv, d), g),
            _randn((n, hkv, d), g))


def _copy_inputs(case, seed):
    past = _lens(case, case["past_lo"], case["past_hi"], case["batch"])
    total = sum(_pages(p + case["new"]) for p in past) * 5 // 4 + 1
    g, hkv, d = _gen(seed), case["hkv"], case["dim"]
    cache = _randn((total, 2, PAGE, hkv, d), g)
    n = case["new"] * case["batch"]
    return (past, total, _order(total, seed), cache, _randn((n, hkv, d), g),
            _randn((n, hkv, d), g))


def _evict_inputs(case, seed):
    order = _order(case["pool"], seed)
    n = case["blocks"]
    ids = [torch.tensor(order[i * n:(i + 1) * n], dtype=torch.int32, device=DEVICE)
           for i in (0, 1)]
    return _randn((case["pool"], 2, PAGE, case["hkv"], case["dim"]), _gen(seed)), ids


def _xpacked_inputs(case, seed):
    """Prompts first, then the decodes; the block table has one row each."""
    dt = getattr(torch, case["dtype"])
    lens = [case["prefill_len"]] * case["prefills"] + \
        [n + 1 for n in _lens(case, case["lo"], case["hi"], case["batch"])]
    first = [0] * case["prefills"] + [n - 1 for n in lens[case["prefills"]:]]
    total = sum(_pages(n) for n in lens) + 1
    rows = _tables([_pages(n) for n in lens], _order(total, seed))
    g, h, d, hq = _gen(seed), case["heads"], 128, case["heads"] * case["group"]
    n_new = sum(n - f for n, f in zip(lens, first))
    kc = _randn((total, h, d // 8, PAGE, 8), g, dt)
    vc = _randn((total, h, d, PAGE), g, dt)
    k, v = _randn((n_new, h, d), g, dt), _randn((n_new, h, d), g, dt)
    q = _randn((case["batch"], hq, d), g, dt)
    slots = [row[p // PAGE] * PAGE + p % PAGE
             for row, n, f in zip(rows, lens, first) for p in range(f, n)]
    return lens, rows, kc, vc, k, v, q, torch.tensor(slots, dtype=torch.int64, device=DEVICE)


# ----------------------------------------------------------------- prepare
def _cache(case, caches, total, order, seqs, max_len):
    """A PagedKVCache whose pages hold ``caches``."""
    c = PagedKVCache(len(caches), case["hkv"], case["dim"], max_seqs=seqs,
                     max_seq_len=max_len, num_qo_heads=case["hkv"] * case.get("group", 1),
                     kv_page_budget=total, free_page_order=order, device=DEVICE)
    for dst, src in zip(c.kv_cache, caches):
        dst.copy_(src)
    return c


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        lens, total, order, caches, q, k, v = _decode_inputs(case, seed)
        seqs = list(range(case["batch"]))
        c = _cache(case, caches, total, order, len(seqs), max(lens) + PAGE)
        for s, n in zip(seqs, lens):
            c.ensure_pages(s, _pages(n))
        c.advance(seqs, [n - 1 for n in lens])
        c.prepare_decode_step(seqs)
        return dict(kind=kind, cache=c, q=q[0], k=k[0], v=v[0], lse=case["lse"])
    if kind == "step":
        lens, total, order, caches, q, k, v = _decode_inputs(case, seed)
        rows = _tables([_pages(n) for n in lens], order)
        indptr = [0]
        for r in rows:
            indptr.append(indptr[-1] + len(r))
        slots = [r[-1] * PAGE + (n - 1) % PAGE for r, n in zip(rows, lens)]
        ws = torch.empty(128 << 20, dtype=torch.uint8, device=DEVICE)
        return dict(kind=kind, wrapper=BatchDecodeWithPagedKVCacheWrapper(ws, "NHD"),
                    indptr=torch.tensor(indptr, dtype=torch.int32),
                    indices=torch.tensor(sum(rows, []), dtype=torch.int32, device=DEVICE),
                    lpl=torch.tensor([(n - 1) % PAGE + 1 for n in lens], dtype=torch.int32),
                    slots=torch.tensor(slots, dtype=torch.int64, device=DEVICE),
                    heads=(case["hkv"] * case["group"], case["hkv"], case["dim"]),
                    kc=[t[:, 0] for t in caches], vc=[t[:, 1] for t in caches], q=q, k=k, v=v)
    if kind == "prefill":
        past, chunk, total, order, cache, q, k, v = _prefill_inputs(case, seed)
        seqs = list(range(case["batch"]))
        top = max(p + n for p, n in zip(past, chunk))
        c = _cache(case, [cache], total, order, len(seqs), top + PAGE)
        for s, p, n in zip(seqs, past, chunk):
            c.ensure_pages(s, _pages(p + n))
        c.advance(seqs, past)
        slots = c.prepare_prefill_chunk(seqs, chunk)
        return dict(kind=kind, cache=c, q=q, k=k, v=v, slots=slots)
    if kind == "copy":
        past, total, order, cache, k, v = _copy_inputs(case, seed)
        seqs = list(range(case["batch"]))
        c = _cache(case, [cache], total, order, len(seqs), max(past) + case["new"] + PAGE)
        for s, p in zip(seqs, past):
            c.ensure_pages(s, _pages(p + case["new"]))
        c.advance(seqs, past)
        slots = c.slot_mapping(seqs, [case["new"]] * len(seqs))
        lens = [p + case["new"] for p in past]
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        shape = (cu[-1], case["hkv"], case["dim"])
        return dict(kind=kind, cache=c, k=k, v=v, slots=slots, table=c.block_table,
                    cu=torch.tensor(cu, dtype=torch.int32, device=DEVICE), max_len=max(lens),
                    out_k=torch.zeros(shape, dtype=torch.bfloat16, device=DEVICE),
                    out_v=torch.zeros(shape, dtype=torch.bfloat16, device=DEVICE))
    if kind == "evict":
        cache, ids = _evict_inputs(case, seed)
        per = PAGE * case["hkv"] * case["dim"]
        staging = torch.zeros((case["blocks"], 2, per), dtype=torch.bfloat16, device=DEVICE)
        return dict(kind=kind, kc=cache[:, 0], vc=cache[:, 1], src=ids[0], dst=ids[1],
                    staging=staging)
    lens, rows, kc, vc, k, v, q, slots = _xpacked_inputs(case, seed)
    dec, dl = rows[case["prefills"]:], lens[case["prefills"]:]
    width = max(len(r) for r in dec)
    bt = torch.tensor([r + [0] * (width - len(r)) for r in dec], dtype=torch.int32,
                      device=DEVICE)
    hq, parts = case["heads"] * case["group"], (max(dl) + 511) // 512
    scratch = (case["batch"], hq, parts)
    return dict(kind=kind, v2=case["v2"], kc=kc, vc=vc, k=k, v=v, q=q, slots=slots, bt=bt,
                lens=torch.tensor(dl, dtype=torch.int32, device=DEVICE), max_len=max(dl),
                out=torch.zeros_like(q),
                exp_sums=torch.zeros(scratch, dtype=torch.float32, device=DEVICE),
                max_logits=torch.zeros(scratch, dtype=torch.float32, device=DEVICE),
                tmp=torch.zeros(scratch + (128,), dtype=q.dtype, device=DEVICE))


# --------------------------------------------------------------------- run
def run(s):
    kind = s["kind"]
    if kind == "decode":
        c = s["cache"]
        got = c.append_and_decode(0, s["k"], s["v"], s["q"], return_lse=s["lse"])
        out, lse = got if s["lse"] else (got, None)
        res = dict(out=out, k=c.k_cache[0], v=c.v_cache[0])
        if s["lse"]:
            res["lse"] = lse
        return res
    if kind == "step":
        w, (hq, hkv, d) = s["wrapper"], s["heads"]
        w.plan(s["indptr"], s["indices"], s["lpl"], num_qo_heads=hq, num_kv_heads=hkv,
               head_dim=d, page_size=PAGE, pos_encoding_mode="NONE",
               q_data_type=torch.bfloat16)
        outs = []
        for layer, (kc, vc) in enumerate(zip(s["kc"], s["vc"])):
            ops.reshape_and_cache_flash(s["k"][layer], s["v"][layer], kc, vc, s["slots"], "auto")
            outs.append(w.run(s["q"][layer], (kc, vc)))
        return dict(out=outs, k=s["kc"], v=s["vc"])
    if kind == "prefill":
        c = s["cache"]
        c.append(0, s["k"], s["v"], s["slots"])
        return dict(out=c.prefill(0, s["q"]), k=c.k_cache[0], v=c.v_cache[0])
    if kind == "copy":
        c = s["cache"]
        c.append(0, s["k"], s["v"], s["slots"])
        ops.gather_kv(c.k_cache[0], c.v_cache[0], s["table"], s["cu"], s["max_len"],
                      s["out_k"], s["out_v"])
        return dict(k=c.k_cache[0], v=c.v_cache[0], out_k=s["out_k"], out_v=s["out_v"])
    if kind == "evict":
        ops.gather_blocks(s["kc"], s["vc"], s["src"], s["staging"])
        ops.scatter_blocks(s["staging"], s["dst"], s["kc"], s["vc"])
        return dict(staging=s["staging"], k=s["kc"], v=s["vc"])
    ops.reshape_and_cache(s["k"], s["v"], s["kc"], s["vc"], s["slots"])
    heads, scale = s["kc"].shape[1], 1.0 / math.sqrt(128)
    if s["v2"]:
        ops.paged_attention_v2(s["out"], s["exp_sums"], s["max_logits"], s["tmp"], s["q"],
                               s["kc"], s["vc"], heads, scale, s["bt"], s["lens"], PAGE,
                               s["max_len"])
    else:
        ops.paged_attention_v1(s["out"], s["q"], s["kc"], s["vc"], heads, scale, s["bt"],
                               s["lens"], PAGE, s["max_len"])
    return dict(out=s["out"], kc=s["kc"], vc=s["vc"])


# -------------------------------------------------------------------- work
def work(case):
    """Every K and V row read once, q and the new rows read once, the output
    and the appended rows written once."""
    kind = case["kind"]
    if kind in ("decode", "step"):
        row = case["hkv"] * case["dim"] * 2
        lens = [n + 1 for n in _lens(case, case["lo"], case["hi"], case["batch"])]
        hq, b, layers = case["hkv"] * case["group"], case["batch"], case.get("layers", 1)
        return dict(bytes=layers * (2 * row * sum(lens) + 4 * row * b
                                    + 4 * b * hq * case["dim"]),
                    flops=layers * 4 * sum(lens) * hq * case["dim"])
    if kind == "prefill":
        past = _lens(case, case["past_lo"], case["past_hi"], case["batch"])
        chunk = _lens(case, case["q_lo"], case["q_hi"], case["batch"], 1)
        row, hq = case["hkv"] * case["dim"] * 2, case["hkv"] * case["group"]
        pairs = sum(n * p + n * (n + 1) // 2 for p, n in zip(past, chunk))
        return dict(bytes=2 * row * sum(p + n for p, n in zip(past, chunk))
                    + 4 * row * sum(chunk) + 4 * sum(chunk) * hq * case["dim"],
                    flops=4 * pairs * hq * case["dim"])
    if kind == "copy":
        row, n = case["hkv"] * case["dim"] * 2, case["new"] * case["batch"]
        past = _lens(case, case["past_lo"], case["past_hi"], case["batch"])
        return dict(bytes=4 * row * n + 4 * row * (n + sum(past)) + 8 * n, flops=0)
    if kind == "evict":
        return dict(bytes=4 * 2 * PAGE * case["hkv"] * case["dim"] * 2 * case["blocks"], flops=0)
    row, hq, b = case["heads"] * 128 * 2, case["heads"] * case["group"], case["batch"]
    total = sum(_lens(case, case["lo"], case["hi"], b)) + b
    new = case["prefills"] * case["prefill_len"] + b
    return dict(bytes=2 * row * total + 4 * row * new + 4 * b * hq * 128,
                flops=4 * total * hq * 128)


# --------------------------------------------------------------- tolerance
def tolerance(case):
    """Byte moves are exact.  Attention: about four times each path's measured
    distance from fp64, which rounding the output to 16 bits makes up (1.7e-3
    in bf16, where the softmax weights stay fp32; 2.3e-3 where they are rounded
    to bf16 as well, in the prefill and the x-packed kernels; 3.3e-4 in
    fp16)."""
    kind = case["kind"]
    if kind in ("copy", "evict"):
        return "exact"
    if kind == "xpacked" and case["dtype"] == "float16":
        return {"rel": 1.5e-3, "max": 0.03}
    if kind in ("prefill", "xpacked"):
        return {"rel": 9e-3, "max": 0.15}
    return {"rel": 7e-3, "max": 0.1}


# ------------------------------------------------------------------- exact
def _attend(q, k, v, causal_from=None):
    """fp64 attention of q [n, hq, d] over k, v [len, hkv, d]: (out, lse)."""
    n, hq, d = q.shape
    group = hq // k.shape[1]
    out = torch.empty(n, hq, d, dtype=torch.float64, device=q.device)
    lse = torch.empty(n, hq, dtype=torch.float64, device=q.device)
    for h in range(k.shape[1]):
        qq = q[:, h * group:(h + 1) * group].double().reshape(n * group, d)
        s = (qq @ k[:, h].double().t().contiguous()) / math.sqrt(d)
        if causal_from is not None:
            last = causal_from + torch.arange(n, device=q.device).repeat_interleave(group)
            s.masked_fill_(torch.arange(k.shape[0], device=q.device)[None] > last[:, None],
                           -math.inf)
        top = torch.logsumexp(s, dim=1, keepdim=True)
        o = (s - top).exp_() @ v[:, h].double()
        out[:, h * group:(h + 1) * group] = o.view(n, group, d)
        lse[:, h * group:(h + 1) * group] = top.view(n, group)
    return out, lse


def _rows(cache, pages, n):
    """The first n token rows of a sequence, [n, heads, dim], K and V."""
    t = cache[torch.tensor(pages, device=cache.device)]
    return t[:, 0].flatten(0, 1)[:n], t[:, 1].flatten(0, 1)[:n]


def _write(cache, pages, first, k, v):
    """Token rows first .. of a sequence take k, v."""
    pos = torch.arange(first, first + k.shape[0], device=cache.device)
    page = torch.tensor(pages, device=cache.device)[pos // PAGE]
    cache[page, 0, pos % PAGE] = k
    cache[page, 1, pos % PAGE] = v


def _exact_decode(case, seed):
    lens, _, order, caches, q, k, v = _decode_inputs(case, seed)
    rows = _tables([_pages(n) for n in lens], order)
    outs, lses = [], []
    for layer, cache in enumerate(caches):
        out, lse = torch.empty_like(q[layer], dtype=torch.float64), []
        for b, (n, pages) in enumerate(zip(lens, rows)):
            _write(cache, pages, n - 1, k[layer][b:b + 1], v[layer][b:b + 1])
            o, top = _attend(q[layer][b:b + 1], *_rows(cache, pages, n))
            out[b] = o[0]
            lse.append(top)
        outs.append(out)
        lses.append(torch.cat(lse))
    return outs, lses, caches


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        outs, lses, caches = _exact_decode(case, seed)
        res = dict(out=outs[0], k=caches[0][:, 0], v=caches[0][:, 1])
        if case["lse"]:
            res["lse"] = lses[0]
        return res
    if kind == "step":
        outs, _, caches = _exact_decode(case, seed)
        return dict(out=outs, k=[c[:, 0] for c in caches], v=[c[:, 1] for c in caches])
    if kind == "prefill":
        past, chunk, _, order, cache, q, k, v = _prefill_inputs(case, seed)
        rows = _tables([_pages(p + n) for p, n in zip(past, chunk)], order)
        out, at = torch.empty_like(q, dtype=torch.float64), 0
        for p, n, pages in zip(past, chunk, rows):
            _write(cache, pages, p, k[at:at + n], v[at:at + n])
            out[at:at + n] = _attend(q[at:at + n], *_rows(cache, pages, p + n),
                                     causal_from=p)[0]
            at += n
        return dict(out=out, k=cache[:, 0], v=cache[:, 1])
    if kind == "copy":
        past, _, order, cache, k, v = _copy_inputs(case, seed)
        new, got = case["new"], []
        for b, (p, pages) in enumerate(zip(past, _tables([_pages(p + new) for p in past],
                                                         order))):
            _write(cache, pages, p, k[b * new:(b + 1) * new], v[b * new:(b + 1) * new])
            got.append(_rows(cache, pages, p + new))
        return dict(k=cache[:, 0], v=cache[:, 1], out_k=torch.cat([g[0] for g in got]),
                    out_v=torch.cat([g[1] for g in got]))
    if kind == "evict":
        cache, (src, dst) = _evict_inputs(case, seed)
        moved = cache[src.long()]
        cache[dst.long()] = moved
        return dict(staging=moved.flatten(2), k=cache[:, 0], v=cache[:, 1])
    lens, rows, kc, vc, k, v, q, slots = _xpacked_inputs(case, seed)
    blk, off = slots // PAGE, slots % PAGE
    kc[blk, :, :, off] = k.unflatten(2, (16, 8))
    vc[blk, :, :, off] = v
    out, first = torch.empty_like(q, dtype=torch.float64), case["prefills"]
    for b, (n, pages) in enumerate(zip(lens[first:], rows[first:])):
        at = torch.tensor(pages, device=DEVICE)
        kk = kc[at].permute(0, 3, 1, 2, 4).flatten(3).flatten(0, 1)[:n]   # [tokens, heads, 128]
        vv = vc[at].permute(0, 3, 1, 2).flatten(0, 1)[:n]
        out[b] = _attend(q[b:b + 1], kk, vv)[0][0]
    return dict(out=out, kc=kc, vc=vc)
