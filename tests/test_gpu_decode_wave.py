"""The wave streaming decode kernel at the sizes where it can go wrong: every
(group, head_dim) it is built for, KV head counts that leave 1, 2 and 4 heads
per workgroup, requests ending on every side of a page, of a unit of pages and
of a segment; and its fused append, bit for bit the two calls."""
import math

import numpy as np
import pytest
import torch

from gpu_offloading_amd import workloads
from gpu_offloading_amd.kv_cache import PagedKVCache
from helpers import assert_attn_close, randn_bf16, u16
from oracle import kv_oracle as orc
from test_gpu_decode import _paged, _run

pytestmark = pytest.mark.gpu

LENS = [0, 1, 15, 16, 17, 32, 33, 100, 257, 0, 700, 513]


def _check(gpu, lens, group, d, hkv, segs, seed):
    hq = hkv * group
    kc, vc, bt, indptr, indices, lpl = _paged(lens, hkv, d, seed)
    # NaN bits past every request's end, and a missing page in the longest
    for b, n in enumerate(lens):
        if n % 16:
            kc[bt[b, n // 16], n % 16:] = math.nan
            vc[bt[b, n // 16], n % 16:] = math.nan
    long = int(np.argmax(lens))
    indices = indices.copy()
    if lens[long] > 64:
        indices[indptr[long] + 2] = -1
    q = randn_bf16((len(lens), hq, d), seed + 1, device=gpu)
    (out, lse), w = _run(gpu, q, kc.to(gpu), vc.to(gpu), indptr, indices, lpl, hq, hkv, d,
                         segs=segs)
    ref, ref_lse = orc.paged_decode(u16(q), u16(kc), u16(vc), indptr, indices, lpl)
    assert_attn_close(out.float().cpu().numpy(), ref)
    got = lse.cpu().numpy()
    fin = np.isfinite(ref_lse)
    assert np.array_equal(np.isneginf(got), ~fin)
    assert np.abs(got[fin] - ref_lse[fin]).max() < 2e-3   # fp32 sums, values below 12
    return w.schedule


@pytest.mark.parametrize("segs", [None, 5, 37])
@pytest.mark.parametrize("group,d,hkv", [(1, 64, 16), (2, 64, 6), (4, 64, 8), (8, 64, 1),
                                         (1, 128, 3), (2, 128, 4), (4, 128, 1), (8, 128, 8),
                                         (1, 256, 2), (4, 256, 4), (8, 256, 2)])
def test_wave_kernel_layouts(gpu, group, d, hkv, segs):
    sched = _check(gpu, LENS, group, d, hkv, segs, 400 + hkv)
    assert sched.heads_per_group in (1, 2, 4)


@pytest.mark.parametrize("d", [64, 256])
def test_short_requests_are_one_segment_each(gpu, d):
    sched = _check(gpu, [256, 0, 1, 17, 90, 33], 4, d, 4, None, 431)
    assert sched.num_segments == 5 and sched.max_partitions == 1


@pytest.mark.parametrize("group,lens,heads", [
    (4, [4000], 1),                     # few pages of one request
    (4, [4001, 9000, 8000], 2),
    (4, [300, 500, 16, 410, 290], 4),   # short requests
    (1, [3000, 1600], 2),
    (4, [20] * 29 + [300], 8),          # very short: the LDS kernel
    (2, [600, 500], 8),
])
def test_small_batches_of_the_lds_layout(gpu, group, lens, heads):
    assert _check(gpu, lens, group, 128, 8, None, 440).heads_per_group == heads


@pytest.mark.parametrize("hkv,group,d,lens,segs", [
    (2, 4, 128, [100, 7, 600, 64], None),
    (6, 4, 128, [300, 16, 15, 31], None),
    (8, 8, 128, [300, 1, 513], None),
    (8, 4, 128, [900, 0, 15, 700, 16], None),      # LDS layout, wave schedule
    (4, 4, 64, list(range(1, 41)), 3),             # more request ends than are loaded ahead
    (4, 1, 64, [16, 31, 47, 48, 500], None),
    (2, 8, 256, [31, 32, 300], None),
    (3, 2, 256, [20] * 9, 2),
])
@pytest.mark.parametrize("offset", [0, 1])         # elements: rows off any 4-byte boundary
def test_append_in_the_decode_launch(gpu, hkv, group, d, lens, segs, offset):
    total = sum((n + 1 + 15) // 16 for n in lens) + 3
    caches = []
    for _ in range(2):
        c = PagedKVCache(1, hkv, d, max_seqs=len(lens), max_seq_len=max(lens) + 32,
                         num_qo_heads=hkv * group, kv_page_budget=total, num_segments=segs,
                         free_page_order=workloads.randperm(total, 5), device=gpu,
                         workspace_bytes=1 << 24, staging_bytes=1 << 20)
        for s, n in enumerate(lens):
            c.ensure_pages(s, (n + 1 + 15) // 16)
        c.advance(list(range(len(lens))), lens)
        c.fill_kv_random(1.0, generator=torch.Generator(device=gpu).manual_seed(6))
        caches.append(c)
    a, b = caches
    n, seqs = len(lens), list(range(len(lens)))
    g = torch.Generator(device=gpu).manual_seed(7)
    row = hkv * d
    k, v = (torch.randn(n * row + 8, generator=g, device=gpu).to(torch.bfloat16)
            [offset:offset + n * row].view(n, hkv, d) for _ in range(2))
    q = torch.randn(n, hkv * group, d, generator=g, device=gpu).to(torch.bfloat16)
    slots = a.prepare_decode_step(seqs)
    a.append(0, k, v, slots)
    out_a, lse_a = a.decode(0, q, return_lse=True)
    b.prepare_decode_step(seqs)
    if offset and b._decode_wrapper.fused_append_supported:
        with pytest.raises(RuntimeError, match="aligned"):
            b.append_and_decode(0, k, v, q)
        return
    out_b, lse_b = b.append_and_decode(0, k, v, q, return_lse=True)
    torch.cuda.synchronize()
    assert torch.equal(a.k_cache[0], b.k_cache[0]) and torch.equal(a.v_cache[0], b.v_cache[0])
    assert torch.equal(out_a, out_b) and torch.equal(lse_a, lse_b)
    assert not torch.equal(out_a, torch.zeros_like(out_a))
