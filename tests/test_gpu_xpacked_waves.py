"""x-packed decode at each workgroup size: partitions of 4 and (large grids) 8
waves, whole sequences of 8, each wave taking page pairs.  Odd page counts,
waves without pages, block-table entries of -1 and past the cache (whose tokens
are hidden) and NaN bits in hidden pages and rows past the end; against the fp32
oracle within the attention tolerance."""
import numpy as np
import pytest
import torch

from gpu_offloading_amd import ops
from helpers import assert_attn_close, u16
from oracle import kv_oracle as orc
from test_gpu_xpacked import _attn_case, _run_v2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,group,hkv,many", [
    ("fp16", 1, 32, True), ("bf16", 2, 16, True), ("bf16", 8, 4, True),
    ("fp16", 1, 3, False), ("bf16", 4, 2, False), ("fp16", 8, 1, False),
    ("fp16", 1, 8, False), ("bf16", 4, 6, False), ("bf16", 8, 6, False)])
def test_page_pairs_and_missing_pages(gpu, dt, group, hkv, many):
    lens = [0, 1, 15, 16, 17, 31, 32, 33, 129, 255, 257, 511, 512, 513, 545, 1100]
    # v2 runs 8 waves from 4096 (KV head, sequence, partition) workgroups on, with
    # fewer than 16 KV heads from 8192, and up to 256; here 48, 96, 144 and 288, 384
    max_len = 512 * ((4096 if hkv >= 16 else 8192) // (hkv * len(lens))) if many else 1100
    q, kc, vc, bt = _attn_case(lens, hkv * group, hkv, dt, 90 + group, gpu)
    hidden = [(9, 3, -1), (10, 0, kc.shape[0]), (10, 1, -1), (13, 31, -1), (13, 32, -1),
              (14, 34, kc.shape[0] + 3)] + [(15, p, -1) for p in range(2, 20)]
    for b, page, value in hidden:
        kc[bt[b, page]] = vc[bt[b, page]] = float("nan")
        bt[b, page] = value
    ref_bt, ref_lens = np.full_like(bt, -1), []
    for b, n in enumerate(lens):
        ids = [(int(i), min(16, n - 16 * p)) for p, i in enumerate(bt[b, :(n + 15) // 16])]
        ids = [(i, t) for i, t in ids if 0 <= i < kc.shape[0]]
        # a partial page stays last: only its rows from t on are past the end
        assert all(t == 16 for _, t in ids[:-1])
        if ids and ids[-1][1] < 16:
            kc[ids[-1][0], :, :, ids[-1][1]:] = float("nan")
            vc[ids[-1][0], :, :, ids[-1][1]:] = float("nan")
        ref_bt[b, :len(ids)] = [i for i, _ in ids]
        ref_lens.append(sum(t for _, t in ids))
    scale = 0.08
    ref, *_ = orc.paged_attention_xpacked(u16(q), u16(kc), u16(vc), ref_bt, np.array(ref_lens),
                                          scale, dtype=dt)
    out1 = torch.empty_like(q)
    ops.paged_attention_v1(out1, q, kc, vc, hkv, scale, torch.from_numpy(bt).to(gpu),
                           torch.tensor(lens, dtype=torch.int32, device=gpu), 16, max(lens),
                           None, "auto", 1.0, 1.0)
    out2, *_ = _run_v2(q, kc, vc, bt, lens, hkv, scale, gpu, max_seq_len=max_len)
    for out in (out1, out2):
        assert_attn_close(out.float().cpu().numpy(), ref)


@pytest.mark.parametrize("dt,group,hkv", [("fp16", 1, 8), ("bf16", 4, 2), ("fp16", 8, 1)])
@pytest.mark.parametrize("longest", [512, 513])
@pytest.mark.parametrize("times", [1, 26])
def test_v1_of_short_sequences(gpu, dt, group, hkv, longest, times):
    # v1: 4 waves up to 512 tokens and from 257 workgroups (here 12 to 312 a KV head)
    lens = [0, 1, 16, 17, 33, 100, 128, 129, 160, 255, 257, longest] * times
    q, kc, vc, bt = _attn_case(lens, hkv * group, hkv, dt, 130 + group, gpu)
    for b, n in enumerate(lens):
        if n % 16:
            kc[bt[b, n // 16], :, :, n % 16:] = float("nan")
            vc[bt[b, n // 16], :, :, n % 16:] = float("nan")
    ref, *_ = orc.paged_attention_xpacked(u16(q), u16(kc), u16(vc), bt, np.array(lens), 0.08,
                                          dtype=dt)
    out = torch.empty_like(q)
    ops.paged_attention_v1(out, q, kc, vc, hkv, 0.08, torch.from_numpy(bt).to(gpu),
                           torch.tensor(lens, dtype=torch.int32, device=gpu), 16, longest,
                           None, "auto", 1.0, 1.0)
    assert_attn_close(out.float().cpu().numpy(), ref)
