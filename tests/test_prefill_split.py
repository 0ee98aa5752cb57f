"""Continuation prefill of few units over long histories: units cut along their
keys, merged from fp32 partials.  The plan on the CPU (every key tile of every
unit once, the whole units' plan behind it), the kernels against the fp32
oracle within the bounds of tests/test_gpu_prefill.py: the merge adds only fp32
rounding (partials stay fp32, weights are exp2 of fp32 differences)."""
import numpy as np
import pytest
import torch

from gpu_offloading_amd import _lib
from gpu_offloading_amd.prefill import BatchPrefillWithPagedKVCacheWrapper
from helpers import assert_attn_close, u16
from oracle import kv_oracle as orc
from test_gpu_prefill import LSE_TOL, WS, _case

KEYS = 64  # keys per tile


def _plan(q_lens, kv_lens, group, hkv, causal):
    qo = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    kvi, lpl = orc.plan_decode(kv_lens)
    kvi, lpl = kvi.astype(np.int32), lpl.astype(np.int32)
    cap = BatchPrefillWithPagedKVCacheWrapper._plan_capacity(np.asarray(q_lens), group, hkv)

    def image(split):
        sched, img = _lib.KvcPrefillSchedule(), np.full(cap, -7, np.int32)
        args = [qo.ctypes.data, kvi.ctypes.data, lpl.ctypes.data, len(q_lens), group * hkv, hkv,
                128, 16, causal, sched]
        if split is None:
            _lib.call("kvc_prefill_plan", *args, img.ctypes.data, cap)
        else:
            _lib.call("kvc_prefill_plan_split", *args, split, img.ctypes.data, cap)
        return sched, img

    split = _lib.KvcPrefillSplit()
    return image(None), image(split), split


def _units(img, num_units, workgroups):
    table = (2 * workgroups + 3) // 4 * 4
    return (img[table:table + 8 * num_units].reshape(-1, 8),
            img[:2 * workgroups].reshape(-1, 2))


@pytest.mark.parametrize("q_lens,kv_lens,group,hkv,causal,cut", [
    ([40, 41, 39], [26000, 29000, 25000], 8, 1, 1, True),
    ([1, 0, 300, 7], [2500, 90, 1500, 1025], 4, 2, 1, True),
    ([700], [1400], 4, 8, 0, True),
    ([40] * 9, [3000 + 77 * i for i in range(9)], 1, 4, 1, True),
    ([256 * 16], [256 * 16], 1, 32, 1, False),      # 512 units, balanced as they are
    ([40] + [64] * 20, [9000] + [0] * 20, 4, 8, 1, True),   # units without keys
    ([257 * 2], [30000], 1, 32, 1, True),
    ([300], [30000], 1, 32, 1, True),
    ([1024], [1024], 4, 8, 1, False),               # 16 key tiles: never cut
    ([2048] * 4, [2048] * 4, 4, 8, 1, False),       # more units: never cut
])
def test_split_plan_covers_every_key_once(q_lens, kv_lens, group, hkv, causal, cut):
    (base, base_img), (sched, img), split = _plan(q_lens, kv_lens, group, hkv, causal)
    n, off = base.num_items * hkv, split.base_offset
    assert sched.plan_ints <= img.size
    assert (img[sched.plan_ints:] == -7).all()
    assert np.array_equal(img[off:off + base.plan_ints], base_img[:base.plan_ints])
    if split.num_parts == 0:
        assert off == 0 and sched.plan_ints == base.plan_ints
        assert split.workspace_bytes == 0 and split.num_units == n
        assert not cut
        return
    assert cut
    whole, _ = _units(base_img, n, min(256, n))
    assert split.num_workgroups <= 256
    rec, wg = _units(img, split.num_units, split.num_workgroups)
    assert np.array_equal(wg[:, 0], np.concatenate([[0], np.cumsum(wg[:-1, 1])]))
    assert wg[:, 1].min() >= 1 and wg[:, 1].sum() == split.num_units
    part = img[split.parts_offset:split.parts_offset + split.num_units]
    merges = img[split.merges_offset:split.merges_offset + 8 * split.num_merges].reshape(-1, 8)
    assert sorted(part[part >= 0]) == list(range(split.num_parts))
    assert split.workspace_bytes == split.num_parts * 256 * 129 * 4
    by_unit = {}
    for r, p in zip(rec, part):
        by_unit.setdefault((r[0], r[4], r[1]), []).append((r, p))
    folded = set()
    for w in whole:
        pieces = sorted(by_unit.pop((w[0], w[4], w[1])), key=lambda x: x[0][5])
        first = 0
        for r, _ in pieces:
            assert r[2] == w[2] and r[3] == w[3] - KEYS * first
            assert r[5] - w[5] == min(first * KEYS // 16, w[7]) and r[7] == w[7] - (r[5] - w[5])
            first += r[6]
        assert first == w[6]
        ids = [int(p) for _, p in pieces]
        if len(ids) == 1:
            assert ids == [-1]
            continue
        assert w[6] > 16 and min(r[6] for r, _ in pieces) >= 1
        assert ids == list(range(ids[0], ids[0] + len(ids)))
        m = merges[(merges[:, 3] == ids[0])]
        assert len(m) == 1
        rows = min(256 // group, w[2] - w[1]) * group
        assert list(m[0]) == [w[0], w[4] + w[1], rows, ids[0], len(ids), 0, 0, 0]
        folded.add(ids[0])
    assert not by_unit and len(folded) == split.num_merges


@pytest.mark.parametrize("q_lens,cached,group,hkv,cut", [
    ([388, 510, 537], [2338, 2326, 1937], 4, 8, False),             # 391 full partials
    ([1191, 1257, 1163, 1149, 1424], [1291, 1129, 859, 1104, 1101], 1, 8, False),   # 352
    ([115, 152, 130, 138, 145, 166, 123, 194], [994, 1397, 1137, 1121, 833, 860, 1180, 1426], 1, 4, True),
    ([374, 392], [6335, 8879], 8, 8, True),                         # long enough for many
    ([1] * 40, [3000] * 40, 8, 4, True)])                           # partials of 8 rows
def test_many_partials_over_short_units_stay_whole(q_lens, cached, group, hkv, cut):
    kv_lens = [q + c for q, c in zip(q_lens, cached)]
    split = _plan(q_lens, kv_lens, group, hkv, 1)[2]
    assert (split.num_parts > 0) == cut, split.num_parts


def _check(gpu, q_lens, kv_lens, group, hkv, seed, causal, hide=()):
    q, kc, vc, qo, kvi, idx, lpl = _case(q_lens, kv_lens, group * hkv, hkv, seed, device=gpu)
    idx = idx.copy()
    for b, page, value in hide:   # the blocks hold NaN, no page reads them
        p = kvi[b] + page
        kc[idx[p]] = vc[idx[p]] = float("nan")
        idx[p] = value if value < 0 else kc.shape[0] + value
    for b, n in enumerate(lpl):   # rows past the end
        if kvi[b + 1] > kvi[b] and idx[kvi[b + 1] - 1] >= 0:
            kc[idx[kvi[b + 1] - 1], n:] = vc[idx[kvi[b + 1] - 1], n:] = float("nan")
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(WS, dtype=torch.uint8, device=gpu))
    w.plan(*(torch.from_numpy(x) for x in (qo, kvi, idx, lpl)), num_qo_heads=group * hkv,
           num_kv_heads=hkv, head_dim_qk=128, page_size=16, causal=causal)
    assert w._sched.split.num_parts > 0
    caches = (kc.to(gpu), vc.to(gpu))
    ref, ref_lse = orc.paged_prefill(u16(q), u16(kc), u16(vc), qo, kvi, idx, lpl, causal=causal)
    fin = np.isfinite(ref_lse)

    def check(out, lse):
        assert_attn_close(out.float().cpu().numpy(), ref)
        got = lse.cpu().numpy()
        assert np.array_equal(np.isneginf(got), ~fin)
        assert np.abs(got[fin] - ref_lse[fin]).max() < LSE_TOL

    total = int(qo[-1])
    buf = torch.full((total + 2, group * hkv, 128), 7.0, dtype=torch.bfloat16, device=gpu)
    lse = torch.full((total + 2, group * hkv), 7.0, device=gpu)
    for _ in range(2):
        w.run(q, caches, out=buf, lse=lse)
        check(buf[:total], lse[:total])
    assert (buf[total:] == 7).all() and (lse[total:] == 7).all()
    first = buf[:total].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    out2 = torch.empty_like(first)
    w.run(q, caches, out=out2, stream=side)
    side.synchronize()
    assert torch.equal(out2, first)
    return w, q, caches, check


@pytest.mark.gpu
@pytest.mark.parametrize("group,hkv", [(1, 4), (2, 2), (4, 2), (8, 1)])
@pytest.mark.parametrize("causal", [True, False])
def test_split_units_match_the_oracle(gpu, group, hkv, causal):
    """Chunks over long caches, a single-shot prefill (whose last pieces some
    rows of a tile see nothing of), a short and an empty request."""
    _check(gpu, [37, 0, 1300, 5, 1], [2500, 30, 1300, 40, 1025], group, hkv, 60 + group, causal)


@pytest.mark.gpu
def test_split_units_with_missing_pages(gpu):
    """Missing pages inside a piece, and all pages of whole pieces; a request
    whose pages are all missing (0 / -inf)."""
    hide = [(0, 9, -1), (0, 70, 5)] + [(1, p, -1) for p in range(40, 75)]
    hide += [(2, p, -1) for p in range(70)]
    _check(gpu, [33, 64, 20], [2000, 1600, 1120], 4, 2, 70, True, hide)


@pytest.mark.gpu
def test_without_workspace_the_whole_units_run(gpu):
    """No workspace, or one that is too small: the plan of whole units."""
    q_lens, kv_lens = [37, 70], [2500, 1100]
    w, q, (kc, vc), check = _check(gpu, q_lens, kv_lens, 4, 2, 80, True)
    need = w._sched.split.workspace_bytes
    ws = torch.empty(need, dtype=torch.uint8, device=gpu)
    for ptr, nbytes in ((None, 0), (None, need), (ws.data_ptr(), need - 1)):
        out = torch.empty_like(q)
        lse = torch.empty(sum(q_lens), 8, device=gpu)
        _lib.call("kvc_batch_prefill_split_run", w._sched, w._sched.split,
                  w._plan_dev.data_ptr(), ptr, nbytes, q.data_ptr(), q.stride(0), kc.data_ptr(),
                  vc.data_ptr(), kc.stride(0), kc.stride(1), kc.shape[0], w._indices.data_ptr(),
                  w._indices.numel(), w._sm_scale, out.data_ptr(), out.stride(0), lse.data_ptr(),
                  _lib.current_stream_handle(torch.device(gpu)))
        torch.cuda.synchronize()
        check(out, lse)


@pytest.mark.gpu
@pytest.mark.parametrize("kv_len,group,parts", [(30000, 8, 117), (17100, 4, 67), (20000, 2, 78)])
def test_merge_of_more_partials_than_lanes(gpu, kv_len, group, parts):
    """One chunk over a long history: the merge's maximum takes a second pass over
    the partials, its fold many, with a remainder of a batch of eight."""
    w, *_ = _check(gpu, [40], [kv_len], group, 1, 90 + group, True)
    s = w._sched.split
    merges = w._plan_dev[s.merges_offset:s.merges_offset + 8 * s.num_merges].cpu().view(-1, 8)
    assert int(merges[:, 4].max()) == parts
