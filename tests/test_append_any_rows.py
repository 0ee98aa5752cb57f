"""A decode step's new rows off a 16-byte boundary: batches that the fused append
does not serve (by the LDS kernel's count of request ends per segment, whichever
kernel could stream them) take them through the two calls."""
import pytest
import torch

from gpu_offloading_amd.kv_cache import PagedKVCache
from test_abi import _plan, lib  # noqa: F401

# (KV heads, group, lengths before the step)
ONES = [3] * 40 + [1590] * 30       # six request ends in a segment of the LDS kernel
PAIRS = [30] * 512                  # two pages each, no segment cuts one


def test_which_batches_the_fused_append_serves(lib):  # noqa: F811
    s = _plan(lib, [n + 1 for n in ONES], hq=32, hkv=8)[1]
    assert s.heads_per_group == 8 and s.append_pieces == 6
    # few ends per segment: the wave kernel, with the append of the LDS kernel's batches
    s = _plan(lib, [61] * 40 + [1591] * 28, hq=32, hkv=8)[1]
    assert s.heads_per_group == 4 and s.num_segments == 256
    assert _plan(lib, [n + 1 for n in PAIRS], hq=16, hkv=4)[1].small_batch == 0
    assert _plan(lib, [n + 1 for n in PAIRS[1:]], hq=16, hkv=4)[1].small_batch == 1


@pytest.mark.gpu
@pytest.mark.parametrize("hkv,group,lens", [(8, 4, ONES), (4, 4, PAIRS), (1, 1, PAIRS * 4)])
def test_rows_of_any_alignment_without_the_fused_append(gpu, hkv, group, lens):
    n, hq = len(lens), hkv * group
    total = sum((x + 16) // 16 for x in lens)
    c = PagedKVCache(1, hkv, 128, max_seqs=n, max_seq_len=1700, num_qo_heads=hq,
                     kv_page_budget=total, device=gpu, workspace_bytes=1 << 26,
                     staging_bytes=1 << 20)
    for s, x in enumerate(lens):
        c.ensure_pages(s, (x + 16) // 16)
    c.advance(list(range(n)), lens)
    g = torch.Generator(device=gpu).manual_seed(8)
    c.fill_kv_random(1.0, generator=g)
    c.prepare_decode_step(list(range(n)))
    w = c._decode_wrapper
    assert not w.fused_append_supported
    buf = torch.randn(2, n * hkv * 128 + 8, generator=g, device=gpu).to(torch.bfloat16)
    q = torch.randn(n, hq, 128, generator=g, device=gpu).to(torch.bfloat16)
    rows = [b[:n * hkv * 128].clone().view(n, hkv, 128) for b in buf]
    with pytest.raises(RuntimeError, match="fused append needs"):
        w.run_with_append(q, (c.k_cache[0], c.v_cache[0]), *rows)
    want = c.append_and_decode(0, *rows, q)
    cache = c.kv_cache[0].clone()
    for offset in (1, 2):   # elements: off any 4-byte boundary, on one
        buf[:, offset:offset + n * hkv * 128] = torch.stack([r.flatten() for r in rows])
        odd = [b[offset:offset + n * hkv * 128].view(n, hkv, 128) for b in buf]
        got = c.append_and_decode(0, *odd, q)
        assert torch.equal(got, want) and torch.equal(c.kv_cache[0], cache)
