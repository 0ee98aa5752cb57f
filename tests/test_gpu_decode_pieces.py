"""Pieces of the wave decode kernel inside one segment: pieces of one unit (which
their wave closes alone) between pieces that several waves share, in every order
of the two, for every (group, head_dim) the kernel is built for; and its narrow
form, a wave per head and segment."""
import pytest
import torch

import test_gpu_decode_wave as wave
from gpu_offloading_amd.decode import BatchDecodeWithPagedKVCacheWrapper

pytestmark = pytest.mark.gpu

# 1, 2, 3, ... pages: one unit (of one page, or of two where it starts on an even
# page), units shared by some of the waves, by all of them, more than once round
LENS = [1, 16, 40, 3, 290, 17, 0, 31, 33, 5, 9, 600, 16, 32, 64, 1, 1, 1, 200, 15]


@pytest.mark.parametrize("group,d,hkv", [(1, 64, 4), (2, 64, 2), (4, 64, 1), (8, 64, 4),
                                         (1, 128, 4), (2, 128, 1), (4, 128, 2), (8, 128, 4),
                                         (1, 256, 2), (4, 256, 4), (8, 256, 1)])
@pytest.mark.parametrize("segs", [1, 4])
def test_short_pieces_between_shared_ones(gpu, group, d, hkv, segs):
    sched = wave._check(gpu, LENS, group, d, hkv, segs, 470 + segs)
    assert sched.num_segments == segs and sched.heads_per_group in (1, 2, 4)
    assert sched.num_pieces >= len(LENS) - 1


# With more segments than CUs the kernel runs its narrow form: a wave per head and
# segment, several workgroups a CU.  Segments of one page and of a few, pieces of
# one page to a whole segment, two KV heads and four per workgroup and one.
MANY = LENS * 5


@pytest.mark.parametrize("group,d,hkv", [(1, 64, 4), (2, 64, 2), (4, 64, 3), (8, 64, 4),
                                         (1, 128, 3), (2, 128, 2), (4, 128, 1), (8, 128, 4),
                                         (1, 256, 2), (4, 256, 4), (8, 256, 1)])
@pytest.mark.parametrize("segs", [270, 500])
def test_narrow_form(gpu, group, d, hkv, segs):
    sched = wave._check(gpu, MANY, group, d, hkv, segs, 480 + segs)
    assert sched.num_segments == min(segs, sched.total_pages)
    assert sched.num_segments * sched.num_head_groups > 256


@pytest.mark.parametrize("hkv,group,d", [(1, 1, 64), (4, 4, 64), (2, 8, 64), (2, 4, 128),
                                         (2, 8, 128), (2, 8, 256)])
@pytest.mark.parametrize("offset", [0, 1])
def test_narrow_form_appends(gpu, hkv, group, d, offset):
    lens = [min(n, 90) for n in LENS] * 8
    wave.test_append_in_the_decode_launch(gpu, hkv, group, d, lens, 300, offset)


def test_long_narrow_segments(gpu):
    """96 pages per segment (more ids than lanes), against the form whose waves
    share a segment: both keep sums and weights in fp32, so the bf16 results may
    differ by one rounding (2^-8 of values below 1)."""
    hkv, d, pages = 16, 64, 19200
    g = torch.Generator(device=gpu).manual_seed(5)
    cache = torch.empty(pages, 2, 16, hkv, d, dtype=torch.bfloat16, device=gpu)
    cache.normal_(generator=g)
    q = torch.randn(60, hkv, d, generator=g, device=gpu).to(torch.bfloat16)
    indptr = torch.arange(0, pages + 1, pages // 60, dtype=torch.int32)
    indices = torch.randperm(pages, generator=g, device=gpu).to(torch.int32)
    got = []
    for segs in (200, 150):   # 3200 and 2400 of the chip's 4096 waves
        w = BatchDecodeWithPagedKVCacheWrapper(
            torch.empty(1 << 26, dtype=torch.uint8, device=gpu), num_segments=segs)
        w.plan(indptr, indices, torch.full((60,), 7, dtype=torch.int32), num_qo_heads=hkv,
               num_kv_heads=hkv, head_dim=d, page_size=16)
        assert w.schedule.num_segments == segs and w.schedule.num_head_groups == 4
        out, lse = w.run(q, (cache[:, 0], cache[:, 1]), return_lse=True)
        got.append((out.float(), lse))
    assert (got[0][0] - got[1][0]).abs().max().item() <= 2 ** -8
    assert (got[0][1] - got[1][1]).abs().max().item() < 1e-4
    assert got[0][0].abs().max().item() > 0.05
