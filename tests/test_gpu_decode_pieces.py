"""Pieces of the wave decode kernel inside one segment: pieces of one unit (which
their wave closes alone) between pieces that several waves share, in every order
of the two, for every (group, head_dim) the kernel is built for."""
import pytest

from test_gpu_decode_wave import _check

pytestmark = pytest.mark.gpu

# 1, 2, 3, ... pages: one unit (of one page, or of two where it starts on an even
# page), units shared by some of the waves, by all of them, more than once round
LENS = [1, 16, 40, 3, 290, 17, 0, 31, 33, 5, 9, 600, 16, 32, 64, 1, 1, 1, 200, 15]


@pytest.mark.parametrize("group,d,hkv", [(1, 64, 4), (2, 64, 2), (4, 64, 1), (8, 64, 4),
                                         (1, 128, 4), (2, 128, 1), (4, 128, 2), (8, 128, 4),
                                         (1, 256, 2), (4, 256, 4), (8, 256, 1)])
@pytest.mark.parametrize("segs", [1, 4])
def test_short_pieces_between_shared_ones(gpu, group, d, hkv, segs):
    sched = _check(gpu, LENS, group, d, hkv, segs, 470 + segs)
    assert sched.num_segments == segs and sched.heads_per_group in (1, 2, 4)
    assert sched.num_pieces >= len(LENS) - 1
