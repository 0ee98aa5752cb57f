"""Short requests in the decode plan, on the CPU: a request of up to 16 pages is one
segment, and needs no merge, with fewer heads per workgroup where CUs would be left
over; at head_dim 256 unless its workgroup would be on it for longer than the
segments of an idle chip take."""
import pytest

from test_abi import _check_plan_image, _plan, lib  # noqa: F401


@pytest.mark.parametrize("d,hkv,group,batch,pages,heads", [
    # head_dim 64: whole, as few heads per workgroup as still fill one round
    (64, 8, 1, 1, 16, 1), (64, 8, 4, 32, 16, 1), (64, 8, 4, 33, 16, 2), (64, 8, 8, 64, 16, 2),
    (64, 8, 1, 65, 16, 4), (64, 2, 1, 3, 7, 1), (64, 4, 1, 3, 6, 2), (64, 6, 2, 42, 9, 1), (64, 6, 2, 43, 9, 2), (64, 3, 4, 8, 16, 1),
    # head_dim 256: whole up to 8, 12, 16 pages of a head on an idle chip (0: cut)
    (256, 8, 1, 8, 8, 1), (256, 8, 1, 8, 9, 0), (256, 1, 2, 8, 12, 1), (256, 1, 2, 8, 13, 0),
    (256, 4, 4, 8, 16, 1), (256, 4, 8, 8, 16, 1), (256, 4, 8, 32, 16, 1), (256, 4, 8, 33, 11, 2),
    # requests that fill the CUs are whole whatever their length
    (64, 16, 4, 64, 16, 4), (256, 16, 4, 64, 16, 4), (256, 8, 8, 64, 16, 4)])
def test_short_requests_are_whole(lib, d, hkv, group, batch, pages, heads):  # noqa: F811
    lens = [16 * pages - 3] * batch
    hq = hkv * group
    whole = heads > 0
    indptr, sched, img, lpl = _plan(lib, lens, hq=hq, hkv=hkv, d=d)
    _check_plan_image(indptr, sched, img, lpl)
    assert (sched.max_partitions == 1) == whole, (sched.num_segments, sched.max_partitions)
    if whole:
        assert sched.heads_per_group == heads
        assert sched.num_segments == batch and sched.workspace_bytes == 0
    # without partials the requests are never cut
    none = _plan(lib, lens, hq=hq, hkv=hkv, d=d, hint=-1)
    _check_plan_image(none[0], none[1], none[2], none[3])
    assert none[1].max_partitions == 1 and none[1].workspace_bytes == 0


def test_short_requests_beside_empty_ones(lib):  # noqa: F811
    lens = [0, 90, 0, 250, 17, 0]
    indptr, sched, img, lpl = _plan(lib, lens, hq=8, hkv=8, d=256)
    _check_plan_image(indptr, sched, img, lpl)
    assert sched.num_empty == 3 and sched.max_partitions == 16
    indptr, sched, img, lpl = _plan(lib, lens, hq=32, hkv=8, d=256)
    assert sched.num_empty == 3 and sched.num_segments == 3 and sched.max_partitions == 1
    indptr, sched, img, lpl = _plan(lib, [0] * 3, hq=8, hkv=8, d=256)
    assert sched.num_segments == 0 and sched.num_pieces == 0


def test_short_requests_stay_whole_where_partials_are_many(lib):  # noqa: F811
    # one of 16 pages beside short ones, 128 rows of 256 floats a piece: 12 pieces or more
    # of each of 4 requests take 8 MiB at most, 5 of 32 would take 20, above the 16 of the
    # allocation-free run
    few = _plan(lib, [3] * 3 + [250], hq=128, hkv=64, d=256)[1]
    assert few.max_partitions > 4 and 0 < few.workspace_bytes <= 16 << 20
    many = _plan(lib, [3] * 31 + [250], hq=128, hkv=64, d=256)[1]
    assert many.num_segments == 32 and many.max_partitions == 1 and many.workspace_bytes == 0


@pytest.mark.parametrize("hkv,group,batch,n", [
    (24, 8, 344, 26), (6, 4, 342, 180), (12, 1, 684, 66), (1, 8, 1024, 66), (4, 8, 256, 180), (3, 2, 683, 256)])
def test_many_alike_at_head_dim_128(lib, hkv, group, batch, n):  # noqa: F811
    # lined up with the fine segments, so not for the kernel of one workgroup per
    # request: no segment of the wave kernel cuts one, either
    indptr, sched, img, lpl = _plan(lib, [n] * batch, hq=hkv * group, hkv=hkv, d=128)
    _check_plan_image(indptr, sched, img, lpl)
    assert sched.small_batch == 0 and sched.num_segments == batch
    assert sched.max_partitions == 1 and sched.workspace_bytes == 0
