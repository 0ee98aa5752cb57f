"""Short requests in the decode plan, on the CPU: at head_dim 64 and 256 a request
of up to 16 pages is one segment, and needs no merge, unless its workgroup would be
on it for longer than the segments of an idle chip take."""
import numpy as np
import pytest

from test_abi import _check_plan_image, _plan, lib  # noqa: F401


@pytest.mark.parametrize("d,hkv,group,batch,pages,whole", [
    # few requests: whole up to about 16 pages of a head (8 for groups of 8), 6 at head_dim 256
    (64, 8, 1, 1, 5, True), (64, 8, 1, 1, 7, False), (64, 4, 4, 8, 6, True), (64, 4, 4, 8, 7, False),
    (64, 2, 1, 3, 10, True), (64, 2, 1, 3, 11, False), (64, 1, 4, 8, 16, True),
    (64, 8, 8, 3, 4, True), (64, 8, 8, 3, 5, False), (64, 1, 8, 3, 10, True), (64, 1, 8, 3, 11, False),
    (256, 8, 4, 8, 3, True), (256, 8, 4, 8, 4, False), (256, 2, 1, 8, 5, True), (256, 2, 1, 8, 6, False),
    (256, 1, 4, 8, 8, True), (256, 1, 4, 8, 9, False), (256, 4, 1, 8, 16, False),
    # requests that fill the CUs are whole whatever their length
    (64, 16, 4, 64, 16, True), (256, 16, 4, 64, 16, True), (256, 8, 8, 64, 16, True),
    (256, 4, 1, 64, 16, False)])
def test_short_requests_are_cut_where_the_chip_is_idle(lib, d, hkv, group, batch, pages, whole):  # noqa: F811
    lens = [16 * pages - 3] * batch
    hq = hkv * group
    indptr, sched, img, lpl = _plan(lib, lens, hq=hq, hkv=hkv, d=d)
    _check_plan_image(indptr, sched, img, lpl)
    assert (sched.max_partitions == 1) == whole, (sched.num_segments, sched.max_partitions)
    if whole:
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
    indptr, sched, img, lpl = _plan(lib, [0] * 3, hq=8, hkv=8, d=256)
    assert sched.num_segments == 0 and sched.num_pieces == 0


def test_short_requests_stay_whole_where_partials_are_many(lib):  # noqa: F811
    # one of 16 pages beside short ones, 128 rows of 256 floats a piece: 16 pieces
    # each of 4 requests take 8 MiB, 8 of 32 would take 32, above the 16 of the
    # allocation-free run
    few = _plan(lib, [3] * 3 + [250], hq=128, hkv=16, d=256)[1]
    assert few.max_partitions > 4 and 0 < few.workspace_bytes <= 16 << 20
    many = _plan(lib, [3] * 31 + [250], hq=128, hkv=16, d=256)[1]
    assert many.num_segments == 32 and many.max_partitions == 1 and many.workspace_bytes == 0
