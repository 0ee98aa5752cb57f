"""The decode plan's grid, on the CPU: a round of workgroups fits the CUs whatever
the head count, the plan past the 128-page cap is whole rounds, and which batches
get the narrow form's segments (a wave per head and segment)."""
import numpy as np
import pytest

from test_abi import _check_plan_image, _plan, lib  # noqa: F401


def _workgroups(sched):
    group = sched.num_qo_heads // sched.num_kv_heads
    q_splits = 2 if sched.head_dim == 256 and group == 8 else 1   # served as two workgroups of four
    return sched.num_segments * sched.num_head_groups * q_splits


@pytest.mark.parametrize("d,group", [(64, 1), (64, 8), (128, 4), (128, 8), (256, 4), (256, 8)])
@pytest.mark.parametrize("cus", [256, 100])
def test_one_round_of_workgroups_fits_the_cus(lib, d, group, cus):  # noqa: F811
    lens = np.random.default_rng(3).integers(500, 3000, 32).tolist()
    for hkv in range(1, 17):
        indptr, sched, img, lpl = _plan(lib, lens, hq=hkv * group, hkv=hkv, d=d, cus=cus, hint=-1)
        pages = int(indptr[-1])
        if sched.heads_per_group < 8 and pages <= 128 * (cus // sched.num_head_groups // 2):
            assert cus // 2 < _workgroups(sched) <= cus, (hkv, sched.num_segments)
        _check_plan_image(indptr, sched, img, lpl)


def test_rounds_past_the_page_cap(lib):  # noqa: F811
    # 6 KV heads, two per workgroup: 85 segments a round; 20,000 pages need 157
    indptr, sched, img, lpl = _plan(lib, [16 * 10000] * 2, hq=24, hkv=6, d=64, hint=-1)
    assert sched.heads_per_group == 2 and sched.num_segments == 170
    _check_plan_image(indptr, sched, img, lpl)
    # more head groups than CUs: one segment each at least
    indptr, sched, img, lpl = _plan(lib, [300] * 4, hq=7, hkv=7, d=64, cus=4, hint=-1)
    assert sched.num_segments == 1 and sched.num_head_groups == 7
    _check_plan_image(indptr, sched, img, lpl)


MANY = [20 + 7 * i % 280 for i in range(700)]


@pytest.mark.parametrize("hkv,group,d,want", [
    (1, 4, 128, 2048), (2, 4, 128, 1024), (3, 4, 128, 682), (4, 1, 128, 512), (8, 8, 128, 256),
    (8, 1, 64, 512), (8, 4, 64, 384), (8, 8, 64, 384), (6, 1, 64, 682), (1, 1, 64, 2048),
    (8, 4, 128, 256),                      # the LDS kernel's layout and count: its own plan
    (8, 4, 256, 128), (2, 8, 256, 128)])   # head_dim 256: its waves share a segment
def test_many_requests_get_a_segment_per_wave(lib, hkv, group, d, want):  # noqa: F811
    indptr, sched, img, lpl = _plan(lib, MANY, hq=hkv * group, hkv=hkv, d=d)
    assert sched.num_segments == want
    assert sched.plan_ints <= lib.kvc_decode_plan_ints(len(MANY), 8 * 256)
    _check_plan_image(indptr, sched, img, lpl)
    fewer = _plan(lib, MANY, hq=hkv * group, hkv=hkv, d=d, hint=-1)[1]
    assert fewer.num_segments <= sched.num_segments
    assert fewer.workspace_bytes <= sched.workspace_bytes


def test_narrow_segments_stay_within_a_request_and_the_partials(lib):  # noqa: F811
    # few requests over many waves: more than 16 segments each
    assert _plan(lib, [3000] * 30, hq=4, hkv=1)[1].num_segments == 256
    assert _plan(lib, [3000] * 130, hq=4, hkv=1)[1].num_segments == 2048
    # a 30,000-token request beside 200 short ones: its 1,290 narrow pieces would
    # need 4 x the partials of the allocation-free run's array
    lens = [40] * 200 + [30000]
    sched = _plan(lib, lens, hq=4, hkv=1)[1]
    assert sched.num_segments == 256
    assert sched.workspace_bytes <= 200 * 2 ** 20
    # short requests: one segment each where they fill the waves
    for n, want in ((1024, 1024), (256, 256), (500, 500)):
        s = _plan(lib, [20 + i % 12 for i in range(n)], hq=32, hkv=8, d=64)[1]
        assert s.num_segments == want and s.max_partitions == 1


@pytest.mark.parametrize("seed", range(4))
def test_random_plans_of_every_layout(lib, seed):  # noqa: F811
    rng = np.random.default_rng(seed)
    for _ in range(60):
        hi = int(rng.choice([20, 60, 300, 2000]))
        lens = rng.integers(0, hi + 1, int(rng.integers(1, 600))).tolist()
        hkv, group = int(rng.integers(1, 17)), int(rng.choice([1, 2, 4, 8]))
        d = int(rng.choice([64, 128, 256]))
        cus = int(rng.choice([256, 256, 64, 10]))
        indptr, sched, img, lpl = _plan(lib, lens, hq=hkv * group, hkv=hkv, d=d, cus=cus)
        if indptr[-1] == 0:
            continue
        S = sched.num_segments
        one_each = S + sched.num_empty == len(lens) and sched.max_partitions == 1
        if not one_each:
            _check_plan_image(indptr, sched, img, lpl)
        assert sched.num_head_groups * sched.heads_per_group == hkv
        few = _plan(lib, lens, hq=hkv * group, hkv=hkv, d=d, cus=cus, hint=-1)[1]
        assert sched.workspace_bytes <= max(16 << 20, few.workspace_bytes)


def test_narrow_segments_leave_few_waves_out(lib):  # noqa: F811
    # 20 requests, at most 16 segments each: 320 of the 384 that the chip has waves for
    lens = [1100 + 500 * i for i in range(20)]
    for group, want in ((2, 128), (4, 128), (8, 320)):
        assert _plan(lib, lens, hq=8 * group, hkv=8, d=64)[1].num_segments == want
    assert _plan(lib, lens * 2, hq=32, hkv=8, d=64)[1].num_segments == 384
