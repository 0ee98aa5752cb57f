"""The decode plan's grid, on the CPU: a round of workgroups fits the CUs whatever
the head count, and the plan past the 128-page cap is whole rounds."""
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
        indptr, sched, img, lpl = _plan(lib, lens, hq=hkv * group, hkv=hkv, d=d, cus=cus)
        pages = int(indptr[-1])
        if sched.heads_per_group < 8 and pages <= 128 * (cus // sched.num_head_groups // 2):
            assert cus // 2 < _workgroups(sched) <= cus, (hkv, sched.num_segments)
        _check_plan_image(indptr, sched, img, lpl)


def test_rounds_past_the_page_cap(lib):  # noqa: F811
    # 6 KV heads, two per workgroup: 85 segments a round; 20,000 pages need 157
    indptr, sched, img, lpl = _plan(lib, [16 * 10000] * 2, hq=24, hkv=6, d=64)
    assert sched.heads_per_group == 2 and sched.num_segments == 170
    _check_plan_image(indptr, sched, img, lpl)
    # more head groups than CUs: one segment each at least
    indptr, sched, img, lpl = _plan(lib, [300] * 4, hq=7, hkv=7, d=64, cus=4)
    assert sched.num_segments == 1 and sched.num_head_groups == 7
    _check_plan_image(indptr, sched, img, lpl)
