"""The decode plan's cuts, on the CPU, against a walk over every page: cut s goes
where the cost before it (8 a page, 9 a switch to another request) is nearest to
s/S of the total, the later of two equally near ones."""
import numpy as np
import pytest

from test_abi import _plan, lib  # noqa: F401


def _cuts(indptr, segs):
    total = int(indptr[-1])
    starts = [int(indptr[b]) for b in range(1, len(indptr) - 1)
              if indptr[b + 1] > indptr[b] and indptr[b] > 0]
    cost = [0]                                   # of pages [0, x)
    begins = set(starts)
    for x in range(total):                       # page x is counted with its start
        cost.append(cost[-1] + 8 + (9 if x in begins else 0))
    cut, x = [0], 0
    for s in range(1, segs):
        target = s * cost[-1] // segs
        while x < total and cost[x] < target:
            x += 1
        pick = x - 1 if x > 0 and target - cost[x - 1] < cost[x] - target else x
        cut.append(min(max(pick, cut[-1] + 1), total - (segs - s)))
    ends = cut[1:] + [total]
    if segs > 1 and max(e - c for c, e in zip(cut, ends)) > 128:
        cut = [s * total // segs for s in range(segs)]
    return cut


@pytest.mark.parametrize("seed", range(6))
def test_cuts_equal_the_walk_over_every_page(lib, seed):  # noqa: F811
    rng = np.random.default_rng(seed)
    for _ in range(40):
        hi = int(rng.choice([10, 40, 300, 3000]))
        lens = rng.integers(0, hi + 1, int(rng.integers(1, 120))).tolist()
        if rng.random() < 0.3:
            lens += [16 * int(rng.integers(100, 2000))]
        indptr, sched, img, _ = _plan(lib, lens, hint=int(rng.choice([1, 2, 7, 64, 333, 1000])))
        if indptr[-1]:
            segs = img[:4 * sched.num_segments].reshape(-1, 4)
            assert segs[:, 2].tolist() == _cuts(indptr, sched.num_segments)
