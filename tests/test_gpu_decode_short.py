"""Short requests on the GPU, as the plan takes them: one segment each, with 1, 2 or
4 heads per workgroup (head_dim 64 and 256), or many of a length (head_dim 128)."""
import pytest

import test_gpu_decode_wave as wave

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group,d,hkv,batch,heads", [
    (1, 64, 8, 3, 1), (2, 64, 6, 43, 2), (4, 64, 4, 70, 2), (8, 64, 8, 33, 2), (8, 64, 2, 5, 1), (4, 64, 16, 20, 2),
    (1, 64, 8, 100, 4), (4, 256, 2, 4, 1), (8, 256, 4, 20, 1), (2, 256, 8, 128, 4), (4, 256, 8, 64, 2)])
def test_heads_per_workgroup(gpu, group, d, hkv, batch, heads):
    lens = [17 + 97 * i % 240 for i in range(batch)]
    sched = wave._check(gpu, lens, group, d, hkv, None, 610 + batch)
    assert sched.num_segments == batch and sched.max_partitions == 1
    assert sched.heads_per_group == heads


@pytest.mark.parametrize("group,hkv,batch,n", [(8, 24, 43, 180), (4, 6, 342, 26), (1, 12, 171, 66), (8, 1, 1024, 40)])
def test_many_alike(gpu, group, hkv, batch, n):
    sched = wave._check(gpu, [n] * batch, group, 128, hkv, None, 630 + hkv)
    assert sched.num_segments == batch and sched.max_partitions == 1
