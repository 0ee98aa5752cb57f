"""One softmax state per row of 16 lanes in the wave decode kernel.  The lanes
of a row sum the q.k products of a score's chunks in an order of their own; were
the sums not the same bits in all of them, a score within rounding of the lazy
rescale's threshold would leave some output dims under another maximum than the
sum of weights they are divided by.  Here a score's chunks are 2^27, -2^27 and
62, whose fp32 sum is 62 or 64 depending on the order, and the threshold (a
growth of 2^8 over the maximum 0 of the wave's first page) lies between
62 / sqrt(128) log2(e) = 7.9 and 64 / sqrt(128) log2(e) = 8.2."""
import math

import numpy as np
import pytest
import torch

from gpu_offloading_amd.decode import BatchDecodeWithPagedKVCacheWrapper

pytestmark = pytest.mark.gpu

PAGES = 40   # more than two units of pages for every wave (at most 16 waves of 2 pages)


@pytest.mark.parametrize("group", [1, 4, 8])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_every_dim_has_its_rows_softmax_state(gpu, d, group):
    q = torch.zeros(1, group, d, device=gpu)
    q[..., 0] = q[..., 8] = 2.0 ** 13
    q[..., 16] = 1.0
    q = q.to(torch.bfloat16)
    kc = torch.zeros(PAGES, 16, 1, d, dtype=torch.bfloat16, device=gpu)
    vc = torch.ones_like(kc)
    w = BatchDecodeWithPagedKVCacheWrapper(torch.empty(1 << 24, dtype=torch.uint8, device=gpu),
                                           num_segments=1)
    scale = 1.0 / math.sqrt(128)
    w.plan(torch.tensor([0, PAGES], dtype=torch.int32),
           torch.arange(PAGES, dtype=torch.int32, device=gpu),
           torch.tensor([16], dtype=torch.int32), num_qo_heads=group, num_kv_heads=1, head_dim=d,
           page_size=16, sm_scale=scale)
    assert w.schedule.small_batch == 0 and w.schedule.heads_per_group == 1
    # The output for a score s: one value 2 of weight e^s among n - 1 of 1.
    n = 16 * PAGES
    low, high = ((n - 1 + 2 * math.exp(s * scale)) / (n - 1 + math.exp(s * scale))
                 for s in (62 - 4, 62 + 4))   # an fp32 sum at 2^27 rounds by up to 4
    for page in range(PAGES):   # the wave's second unit among them, whatever its size
        kc[page, 0, 0, 0], kc[page, 0, 0, 8], kc[page, 0, 0, 16] = 2.0 ** 14, -2.0 ** 14, 62.0
        vc[page, 0] = 2.0
        out = w.run(q, (kc, vc)).float().cpu().numpy()[0]
        kc[page] = 0.0
        vc[page] = 1.0
        # V has the same value in every dim, so the dims' sums are the same bits
        assert float(np.ptp(out, axis=1).max()) == 0.0, (page, out[0, ::16])
        assert out.min() > low - 2e-2 and out.max() < high + 2e-2, (page, out[0, 0])
