"""The split-K merge alone, over partials written by the test (a schedule without
segments launches nothing else): the one-wave kernel (16 partials) and the
four-wave one (17 and more) follow one rule, also where a log-sum-exp is NaN or
infinite and where no partial has a key."""
import math

import pytest
import torch

from gpu_offloading_amd import _lib

pytestmark = pytest.mark.gpu


def _merge(gpu, o, lse2):
    """o [parts, d], lse2 [parts] (base 2) of one request and head -> (out, lse)."""
    parts, d = o.shape
    s = _lib.KvcDecodeSchedule(batch=1, num_qo_heads=1, num_kv_heads=1, head_dim=d, page_size=16,
                               num_head_groups=1, heads_per_group=1, max_partitions=parts,
                               nparts_offset=8)
    s.plan_ints = _lib.load().kvc_decode_plan_ints(1, 0)
    plan = torch.zeros(12, dtype=torch.int32, device=gpu)
    plan[8] = parts
    need = _lib.load().kvc_decode_workspace_bytes(1, 1, d, parts)
    ws = torch.zeros(need // 4, device=gpu)
    ws[:parts * d] = o.flatten()
    at = (parts * d * 4 + 255) // 256 * 64
    ws[at:at + parts] = lse2
    q = torch.zeros(1, 1, d, dtype=torch.bfloat16, device=gpu)
    cache = torch.zeros(1, 16, 1, d, dtype=torch.bfloat16, device=gpu)
    out, lse = torch.empty_like(q), torch.empty(1, 1, device=gpu)
    _lib.call("kvc_batch_decode_run", s, plan.data_ptr(), q.data_ptr(), d, cache.data_ptr(),
              cache.data_ptr(), 16 * d, d, 1, None, None, 0, None, 0.1, ws.data_ptr(), need,
              out.data_ptr(), d, lse.data_ptr(), _lib.current_stream_handle(torch.device(gpu)))
    torch.cuda.synchronize()
    return out.float().flatten(), lse.item()


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("parts", [2, 16, 17, 64, 65, 150])
def test_merge_rule(gpu, parts, d):
    g = torch.Generator(device=gpu).manual_seed(parts)
    o = torch.randn(parts, d, generator=g, device=gpu)
    lse2 = 4 * torch.randn(parts, generator=g, device=gpu)
    lse2[parts // 2] = -math.inf                      # a piece without keys
    w = torch.softmax(lse2.double() * math.log(2), 0)
    out, lse = _merge(gpu, o, lse2)
    want = (w[:, None] * o.double()).sum(0)
    assert (out.double() - want).abs().max().item() < 2e-2
    assert abs(lse - torch.logsumexp(lse2.double() * math.log(2), 0).item()) < 1e-4
    # none has a key
    out, lse = _merge(gpu, o, torch.full_like(lse2, -math.inf))
    assert lse == -math.inf and (out == 0).all()
    # a weight that is not a number is not lost
    for bad in (math.nan, math.inf):
        x = lse2.clone()
        x[-1] = bad
        out, lse = _merge(gpu, o, x)
        assert math.isnan(lse) and out.isnan().all(), (bad, lse)
