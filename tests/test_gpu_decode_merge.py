"""The split-K merge around the piece counts where its kernels change: one wave
up to 16 pieces per request, four waves above, folding 64 pieces at a time; at
every head_dim, with single-piece and empty requests beside the split one."""
import numpy as np
import pytest

from helpers import assert_attn_close, u16
from oracle import kv_oracle as orc
from test_gpu_decode import _paged, _run, randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("parts", [16, 17, 20, 64, 65, 130])
def test_merge_piece_counts(gpu, parts, d):
    # one page per segment: the first request is cut into `parts` pieces
    lens = [16 * parts - 5, 0, 7, 40]
    pages = sum((n + 15) // 16 for n in lens)
    hkv, hq = 2, 8
    kc, vc, bt, indptr, indices, lpl = _paged(lens, hkv, d, 300 + parts)
    q = randn_bf16((len(lens), hq, d), 301, device=gpu)
    (out, lse), w = _run(gpu, q, kc.to(gpu), vc.to(gpu), indptr, indices, lpl, hq, hkv, d,
                         segs=pages)
    assert w.schedule.max_partitions == parts
    ref, ref_lse = orc.paged_decode(u16(q), u16(kc), u16(vc), indptr, indices, lpl)
    assert_attn_close(out.float().cpu().numpy(), ref)
    got = lse.cpu().numpy()
    fin = np.isfinite(ref_lse)
    assert np.array_equal(np.isneginf(got), ~fin) and not fin[1].any()
    # natural-log lse: fp32 sums of at most 2,100 terms, about 1e-6 of values near 8
    assert np.abs(got[fin] - ref_lse[fin]).max() < 2e-3
    assert (out[1] == 0).all()
