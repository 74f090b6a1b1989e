"""GPU: short passes (rows of up to 64 blocks, up to 2048 blocks in all) take launches of their own for the gather with the pooling and for the
estimate with the selection.  Against the stage-by-stage calls, bit for bit, at the edges of the rule and of their tiles."""
import pytest
import torch

from pbs_attn_amd import pbs as P
from tests.test_hip_prefill_routes import _single_and_staged
from tests.util import small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,S,seg,thr,kind,kw", [
    (1, 32, 8, 8192, 256, 0.9, "uniform_heavy", {}),                 # 2048 blocks of rows of 64: the last short pass
    (1, 32, 8, 8193, 256, 0.9, "uniform_heavy", {}),                 # one block more in a row
    (1, 33, 11, 62 * 128 + 1, 384, "rows", "strong_uniform", {}),    # 2079 blocks
    (3, 5, 1, 33 * 128 - 3, 128, "rows", "uniform_heavy", dict(query_pool_mode="max", key_pool_mode="max")),   # a second tile of 32 rows, of one row
    (2, 4, 4, 31 * 128, 256, 0.8, "strong_heavy", dict(key_pool_mode="max")),
    (1, 3, 1, 129, 128, 0.9, "uniform_heavy", {}),                   # two blocks, one candidate
    (1, 2, 2, 7 * 128 + 64, 384, 0.0, "local_window", {}),           # rows without candidates are selected too; ragged last block
    (1, 28, 4, 1000, 256, 1.0, "strong_heavy", dict(force_select_first_block=False)),   # sums that may never reach the threshold
])
def test_short_passes(dev, B, Hq, Hkv, S, seg, thr, kind, kw):
    assert torch.equal(*_single_and_staged(dev, B, Hq, Hkv, S, seg, thr, kind, **kw))


def test_short_pass_of_projection_shaped_tensors(dev):
    """(batch, token, head, d) memory, K and V slices of one tensor, rows of 16-byte alignment only."""
    q, k, v = (x.to(dev) for x in small_case(2, 8, 2, 1500, seed=5))
    want = P.permuted_block_sparse_attn_fwd(q, k, v, 128, 256, 0.9, True)
    kv = torch.zeros(2, 1500, 2, 3 * 128 + 8, dtype=torch.bfloat16, device=dev)
    kv[..., 8:136], kv[..., 264:392] = k.transpose(1, 2), v.transpose(1, 2)
    qt = q.transpose(1, 2).contiguous().transpose(1, 2)
    got = P.permuted_block_sparse_attn_fwd(qt, kv[..., 8:136].transpose(1, 2), kv[..., 264:392].transpose(1, 2), 128, 256, 0.9, True)
    assert torch.equal(got, want)
