"""GPU: short passes (rows of up to 64 blocks, up to 2048 blocks in all) take launches of their own for the gather with the pooling and for the
estimate with the selection, scoring passes of short segments sort, and longer passes pool their query blocks in the sort's launch.  Against the stage-by-stage calls, bit for bit, at the edges of the rule and of their tiles."""
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
    # scoring passes that sort, and their neighbours: 768 and 792 segments, segments of two chunks and of four, a partial last segment
    (1, 32, 8, 24 * 128, 128, 0.9, "strong_uniform", {}), (1, 33, 11, 24 * 128, 128, 0.9, "strong_uniform", {}),
    (1, 4, 1, 4096 + 77, 256, "rows", "strong_heavy", {}), (1, 8, 2, 2048, 256, 0.9, "strong_heavy", {}), (2, 3, 3, 300, 128, 0.9, "uniform_heavy", {}),
    (25, 32, 8, 200, 128, 0.9, "strong_uniform", {}),   # 800 heads of one segment: more than run at once, two chunks a head
    # query poolings that ride with the sort: 16384 blocks, the last; one block a head more; segments too long for the sort by waves
    (1, 64, 8, 32768, 1024, 0.9, "strong_heavy", {}), (1, 64, 8, 32769, 1024, 0.9, "strong_heavy", {}),
    (1, 3, 1, 70 * 128 + 5, 2048, 0.9, "strong_uniform", dict(query_pool_mode="max")), (1, 3, 1, 9000, 4096, 0.9, "uniform_heavy", {}),
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


@pytest.mark.parametrize("B,Hq,Hkv,S,seg,one_launch", [
    (1, 32, 8, 77, 256, True), (1, 2, 1, 1, 128, True), (4, 64, 8, 128, 128, True), (1, 257, 257, 100, 256, False),
    (2, 128, 8, 256, 256, True), (2, 129, 3, 256, 256, False), (1, 1, 1, 511 * 128, 65536, False), (1, 4, 4, 300, 256, False),
])
def test_one_launch_entry_point(dev, B, Hq, Hkv, S, seg, one_launch):
    """pbs_one_segment_attn_fwd against pbs_prefill_attn_fwd on the same tensors, and where it hands the call back, without a trace in the output."""
    from pbs_attn_amd import _lib
    lib = _lib.load()
    q, k, v = (x.to(dev) for x in small_case(B, Hq, Hkv, S, seed=S))
    out = torch.full_like(q, 7.0)
    common = (q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), B, Hq, Hkv, S, 128, 128, seg, *q.stride()[:3], *k.stride()[:3],
              *v.stride()[:3], *out.stride()[:3])
    st = torch.cuda.current_stream().cuda_stream
    rc = lib.pbs_one_segment_attn_fwd(*common, 128 ** -0.5, st)
    got = out.clone()
    if not one_launch:
        assert rc == _lib.NOT_ONE_LAUNCH and torch.equal(got, torch.full_like(q, 7.0))
        return
    assert rc == 0
    n = lib.pbs_prefill_attn_workspace_bytes(B, Hq, Hkv, S, 128, 128, seg)
    ws = torch.empty(n, dtype=torch.uint8, device=dev)
    assert lib.pbs_prefill_attn_fwd(*common, 0.9, None, 0, 1, 0, 0, 128 ** -0.5, ws.data_ptr(), n, st) == 0
    assert torch.equal(got, out)
    assert lib.pbs_prefill_attn_fwd(*common, 0.9, None, 0, 1, 0, 0, 128 ** -0.5, None, 0, st) == -1   # refused as before
    assert lib.pbs_one_segment_attn_fwd(*common[:8], 64, *common[9:], 128 ** -0.5, st) == -1
    assert lib.pbs_one_segment_attn_fwd(*common[:10], 200, *common[11:], 128 ** -0.5, st) == -1
