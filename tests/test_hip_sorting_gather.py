"""GPU: the gather of short passes that sorts its block's segment itself, against the stage-by-stage calls (sort kernel, gather by indices), bit for bit:
segments of each number of keys a lane, at the limits of the rule and of a segment."""
import pytest
import torch

from pbs_attn_amd import pbs as P
from tests.test_hip_prefill_routes import _NullTimer, _single_and_staged
from tests.util import small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,S,seg,thr,kind,kw", [
    (1, 3, 1, 129, 128, 0.9, "uniform_heavy", {}), (1, 5, 5, 3 * 128 + 1, 128, "rows", "strong_uniform", {}),
    (2, 6, 2, 1000, 256, 0.9, "strong_heavy", {}),                                 # a remainder of more than a block, the last one ragged
    (1, 28, 4, 1000, 384, "rows", "uniform_heavy", dict(key_pool_mode="max")),     # three blocks a segment
    (1, 4, 2, 1280, 640, 0.8, "strong_uniform", dict(query_pool_mode="max")),
    (1, 2, 1, 2 * 1024 + 128, 1024, 0.9, "strong_heavy", {}), (1, 2, 2, 2 * 1024, 1024, 0.0, "local_window", {}),
    (1, 2, 1, 3 * 1152 + 1, 1152, 0.9, "uniform_heavy", {}),                       # segments too long for it
    (1, 32, 8, 24 * 128, 512, 0.9, "uniform_heavy", {}), (1, 33, 11, 24 * 128, 512, 0.9, "uniform_heavy", {}),   # 768 blocks, the last; 792
    (8, 8, 2, 1024, 128, 0.9, "strong_uniform", {}), (9, 8, 2, 1024, 128, 0.9, "strong_uniform", {}),   # batches
    (1, 1, 1, 64 * 128, 256, 0.9, "strong_heavy", {}), (1, 32, 8, 64 * 128, 256, "rows", "strong_uniform", {}),   # 64 blocks a row; 2048 blocks, the last
    (1, 33, 11, 64 * 128, 256, "rows", "strong_uniform", {}),                      # no short pass any more
    (1, 255, 51, 300, 128, 0.9, "uniform_heavy", {}), (1, 256, 64, 300, 128, 0.9, "uniform_heavy", {}),   # the most heads of ranked segments; one more
    (1, 4, 1, 6000, 128, 0.9, "strong_heavy", {}), (1, 4, 1, 6000, 256, 0.9, "strong_heavy", {}),         # segments shorter than a scoring chunk; as long as one
])
def test_against_the_stages(dev, B, Hq, Hkv, S, seg, thr, kind, kw):
    assert torch.equal(*_single_and_staged(dev, B, Hq, Hkv, S, seg, thr, kind, **kw))


@pytest.mark.parametrize("seg", [128, 256, 512, 1024])
def test_equal_scores_and_strided_tensors(dev, seg):
    """Keys that repeat have equal scores and keep their order; K and V slices of one tensor."""
    S = 2 * seg + 200
    q, k, v = (x.to(dev) for x in small_case(2, 4, 2, S, seed=seg))
    k = k[:, :, torch.arange(S, device=dev) % 7].contiguous()
    k[:, :, seg // 2] = 0
    outs = []
    kv = torch.zeros(2, S, 2, 3 * 128 + 8, dtype=torch.bfloat16, device=dev)
    kv[..., 8:136], kv[..., 264:392] = k.transpose(1, 2), v.transpose(1, 2)
    outs.append(P.permuted_block_sparse_attn_fwd(q, k, v, 128, seg, 0.7, True))
    outs.append(P.permuted_block_sparse_attn_fwd(q, kv[..., 8:136].transpose(1, 2), kv[..., 264:392].transpose(1, 2), 128, seg, 0.7, True))
    P.stage_timer = _NullTimer()
    try:
        staged = P.permuted_block_sparse_attn_fwd(q, k, v, 128, seg, 0.7, True)
    finally:
        P.stage_timer = None
    assert all(torch.equal(o, staged) for o in outs)


@pytest.mark.parametrize("S,seg,value", [(300, 128, float("nan")), (700, 256, float("inf")), (1300, 512, float("nan"))])
def test_scores_that_are_not_finite(dev, S, seg, value):
    """Every score of a row is NaN once one of its logits is: keys keep their order."""
    q, k, v = (x.to(dev) for x in small_case(1, 4, 2, S, seed=seg))
    k[:, 0, seg // 3] = value
    single = P.permuted_block_sparse_attn_fwd(q, k, v, 128, seg, 0.9, True)
    P.stage_timer = _NullTimer()
    try:
        staged = P.permuted_block_sparse_attn_fwd(q, k, v, 128, seg, 0.9, True)
    finally:
        P.stage_timer = None
    nan = torch.isnan(single)
    assert torch.equal(nan, torch.isnan(staged)) and torch.equal(single[~nan], staged[~nan])
