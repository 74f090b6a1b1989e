"""GPU: the routes of the single-call path (pbs_prefill_attn_fwd) against the stage-by-stage calls, bit for bit: the same
tiles in the same order, whatever kernel wrote the visit lists.  Shapes at the edges of the routes."""
import numpy as np
import pytest
import torch

from pbs_attn_amd import pbs as P
from tests.util import blocks_of_an_item, small_case

pytestmark = pytest.mark.gpu


class _NullTimer:
    def mark(self, name):
        pass


def _single_and_staged(dev, B, Hq, Hkv, S, seg, thr, kind="uniform_heavy", **kw):
    q, k, v = (x.to(dev) for x in small_case(B, Hq, Hkv, S, kind=kind, seed=S + seg))
    if thr == "rows":
        thr = torch.linspace(0.5, 0.95, B * Hq).view(B, Hq).to(dev)
    single = P.permuted_block_sparse_attn_fwd(q, k, v, 128, seg, thr, True, **kw)
    P.stage_timer = _NullTimer()
    try:
        staged = P.permuted_block_sparse_attn_fwd(q, k, v, 128, seg, thr, True, **kw)
    finally:
        P.stage_timer = None
    return single, staged


@pytest.mark.parametrize("B,Hq,Hkv,S,seg,thr", [
    (1, 2, 1, 1, 128, 0.9), (2, 3, 1, 128, 128, 0.9), (1, 4, 2, 129, 256, 0.9), (1, 2, 2, 255, 1024, 1),
    (1, 1, 1, 511 * 128, 65536, 0.9),      # the longest sequence that is one segment of the kernel's own size
    (1, 1, 1, 511 * 128 + 1, 65536, 0.9),  # one segment, handled as segments of 256 blocks
    (1, 2, 1, 1000, 384, 1), (2, 2, 2, 1536, 256, 1),   # everything selected: lists without a selection
])
def test_routes_without_a_selection(dev, B, Hq, Hkv, S, seg, thr):
    assert torch.equal(*_single_and_staged(dev, B, Hq, Hkv, S, seg, thr))


@pytest.mark.parametrize("B,Hq,Hkv,S,scale", [
    (1, 32, 8, 77, 1), (3, 5, 5, 700, 1), (1, 28, 4, 1000, 1), (1, 32, 8, 2048, 1),   # an item or less per workgroup
    (1, 33, 3, 2048, 1), (1, 64, 8, 1100, 1),                                         # more items: the list kernel
    (1, 4, 2, 900, 20), (1, 2, 1, 2048, 20),   # exponents that overflow: the item is repeated from the same list
    (3, 16, 4, 1100, 20), (8, 16, 4, 900, 20),   # the same in pairs of query blocks: 240 items, 512 (the list kernel)
])
def test_one_segment_with_lists_formed_by_the_attention_kernel(dev, B, Hq, Hkv, S, scale):
    q, k, v = (x.to(dev) for x in small_case(B, Hq, Hkv, S, seed=S))
    q, k = q * scale, k * scale
    if scale > 1:
        assert blocks_of_an_item(dev, B * Hq, S, (S + 127) // 128 * 128) == (1 if B == 1 else 2)
    single = P.permuted_block_sparse_attn_fwd(q, k, v, 128, 2048, 0.9, True)
    P.stage_timer = _NullTimer()
    try:
        staged = P.permuted_block_sparse_attn_fwd(q, k, v, 128, 2048, 0.9, True)
    finally:
        P.stage_timer = None
    assert torch.isfinite(single.float()).all()
    assert torch.equal(single, staged)


@pytest.mark.parametrize("B,Hq,Hkv,S,seg,thr,kind,kw", [
    (2, 3, 1, 1111, 384, 0.8, "uniform_heavy", dict(query_pool_mode="max", key_pool_mode="max")),   # odd blocks per segment, pairs across segments
    (1, 4, 2, 257, 256, 0.9, "uniform_heavy", {}),                  # one complete segment, the last pair a single row
    (1, 5, 5, 130 * 128 + 1, 128, "rows", "strong_uniform", {}),    # groups of 64 / 128 / 256 candidates that end inside a pair
    (1, 2, 1, 66 * 128, 128, 1.0, "strong_heavy", dict(force_select_first_block=False)),   # sums that may never reach the threshold
    (1, 2, 2, 9000, 512, 0.0, "uniform_heavy", {}),                 # rows without candidates are flagged too
    (1, 2, 1, 1024 * 128, 1024, 0.9, "strong_heavy", {}),           # 1024 blocks: the longest rows of the short kernel
    (1, 1, 1, 1025 * 128 + 7, 384, 0.9, "strong_uniform", {}),      # beyond: lists against the block-level sort
    (1, 1, 1, 2048 * 128, 128, 0.95, "uniform_heavy", {}),          # the longest rows of the list-writing selection
    (1, 1, 1, 2048 * 128 + 1, 2048, 0.3, "uniform_heavy", {}),      # one block more: CSR rows and a merge
])
def test_selection_into_pair_lists(dev, B, Hq, Hkv, S, seg, thr, kind, kw):
    assert torch.equal(*_single_and_staged(dev, B, Hq, Hkv, S, seg, thr, kind, **kw))


@pytest.mark.parametrize("seg", [1, 2, 7, 100, 128, 130, 256, 384, 512, 1000, 1024, 1025, 2048, 2049])
def test_segment_sort_is_stable_for_every_score(dev, seg):
    """One wave per segment up to 2048 keys, a workgroup beyond: against a stable sort of the same scores, with ties, both
    zeros, infinities, subnormals and NaN (which counts as the largest), a partial last segment and block padding."""
    from pbs_attn_amd import ops
    nseg, rows = 3, 5
    S = nseg * seg + seg // 2
    g = torch.Generator().manual_seed(seg)
    x = torch.randn((1, rows, nseg * seg), generator=g)
    x[:, 1] = x[:, 1].round()                                   # many ties
    x[:, 2] = torch.rand((nseg * seg,), generator=g) * 1e-38    # subnormal and tiny
    special = torch.tensor([0.0, -0.0, float("inf"), float("-inf"), float("nan"), 1e-45, -1e-45, 3.4e38])
    x[:, 3] = special[torch.randint(0, 8, (nseg * seg,), generator=g)]
    x[:, 4] = 0.0
    idx = ops.segment_argsort(x.to(dev), S, seg, 128).cpu().long()
    s_pad = (S + 127) // 128 * 128
    v = x.view(rows, nseg, seg).double().numpy()
    nan = np.isnan(v)
    order = np.lexsort((np.broadcast_to(np.arange(seg), v.shape), -np.where(nan, 0.0, v), ~nan), axis=-1)
    want = torch.from_numpy(order + np.arange(nseg)[:, None] * seg).view(1, rows, nseg * seg)
    tail = torch.arange(nseg * seg, s_pad).expand(1, rows, -1)
    assert torch.equal(idx, torch.cat((want, tail), -1))


def test_segment_sort_of_more_work_items_than_one_grid_dimension_holds(dev):
    """65535 rows x 1088 units (1025 segments of two keys, 63 pieces of the identity tail) are 2^26 waves of 64 and more."""
    from pbs_attn_amd import ops
    rows, S, seg = 65535, 2050, 2
    x = torch.rand((1, rows, S), device=dev)
    idx = ops.segment_argsort(x, S, seg, 128)[0]
    pairs = x.view(rows, S // 2, 2)
    second_first = (pairs[..., 1] > pairs[..., 0]).int()
    base = torch.arange(0, S, 2, device=dev, dtype=torch.int32)
    assert torch.equal(idx[:, :S:2], base + second_first)
    assert torch.equal(idx[:, 1:S:2], base + 1 - second_first)
    assert torch.equal(idx[:, S:], torch.arange(S, idx.shape[1], device=dev, dtype=torch.int32).expand(rows, -1))


@pytest.mark.parametrize("B,Hq,Hkv,S,seg", [
    (1, 1, 1, 130, 128), (2, 7, 1, 1000, 128), (1, 4, 1, 2048, 128), (1, 4, 1, 2190, 128),   # 2 .. 32 chunks of 64, 17 of 128 keys
    (1, 12, 3, 16384, 128), (1, 12, 3, 16512, 128),   # the longest sequence of the split scoring, and one block more
    (25, 32, 8, 200, 128), (12, 64, 8, 200, 128),     # 800 heads of one segment in two chunks; 768 in one
    (1, 8, 4, 26880, 256), (3, 5, 5, 1111, 256),      # groups that would leave waves idle: 27 chunks of 1024, and a ragged batch
])
def test_key_scores_at_the_edges_of_the_split_form(dev, B, Hq, Hkv, S, seg):
    """Tolerance: logits are bf16 values, and one that falls the other way on a near tie of the rounding moves its
    probability by 2^-8 of the logit (|logit| < 6 here: under 3 %); sums of 128 of them move far less on average."""
    from oracle import pbs_oracle as O
    from pbs_attn_amd import ops
    q, k, _ = small_case(B, Hq, Hkv, S, seed=S + Hq)
    ref = O.key_scores(q, k, 128, seg)
    got = ops.score_keys(q.to(dev), k.to(dev), 128, seg).cpu()
    assert got.shape == ref.shape
    rel = (got - ref).abs() / ref.abs().clamp_min(1e-12)
    assert rel.max().item() < 3e-2 and rel.mean().item() < 2e-3
    assert torch.allclose(got.sum(-1), torch.ones(B, Hq), atol=2e-3)
