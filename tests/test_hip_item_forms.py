"""GPU: how a pass is cut into work items (pairs of query blocks or single ones) and in which order they are handed out does not
touch the arithmetic: the same heads in launches of other sizes, bit for bit, at the limits of either rule."""
import pytest
import torch

from pbs_attn_amd import pbs as P
from tests.util import small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv,S,seg,thr,reps,kind,pool", [
    (4, 1, 96 * 128, 256, 0.9, 2, "uniform_heavy", "mean"),     # 384 blocks of few heads one by one; 768 in pairs, 384 items dealt by heads
    (16, 4, 32 * 128 - 5, 512, 0.9, 3, "strong_uniform", "max"),  # 512 blocks of sixteen heads one by one, 1536 in pairs
    (24, 8, 16 * 128, 256, 0.9, 2, "uniform_heavy", "mean"),    # 384 one by one, 768 in pairs: whole heads per range, three and six of them
    (25, 5, 15 * 128 + 1, 384, 0.8, 1, "strong_heavy", "mean"),  # 400 blocks of 25 heads: pairs, an odd number of blocks
    (28, 4, 13 * 128 + 77, 128, 0.5, 3, "local_window", "mean"),  # 392 in pairs, dealt over all heads; 84 heads
    (7, 7, 9 * 128, 128, 0.0, 9, "uniform_heavy", "mean"),      # rows without selected blocks, items of one tile
    (1, 1, 300 * 128, 1024, 0.9, 5, "strong_heavy", "mean"),    # one head: 300 single blocks; 750 pairs of five
    (8, 2, 350 * 128, 1024, 0.9, 2, "strong_heavy", "mean"),    # 1400 items, dealt; 2800, head by head
    (8, 8, 89 * 128, 128, 0.9, 3, "uniform_heavy", "mean"),     # 45 items a head: one head a range; three, the long lists head by head
    (16, 16, 89 * 128, 512, 0.9, 2, "strong_heavy", "mean"),    # the same length, short lists: dealt
    (8, 4, 87 * 128, 256, 0.9, 7, "local_window", "mean"),      # 44 items a head, seven heads a range: a group of four and one of three
    (5, 5, 559 * 128, 1024, 0.9, 2, "strong_uniform", "mean"),  # 1400 items dealt over all heads; 2800 head by head
])
def test_the_same_heads_in_launches_of_other_sizes(dev, Hq, Hkv, S, seg, thr, reps, kind, pool):
    q, k, v = (x.to(dev) for x in small_case(1, Hq, Hkv, S, kind=kind, seed=S + Hq))
    kw = dict(query_pool_mode=pool, key_pool_mode=pool)
    whole = P.permuted_block_sparse_attn_fwd(q.repeat(reps, 1, 1, 1), k.repeat(reps, 1, 1, 1), v.repeat(reps, 1, 1, 1), 128, seg, thr, True, **kw)
    alone = P.permuted_block_sparse_attn_fwd(q, k, v, 128, seg, thr, True, **kw)
    assert torch.equal(whole, alone.expand(reps, -1, -1, -1))
    # one KV head's query heads by themselves, on the key order and the visit lists of all of them (scores of other head counts come from
    # another split of the keys: their sums may differ in the last bit, and with them the order)
    perm = P.apply_permutation(q, k, v, 128, seg, pool)
    sel = P.permuted_block_selection(q, perm, 128, seg, thr, want_masks=False, **kw)
    together = perm.attention(q, sel["csr_cols"], sel["csr_cnt"], seg)
    g = Hq // Hkv
    part = P.PermutedKV(*(x[:, :g].contiguous() for x in (perm.key_indices, perm.perm_k, perm.perm_vt, perm.pooled_k)), S, k[:, :1], v[:, :1])
    assert torch.equal(part.attention(q[:, :g], *(sel[x][:, :g].contiguous() for x in ("csr_cols", "csr_cnt")), seg), together[:, :g])


@pytest.mark.parametrize("Hq,Hkv,S,reps", [(32, 8, 77, 1), (16, 4, 2048, 3), (32, 8, 295, 4), (32, 8, 1536, 2), (32, 8, 1021, 4), (8, 8, 4096 - 1, 3), (24, 8, 1400, 1), (3, 1, 128, 40), (1, 1, 511 * 128, 2), (28, 4, 1500, 2), (9, 3, 40 * 128 - 1, 2)])
def test_one_segment_in_launches_of_other_sizes(dev, Hq, Hkv, S, reps):
    q, k, v = (x.to(dev) for x in small_case(1, Hq, Hkv, S, seed=S))
    run = lambda a, b, c: P.permuted_block_sparse_attn_fwd(a, b, c, 128, 65536, 0.9, True)
    alone = run(q, k, v)
    assert torch.equal(run(q.repeat(reps, 1, 1, 1), k.repeat(reps, 1, 1, 1), v.repeat(reps, 1, 1, 1)), alone.expand(reps, -1, -1, -1))
    g = Hq // Hkv
    assert torch.equal(run(q[:, -g:], k[:, -1:], v[:, -1:]), alone[:, -g:])
    if S <= 4096:
        ref = torch.nn.functional.scaled_dot_product_attention(q.float(), k.float().repeat_interleave(g, 1), v.float().repeat_interleave(g, 1), is_causal=True)
        assert (alone.float() - ref).abs().max().item() <= 2e-2
