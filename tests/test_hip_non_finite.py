"""GPU: a NaN or an infinity in a token's K or V stays out of the rows that do not attend to the token: the rows before it
(their logits of later keys are masked, whatever they are) and the query blocks that did not select its block."""
import pytest
import torch

from pbs_attn_amd import ops
from pbs_attn_amd import pbs as P
from tests.util import heads_for_items, small_case

pytestmark = pytest.mark.gpu


def _attend(q, k, v, cols, cnt, seg):
    perm = P.apply_permutation(q, k, v, 128, seg, identity=True)
    return perm.attention(q, cols, cnt, seg).float()


def _random_lists(Hq, nb, bps, seed):
    """Visit lists in which every second earlier block, at random, is on a query block's list: (mask, cols, cnt)."""
    g = torch.Generator().manual_seed(seed)
    qb = torch.arange(nb)
    earlier = qb[None, :] < (qb // bps * bps)[:, None]
    mask = (torch.rand((1, Hq, nb, nb), generator=g) < 0.5) & earlier
    cnt = mask.sum(-1).int()
    cols = torch.where(mask, qb, nb).sort(-1).values.clamp(max=nb - 1).int().contiguous()
    return mask, cols, cnt


def _check(dev, Hq, S, seg, token, bad_k, bad_v, seed, scale=1):
    """The rows that do not attend to the token are finite and equal to those of the finite input up to rounding: an item with an
    overflow is repeated with other reference maxima, in which a probability rounded to bf16 differs by 2^-8 of itself at
    most, and the output, a mean of V under them, by that and its own rounding: 2^-7 of the largest |V| in all."""
    q, k, v = (x.to(dev) for x in small_case(1, Hq, 1, S, seed=seed))
    q, k = q * scale, k * scale
    nb, bps = (S + 127) // 128, seg // 128
    mask, cols, cnt = (x.to(dev) for x in _random_lists(Hq, nb, bps, seed))
    want = _attend(q, k, v, cols, cnt, seg)
    k2, v2 = k.clone(), v.clone()
    if bad_k is not None:
        k2[:, :, token] = bad_k if bad_k != bad_k else 0
        k2[:, :, token, 0] = bad_k      # an infinite logit of either sign
    if bad_v is not None:
        v2[:, :, token] = bad_v
    got = _attend(q, k2, v2, cols, cnt, seg)
    rows, block = torch.arange(S, device=dev), token // 128
    sees = mask[0, :, rows // 128, block] | ((rows // seg == token // seg) & (rows >= token))
    if bad_v is not None:
        sees |= rows // 128 == block   # (a probability of zero times an infinite V is NaN: a block's whole diagonal tile is multiplied)
    assert torch.isfinite(got[0][~sees]).all()
    assert (got - want)[0][~sees].abs().max().item() <= v.abs().max().item() / 128
    if "nan" in (str(bad_k), str(bad_v)):
        assert torch.isnan(got[0][sees & (rows >= token)]).all()


@pytest.mark.parametrize("pairs", [False, True])   # work items of one query block, of two
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("S,seg,token", [
    (128, 128, 127), (128, 128, 33), (77, 128, 64),                  # one diagonal tile
    (256, 256, 100), (256, 256, 130), (256, 256, 255), (1000, 512, 999), (1000, 512, 897),   # the pair's second block, a partial one
    (896, 256, 800),                                                 # a pair of one block
    (1024, 128, 991), (1024, 384, 1000),                             # segments of an odd number of blocks
])
def test_later_keys_of_the_diagonal_block(dev, S, seg, token, bad, pairs):
    _check(dev, heads_for_items(dev, pairs, S, seg), S, seg, token, bad, None, S + token)


@pytest.mark.parametrize("pairs", [False, True])
@pytest.mark.parametrize("scale", [1, 20])   # 20: exponents that overflow, the item is repeated
@pytest.mark.parametrize("bad_k,bad_v", [(float("nan"), None), (float("inf"), None), (None, float("nan")), (None, float("inf"))])
@pytest.mark.parametrize("S,seg,token", [
    (2048, 256, 300), (1900, 128, 5),   # a permuted tile that one block of a pair selected
    (1100, 384, 300),                   # the first block's own segment ends inside the pair; a last pair of one block
    (2048, 384, 130),                   # ... a tile before its diagonal
])
def test_blocks_that_did_not_select_the_token(dev, S, seg, token, bad_k, bad_v, scale, pairs):
    seed, heads = S + seg, heads_for_items(dev, pairs, S, seg)
    mask = _random_lists(heads, (S + 127) // 128, seg // 128, seed)[0][..., token // 128]
    first, second = mask[..., :-1:2], mask[..., 1::2]
    assert (first & ~second).any() and (second & ~first).any()
    _check(dev, heads, S, seg, token, bad_k, bad_v, seed, scale)
