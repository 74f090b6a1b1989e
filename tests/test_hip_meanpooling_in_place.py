"""GPU: the MeanPooling mode as one library call, tiles read in place, against its stage-by-stage form (gathered tiles, CSR lists), bit for bit."""
import pytest
import torch

from pbs_attn_amd import _lib, ops
from pbs_attn_amd.meanpooling import MeanPooling_prefill
from tests.util import assert_attn_close, heads_for_items, small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,S,thr,first,kind", [
    (1, 2, 1, 1, 0.9, True, "uniform_heavy"), (2, 3, 1, 128, 0.9, True, "uniform_heavy"), (1, 4, 2, 129, 0.9, True, "strong_heavy"),
    (1, 32, 8, 3000, 0.8, True, "uniform_heavy"),                   # single-block items, short pass
    (2, 6, 2, 64 * 128, "rows", True, "strong_uniform"), (2, 6, 2, 65 * 128 - 7, "rows", False, "strong_uniform"),   # the last short pass; beyond
    (1, 8, 2, 40 * 128, 0.0, False, "uniform_heavy"),               # nothing but diagonal blocks (and ties of nothing)
    (1, 5, 5, 33 * 128, 1.0, True, "local_window"),                 # sums that may never reach the threshold
    (3, 28, 4, 50 * 128 + 1, 0.5, True, "strong_heavy"),            # pairs whose blocks select differently, odd block count
    (1, 1, 1, 1024 * 128, 0.9, True, "strong_heavy"), (1, 1, 1, 1025 * 128, 0.9, True, "strong_uniform"),   # the short selection's longest rows; the long one's shortest
    (1, 1, 1, 2048 * 128, 0.3, True, "uniform_heavy"),   # the longest rows of the single call
])
def test_single_call_equals_stages(dev, B, Hq, Hkv, S, thr, first, kind):
    q, k, v = (x.to(dev) for x in small_case(B, Hq, Hkv, S, kind=kind, seed=S + Hq))
    if thr == "rows":
        thr = torch.linspace(0.5, 0.95, B * Hq).view(B, Hq).to(dev)
    out = MeanPooling_prefill(q, k, v, threshold=thr, force_select_first_block=first)
    staged, _ = MeanPooling_prefill(q, k, v, threshold=thr, force_select_first_block=first, return_masks=True)
    assert torch.equal(out, staged)
    qt, kt, vt = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v))
    assert torch.equal(MeanPooling_prefill(qt, kt, vt, threshold=thr, force_select_first_block=first), out)


def _taken(monkeypatch):
    """Counts the library calls of the whole mode."""
    taken = []
    inner = ops.meanpooling_attn_fwd
    monkeypatch.setattr(ops, "meanpooling_attn_fwd", lambda *a: taken.append(1) or inner(*a))
    return taken


def test_more_blocks_than_the_single_call_takes(dev, monkeypatch):
    """2048 blocks are its longest rows; with one more the stages run, here against dense attention on their mask at sampled query blocks."""
    taken = _taken(monkeypatch)
    S = 2048 * 128 + 1
    q, k, v = (x.to(dev) for x in small_case(1, 1, 1, S, seed=S))
    MeanPooling_prefill(q[:, :, 1:], k[:, :, 1:], v[:, :, 1:], threshold=0.3)
    assert len(taken) == 1
    out = MeanPooling_prefill(q, k, v, threshold=0.3)
    assert len(taken) == 1
    _, masks = MeanPooling_prefill(q, k, v, threshold=0.3, return_masks=True)
    pos = torch.arange(S, device=dev)
    for qb in (0, 5, 1023, 2047, 2048):
        rows = slice(128 * qb, min(128 * qb + 128, S))
        allowed = masks["block_mask"][:, :, qb][:, :, None].repeat_interleave(128, -1)[..., :S] & (pos <= pos[rows, None])
        logits = (q[:, :, rows].float() @ k.float().transpose(-1, -2) / 128 ** 0.5).masked_fill(~allowed, float("-inf"))
        assert_attn_close(out[:, :, rows], torch.softmax(logits, -1) @ v.float(), what=f"query block {qb} of 2049")


def _same(a, b):
    """Bit for bit, NaN in the same places."""
    nan = torch.isnan(a)
    return torch.equal(nan, torch.isnan(b)) and torch.equal(a[~nan], b[~nan])


@pytest.mark.parametrize("pairs", [False, True])   # work items of one query block, of two
@pytest.mark.parametrize("scale", [1, 20])         # 20: exponents that overflow, the item is repeated
@pytest.mark.parametrize("bad_k,bad_v", [(None, None), (float("nan"), None), (float("inf"), None), (None, float("nan")), (None, float("inf"))])
@pytest.mark.parametrize("S,token", [(1900, 300), (2048, 1000), (1100, 1099)])   # a token of a first block, of a second one, of a last pair of one block
def test_non_finite_tokens_and_repeated_items(dev, monkeypatch, S, token, bad_k, bad_v, scale, pairs):
    """Single call and stages alike; a bad V, which the selection does not see, stays out of the rows that do not attend to its token
    (all of its block's rows do: a probability of zero times an infinite V is NaN).  A repeated item uses other reference maxima:
    2^-7 of the largest |V|, for a probability and the output rounded to bf16."""
    taken = _taken(monkeypatch)
    q, k, v = (x.to(dev) for x in small_case(1, heads_for_items(dev, pairs, S, 128), 1, S, seed=S + token))
    q, k = q * scale, k * scale
    want, masks = MeanPooling_prefill(q, k, v, threshold=0.5, return_masks=True)
    if bad_k is None and bad_v is None and scale > 1:   # against dense attention on the mask, where every item may be repeated
        mask = masks["block_mask"].repeat_interleave(128, -1).repeat_interleave(128, -2)[..., :S, :S]
        causal = torch.ones(S, S, dtype=torch.bool, device=dev).tril()
        for h in (0, q.shape[1] - 1):
            logits = (q[0, h].float() @ k[0, 0].float().T / 128 ** 0.5).masked_fill(~(mask[0, h] & causal), float("-inf"))
            assert_attn_close(want[0, h], torch.softmax(logits, -1) @ v[0, 0].float(), what=f"head {h}")
    k2, v2 = k.clone(), v.clone()
    if bad_k is not None:
        k2[:, :, token] = bad_k
    if bad_v is not None:
        v2[:, :, token] = bad_v
    staged, _ = MeanPooling_prefill(q, k2, v2, threshold=0.5, return_masks=True)
    assert not taken
    got = MeanPooling_prefill(q, k2, v2, threshold=0.5)
    assert taken and _same(got, staged)
    if bad_k is None:
        block = token // 128
        apart = ~masks["block_mask"][0, :, :, block].repeat_interleave(128, -1)[:, :S]
        mixed = masks["block_mask"][0, :, :-1:2, block] != masks["block_mask"][0, :, 1::2, block]
        assert apart.any() and (token == S - 1 or mixed.any())   # (of some pairs one block selected the token's)
        assert torch.isfinite(got[0][apart]).all()
        assert (got.float() - want.float())[0][apart].abs().max().item() <= v.abs().max().item() / 128
        if bad_v is not None and bad_v != bad_v:
            assert torch.isnan(got[0][~apart]).all()


def test_single_call_refuses_what_it_cannot_take(dev):
    lib = _lib.load()
    q = torch.zeros(1, 2, 256, 128, dtype=torch.bfloat16, device=dev)
    n = lib.pbs_meanpooling_attn_workspace_bytes(1, 2, 2, 256, 128, 128)
    ws = torch.empty(n, dtype=torch.uint8, device=dev)
    st = q.stride()[:3]

    def call(S=256, D=128, block=128, space=ws.data_ptr(), size=n):
        p = q.data_ptr()
        return lib.pbs_meanpooling_attn_fwd(p, p, p, p, 1, 2, 2, S, D, block, *st, *st, *st, *st, 0.9, None, 1, 0.09, space, size,
                                            torch.cuda.current_stream().cuda_stream)
    assert call(space=None) == -1 and call(size=n - 1) == -1 and call(D=64) == -1 and call(block=64, size=1 << 40) == -1
    assert call(S=2048 * 128 + 1, size=1 << 40) == -1
    with pytest.raises(_lib.PbsHipError):
        MeanPooling_prefill(q.cpu(), q.cpu(), q.cpu())


def test_single_call_refuses_mismatched_shapes(dev):
    q = torch.zeros(2, 4, 256, 128, dtype=torch.bfloat16, device=dev)
    k = q[:, :2]
    for bad_k, bad_v in ((k, k[:, :, :128]), (k, k[:, :1]), (k, k[:1]), (k[:1], k), (k[..., :64], k)):
        with pytest.raises(AssertionError):   # the stage-by-stage form's own host checks refuse the same
            MeanPooling_prefill(q, bad_k, bad_v)
