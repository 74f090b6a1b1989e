"""GPU: sequences of one block (up to 128 tokens) take a kernel of their own, 32 queries a workgroup and 32 keys a wave.  Against the persistent kernel,
which the stage-by-stage calls run, bit for bit, at the edges of its sub-tiles."""
import pytest
import torch

from pbs_attn_amd import pbs as P
from pbs_attn_amd.meanpooling import MeanPooling_prefill
from tests.test_hip_prefill_routes import _NullTimer
from tests.util import assert_attn_close, expand_kv, small_case

pytestmark = pytest.mark.gpu


def _staged(q, k, v):
    P.stage_timer = _NullTimer()
    try:
        return P.permuted_block_sparse_attn_fwd(q, k, v, 128, 256, 0.9, True)
    finally:
        P.stage_timer = None


def _same(a, b):
    nan = torch.isnan(a)
    return torch.equal(nan, torch.isnan(b)) and torch.equal(a[~nan], b[~nan])


@pytest.mark.parametrize("scale", [1, 30])
@pytest.mark.parametrize("B,Hq,Hkv,S", [(1, 1, 1, 1), (1, 3, 3, 16), (2, 6, 2, 17), (1, 28, 4, 31), (1, 4, 4, 32), (3, 8, 1, 33), (1, 8, 2, 64), (2, 5, 5, 65),
                                        (1, 32, 8, 77), (1, 12, 3, 96), (1, 4, 2, 97), (1, 300, 100, 127), (2, 32, 8, 128), (40, 7, 1, 128)])
def test_against_the_persistent_kernel(dev, B, Hq, Hkv, S, scale):
    q, k, v = (x.to(dev) for x in small_case(B, Hq, Hkv, S, seed=S))
    q = q * scale
    got = P.permuted_block_sparse_attn_fwd(q, k, v, 128, 256, 0.9, True)
    assert torch.equal(got, _staged(q, k, v))
    assert torch.equal(got, MeanPooling_prefill(q, k, v, threshold=0.3, force_select_first_block=False))   # its one block is always selected
    if scale == 1:
        ke, ve = expand_kv(q, k), expand_kv(q, v)
        logits = (q.float() @ ke.float().transpose(-1, -2) / 128 ** 0.5).masked_fill(~torch.ones(S, S, dtype=torch.bool, device=dev).tril(), float("-inf"))
        assert_attn_close(got, torch.softmax(logits, -1) @ ve.float())
    # (batch, token, head, d) memory; rows of 16-byte alignment only, inside one tensor whose other entries are NaN
    qt = q.transpose(1, 2).contiguous().transpose(1, 2)
    kv = torch.full((B, S, Hkv, 3 * 128 + 8), float("nan"), dtype=torch.bfloat16, device=dev)
    kv[..., 8:136], kv[..., 264:392] = k.transpose(1, 2), v.transpose(1, 2)
    assert torch.equal(P.permuted_block_sparse_attn_fwd(qt, kv[..., 8:136].transpose(1, 2), kv[..., 264:392].transpose(1, 2), 128, 256, 0.9, True), got)


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("which", "qkv")
@pytest.mark.parametrize("S,token", [(77, 76), (128, 40), (100, 0)])
def test_tokens_that_are_not_finite(dev, S, token, which, value):
    x = {n: t.to(dev) for n, t in zip("qkv", small_case(1, 4, 2, S, seed=S + token))}
    x[which][:, :, token] = value
    assert _same(P.permuted_block_sparse_attn_fwd(x["q"], x["k"], x["v"], 128, 256, 0.9, True), _staged(x["q"], x["k"], x["v"]))
