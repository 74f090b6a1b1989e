"""GPU: the routes of the single-call path (pbs_prefill_attn_fwd) against the stage-by-stage calls, bit for bit: the same
tiles in the same order, whatever kernel wrote the visit lists.  Shapes at the edges of the routes."""
import pytest
import torch

from pbs_attn_amd import pbs as P
from tests.util import small_case

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
