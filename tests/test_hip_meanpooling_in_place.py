"""GPU: the MeanPooling mode as one library call, tiles read in place, against its stage-by-stage form (gathered tiles, CSR lists), bit for bit."""
import pytest
import torch

from pbs_attn_amd import _lib
from pbs_attn_amd.meanpooling import MeanPooling_prefill
from tests.util import small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,S,thr,first,kind", [
    (1, 2, 1, 1, 0.9, True, "uniform_heavy"), (2, 3, 1, 128, 0.9, True, "uniform_heavy"), (1, 4, 2, 129, 0.9, True, "strong_heavy"),
    (1, 32, 8, 3000, 0.8, True, "uniform_heavy"),                   # single-block items, short pass
    (2, 6, 2, 64 * 128, "rows", True, "strong_uniform"), (2, 6, 2, 65 * 128 - 7, "rows", False, "strong_uniform"),   # the last short pass; beyond
    (1, 8, 2, 40 * 128, 0.0, False, "uniform_heavy"),               # nothing but diagonal blocks (and ties of nothing)
    (1, 5, 5, 33 * 128, 1.0, True, "local_window"),                 # sums that may never reach the threshold
    (3, 28, 4, 50 * 128 + 1, 0.5, True, "strong_heavy"),            # pairs whose blocks select differently, odd block count
    (1, 1, 1, 1024 * 128, 0.9, True, "strong_heavy"), (1, 1, 1, 1025 * 128, 0.9, True, "strong_uniform"),   # the short selection's longest rows; the long one's shortest
    (1, 1, 1, 2048 * 128, 0.3, True, "uniform_heavy"), (1, 1, 1, 2048 * 128 + 1, 0.3, True, "uniform_heavy"),  # the longest rows of the single call
])
def test_single_call_equals_stages(dev, B, Hq, Hkv, S, thr, first, kind):
    q, k, v = (x.to(dev) for x in small_case(B, Hq, Hkv, S, kind=kind, seed=S + Hq))
    if thr == "rows":
        thr = torch.linspace(0.5, 0.95, B * Hq).view(B, Hq).to(dev)
    out = MeanPooling_prefill(q, k, v, threshold=thr, force_select_first_block=first)
    if S > 2048 * 128:
        masks = None
        staged = MeanPooling_prefill(q.clone(), k, v, threshold=thr, force_select_first_block=first)
    else:
        staged, masks = MeanPooling_prefill(q, k, v, threshold=thr, force_select_first_block=first, return_masks=True)
    assert torch.equal(out, staged)
    qt, kt, vt = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v))
    assert torch.equal(MeanPooling_prefill(qt, kt, vt, threshold=thr, force_select_first_block=first), out)


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
