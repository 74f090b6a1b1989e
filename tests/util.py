"""Shared helpers for the parity tests."""
import math

import torch

from pbs_attn_amd.synth import make_qkv


def small_case(B=1, Hq=4, Hkv=2, S=1024, D=128, kind="uniform_heavy", seed=0):
    return make_qkv(B, Hq, Hkv, S, D, kind=kind, seed=seed, device="cpu")


def expand_kv(q, x):
    from oracle.pbs_oracle import repeat_kv
    return repeat_kv(x, q.shape[1] // x.shape[1])


def assert_attn_close(out, ref, max_abs=2e-2, mean_abs=2e-3, what=""):
    """North-star tolerance for bf16 attention outputs."""
    diff = (out.float().cpu() - ref.float().cpu()).abs()
    assert torch.isfinite(out.float()).all(), f"{what}: non-finite output"
    assert diff.max().item() <= max_abs, f"{what}: max-abs {diff.max().item():.4g} > {max_abs}"
    assert diff.mean().item() <= mean_abs, f"{what}: mean-abs {diff.mean().item():.4g} > {mean_abs}"


def quantised_scores(shape, levels, seed):
    """Random scores on a coarse grid: plenty of exact ties."""
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, levels, shape, generator=g).float() / levels


def blocks_of_an_item(dev, rows, S, seg):
    """Query blocks of a work item of the attention launch for `rows` heads over the batch (two, or one), read from the visit lists that
    a call leaves in its workspace: a row of uint16 per item, the head's last item first, with [4] the item's first query block and [5] how many."""
    from pbs_attn_amd import _lib
    lib = _lib.load()
    nb, bps = (S + 127) // 128, seg // 128
    assert nb > 1
    x = torch.zeros((1, rows, S, 128), dtype=torch.bfloat16, device=dev)
    cols = torch.zeros((rows, nb, nb), dtype=torch.int32, device=dev)
    cnt = torch.zeros((rows, nb), dtype=torch.int32, device=dev)   # no permuted tile is visited
    ws = torch.zeros(lib.pbs_sparse_attn_workspace_bytes(1, rows, S, seg), dtype=torch.uint8, device=dev)
    out = torch.empty_like(x)
    p, st = x.data_ptr(), x.stride()[:3]
    _lib.check(lib.pbs_sparse_attn_fwd(p, p, p, p, p, cols.data_ptr(), cnt.data_ptr(), out.data_ptr(), 1, rows, 1, S, 128, 128,
                                       seg, *st, *st, *st, *st, 1.0, ws.data_ptr(), torch.cuda.current_stream().cuda_stream), "pbs_sparse_attn_fwd")
    cap = (8 + nb + min(bps, nb) + 1 + 7) // 8 * 8
    lists = ws[256:].view(torch.int16).cpu()
    return int(lists[(nb % 2) * cap + 5])   # (an odd row's last pair is a single block)


def heads_for_items(dev, pairs, S, seg, kv_heads=1, few=3):
    """A number of query heads, a multiple of `kv_heads`, whose launch is cut into pairs of query blocks, or into single ones (`few` of them)."""
    nb = (S + 127) // 128
    heads = (512 // nb + kv_heads) // kv_heads * kv_heads if pairs else few
    assert nb == 1 or blocks_of_an_item(dev, heads, S, seg) == 1 + pairs
    return heads
