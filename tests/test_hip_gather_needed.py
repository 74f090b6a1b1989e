"""GPU: the filtered gather against the unfiltered one, on both sides of the 32768 blocks (16384 where rows have more than 1024) from which on a workgroup takes
four of a head: marked tiles bit for bit, the others untouched."""
import pytest
import torch

from pbs_attn_amd import _lib, ops
from tests.test_hip_routes_taken import _kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,S,four", [
    (8, 64, 8, 33 * 128 - 5, False),      # an odd number of blocks a head, the last one ragged: chunks of one block
    (1, 512, 512, 32 * 128, False),       # a head a group, whole chunks
    (8, 128, 8, 33 * 128 - 5, True), (1, 1024, 1024, 32 * 128, True), (3, 56, 8, 196 * 128 + 1, True),   # the same: 33792 blocks, 32768, 33096
    (1, 16, 2, 1025 * 128 - 5, True), (1, 16, 2, 1024 * 128, False),      # 16400 blocks in long rows, 16384 in rows of 1024
    (3, 28, 4, 196 * 128 + 1, False),     # seven heads a group
])
@pytest.mark.parametrize("share", [0.0, 0.03, 0.6, 1.0])
def test_against_the_unfiltered_gather(dev, B, Hq, Hkv, S, four, share):
    nb = (S + 127) // 128
    g = torch.Generator(device=dev).manual_seed(S)
    k, v = (torch.randn(B, Hkv, S, 128, device=dev, generator=g).bfloat16() for _ in "kv")
    idx = torch.rand(B, Hq, S, device=dev, generator=g).argsort(-1).to(torch.int32)
    idx = torch.cat((idx, torch.arange(S, nb * 128, device=dev, dtype=torch.int32).expand(B, Hq, -1)), -1).contiguous()
    needed = (torch.rand(B, Hq, nb, device=dev, generator=g) < share).to(torch.uint8)
    full_k, full_vt, _ = ops.gather_kv(k, v, idx, Hq, want_pooled=False)
    got_k, got_vt = torch.full_like(full_k, 7.0), torch.full_like(full_vt, 7.0)
    assert _kernels(lambda: _lib.check(_lib.load().pbs_gather_kv(
        k.data_ptr(), v.data_ptr(), idx.data_ptr(), got_k.data_ptr(), got_vt.data_ptr(), None, B, Hq, Hkv, S, 128, 128, *k.stride()[:3], *v.stride()[:3], 0,
        needed.data_ptr(), torch.cuda.current_stream().cuda_stream), "pbs_gather_kv")) == ["gather_needed_kernel" if four else "gather_kv_kernel"]
    on = needed.bool()
    for got, full in ((got_k, full_k), (got_vt, full_vt)):
        got, full = got.view(B, Hq, nb, -1), full.view(B, Hq, nb, -1)
        assert torch.equal(got[on], full[on]) and bool((got[~on] == 7.0).all())
