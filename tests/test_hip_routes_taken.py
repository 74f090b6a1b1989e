"""GPU: which kernels a call launches, on both sides of the rules that choose them.  The routes give the same bits, so a comparison of outputs does not
notice a rule that no longer chooses the kernel it was made for."""
import re

import pytest
import torch

from pbs_attn_amd import pbs as P
from pbs_attn_amd.meanpooling import MeanPooling_prefill
from tests.util import small_case

pytestmark = pytest.mark.gpu

SCORES = ["score_kernel", "score_kernel"]
REST = ["estimate_select_kernel", "sparse_attn_kernel"]
GATHER_SORTS = SCORES + ["sort_gather_pool_kernel"] + REST
PASS_SORTS = SCORES + ["gather_pool_kernel"] + REST
LONG = ["score_kernel", "score_reduce_kernel", "score_kernel", "segment_argsort_wave_kernel", "pool_qk_kernel", "block_logits_softmax_kernel", "select_pair_lists_kernel"]
KERNEL_SORTS = SCORES + ["segment_argsort_wave_kernel", "gather_pool_kernel"] + REST


def _kernels(call):
    """The names of the library's kernels that `call` launches, in order, without their template arguments."""
    call()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA], acc_events=True) as prof:
        call()
        torch.cuda.synchronize()
    events = sorted((e for e in prof.events() if e.device_type == torch.autograd.DeviceType.CUDA), key=lambda e: e.time_range.start)
    names = [re.search(r"(?:anonymous namespace\)::|_GLOBAL__N_1\d+)(\w+?_kernel)\b", e.name) for e in events if "at::" not in e.name]
    return [m.group(1) for m in names if m]


@pytest.mark.parametrize("B,Hq,Hkv,S,seg,thr,kernels", [
    (1, 32, 8, 77, 256, 0.9, ["one_block_attn_kernel"]), (2, 256, 64, 128, 256, 0.9, ["one_block_attn_kernel"]),
    (1, 4, 2, 129, 256, 0.9, ["sparse_attn_kernel"]), (1, 33, 3, 2048, 2048, 0.9, ["merge_pair_lists_kernel", "sparse_attn_kernel"]),
    # the gather sorts: ranks up to 256 keys and 255 heads, where the scoring pass would take no more keys than a segment
    (1, 28, 4, 1000, 256, 0.9, GATHER_SORTS), (1, 255, 51, 300, 128, 0.9, GATHER_SORTS), (1, 256, 64, 300, 128, 0.9, PASS_SORTS),
    (1, 4, 1, 6000, 256, 0.9, GATHER_SORTS), (1, 4, 1, 6000, 128, 0.9, PASS_SORTS),
    # longer segments: up to 1024 keys, 768 blocks and 24 sorting workgroups on a shader engine
    (1, 32, 8, 24 * 128, 512, 0.9, GATHER_SORTS), (1, 33, 11, 24 * 128, 512, 0.9, KERNEL_SORTS),
    (1, 32, 8, 18 * 128, 1024, 0.9, GATHER_SORTS), (2, 32, 8, 9 * 128, 1024, 0.9, KERNEL_SORTS), (1, 28, 4, 20 * 128, 1024, 0.9, KERNEL_SORTS),   # 24; 32; 28
    (4, 28, 4, 6 * 128, 512, 0.9, GATHER_SORTS), (4, 28, 4, 6 * 128, 640, 0.9, KERNEL_SORTS),                                             # 14; 28, five blocks of a chunk
    (1, 2, 1, 2 * 1024 + 128, 1024, 0.9, GATHER_SORTS), (1, 2, 1, 3 * 1152 + 1, 1152, 0.9, KERNEL_SORTS),
    # short passes: up to 2048 blocks, 64 a row
    (1, 32, 8, 64 * 128, 256, 0.9, ["score_kernel", "score_reduce_kernel", "score_kernel"] + GATHER_SORTS[2:]),
    (1, 33, 11, 64 * 128, 256, 0.9, SCORES + ["segment_argsort_wave_kernel", "gather_kv_kernel", "block_logits_softmax_kernel",   # three heads a group: the split
                                              "select_pair_lists_kernel", "gather_kv_kernel", "sparse_attn_kernel"]),             # scoring, without a reduction
    # the filtered gather: from 32768 blocks on four a workgroup
    (1, 1024, 8, 32 * 128, 1024, 0.9, LONG + ["gather_needed_kernel", "sparse_attn_kernel"]), (1, 1016, 8, 32 * 128, 1024, 0.9, LONG + ["gather_kv_kernel", "sparse_attn_kernel"]),
])
def test_prefill(dev, B, Hq, Hkv, S, seg, thr, kernels):
    q, k, v = (x.to(dev) for x in small_case(B, Hq, Hkv, S, seed=S))
    assert _kernels(lambda: P.permuted_block_sparse_attn_fwd(q, k, v, 128, seg, thr, True)) == kernels


@pytest.mark.parametrize("S,kernels", [(128, ["one_block_attn_kernel"]), (129, ["pool_qk_kernel", "estimate_select_kernel", "sparse_attn_kernel"])])
def test_meanpooling(dev, S, kernels):
    q, k, v = (x.to(dev) for x in small_case(1, 4, 2, S, seed=S))
    assert _kernels(lambda: MeanPooling_prefill(q, k, v)) == kernels
