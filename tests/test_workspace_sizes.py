"""CPU: the workspace sizes that the library states, which are host arithmetic over the plans of its launches."""
import pytest

from pbs_attn_amd import _lib


def _chunks(lib, heads, group, S, segment):
    """Chunks of keys that the scoring plan cuts a sequence into, read back from the space for their partials (128 queries x two
    floats a chunk and head, and the statistics as one chunk more)."""
    n = lib.pbs_score_keys_workspace_bytes(1, heads, heads // group, S, segment)
    per_chunk = heads * 128 * 2 * 4
    assert n % per_chunk == 0
    return n // per_chunk - 1


@pytest.mark.parametrize("S,segment", [(128, 128), (200, 128), (255, 128), (256, 256), (300, 128), (1000, 256), (4096, 1024),
                                       (16384, 128), (16512, 128), (131072, 1024)])
def test_scoring_cuts_every_sequence_into_chunks(S, segment):
    lib = _lib.load()
    for group in (1, 3, 4, 7, 16):
        for kv_heads in [*range(1, 100), *range(180, 200), 255, 256, 257, 383, 384, 385, 511, 512, 513, *range(760, 780), 1023, 1024,
                         1535, 1536, 1537, 4096, 65535]:
            heads = kv_heads * group
            if heads <= 65535:
                chunks = _chunks(lib, heads, group, S, segment)
                assert 1 <= chunks <= S // segment * segment // 64, (heads, group, chunks)


def test_scoring_chunks_of_more_heads_than_run_at_once():
    """One segment of 128 keys: up to 768 heads one chunk or two, so that all workgroups run at once; more heads never do, and keep two."""
    lib = _lib.load()
    assert [_chunks(lib, heads, 4, 200, 128) for heads in (384, 388, 768, 772, 800, 1536)] == [2, 1, 1, 2, 2, 2]


LENGTHS = sorted({*range(1, 140), *range(140, 1100, 7), 384, 512, 513, 1024, 2047, 2048, 2049, 4095, 4096})   # in blocks
HEADS = [1, 2, 3, 4, 5, 8, 15, 16, 17, 24, 28, 32, 33, 64, 96, 128, 129, 256, 384, 385, 512, 513, 1000, 4096]


def _not_growing(sizes):
    return [(a, b) for a, b in zip(sizes, sizes[1:]) if a[1] > b[1]]


@pytest.mark.parametrize("segment", [128, 256, 384, 1024, 8192])
def test_attention_workspace_grows_with_the_shape(segment):
    """pbs_sparse_attn_fwd is not told how large its workspace is: one that was made for the longest sequence and the most heads
    has to hold the lists of every smaller call too."""
    lib = _lib.load()
    size = lambda heads, blocks, tail=0, seg=segment: lib.pbs_sparse_attn_workspace_bytes(1, heads, blocks * 128 - tail, seg)
    for heads in HEADS:
        assert not _not_growing([(n, size(heads, n)) for n in LENGTHS]), heads
        assert all(size(heads, n, 127) == size(heads, n) for n in LENGTHS)   # (whole blocks)
    for n in LENGTHS:
        assert not _not_growing([(heads, size(heads, n)) for heads in HEADS]), n
        assert size(6, n) == lib.pbs_sparse_attn_workspace_bytes(3, 2, n * 128, segment)
        assert not _not_growing([(seg, size(32, n, seg=seg)) for seg in (128, 256, 384, 1024, 8192, 65536)]), n


def test_single_call_workspaces_grow_with_the_length():
    """A sequence inside one segment needs the lists alone; the MeanPooling mode its pooled blocks, probabilities and lists."""
    lib = _lib.load()
    for heads in HEADS:
        one_segment = [(n, lib.pbs_prefill_attn_workspace_bytes(1, heads, heads, n * 128, 128, 128, 511 * 128)) for n in LENGTHS if n <= 511]
        assert not _not_growing(one_segment), heads
        assert not _not_growing([(n, lib.pbs_meanpooling_attn_workspace_bytes(1, heads, heads, n * 128, 128, 128)) for n in LENGTHS]), heads


@pytest.mark.parametrize("B,Hq,Hkv", [(1, 1, 1), (1, 4, 1), (1, 8, 2), (1, 12, 3), (1, 16, 16), (1, 28, 4), (1, 32, 8), (2, 32, 8), (4, 28, 4),
                                      (25, 32, 8), (8, 128, 8)])
def test_prefill_workspace_grows_with_the_length(B, Hq, Hkv):
    """The space for the chunk partials of the key scoring covers those of a shorter sequence, which may be cut into more chunks."""
    lib = _lib.load()
    lengths = sorted({*range(1, 6000, 61), *range(6000, 70000, 997), *range(128, 6016, 128), *range(6016, 70000, 896), 131072, 262144})
    for segment in (128, 256, 384, 512, 1024, 4096, 65408):
        assert not _not_growing([(S, lib.pbs_prefill_attn_workspace_bytes(B, Hq, Hkv, S, 128, 128, segment)) for S in lengths]), segment
