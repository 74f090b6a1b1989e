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
