"""The native call of short prompts takes the plain case and hands everything else to the general path, which then serves or refuses it."""
import importlib.machinery
import os
import warnings

import pytest
import torch

from pbs_attn_amd import _lib, ops
from pbs_attn_amd import pbs as P
from tests.util import small_case


@pytest.fixture(params=["missing", "of another kind"])
def without_the_module(request, monkeypatch, tmp_path):
    path = tmp_path / os.path.basename(_lib.HOST_PATH)
    if request.param != "missing":
        path.write_bytes(b"no module")
    monkeypatch.setattr(_lib, "HOST_PATH", str(path))
    monkeypatch.setattr(_lib, "_one_segment", None)


def test_without_the_module_the_general_path_takes_every_call(without_the_module):
    q, k, v = small_case(1, 4, 2, 77)
    with pytest.warns(UserWarning, match="through Python"):
        native = _lib.one_segment()
    assert native(q, k, v, 128, 256, 0.9, True, True, "mean", "mean") is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _lib.one_segment() is native   # looked for once


def test_the_module_is_named_after_its_interpreter():
    from pbs_attn_amd import build
    assert build.HOST_PATH == _lib.HOST_PATH
    assert os.path.basename(_lib.HOST_PATH) == "_pbs_host" + importlib.machinery.EXTENSION_SUFFIXES[0]   # the most specific that is looked for


@pytest.mark.gpu
@pytest.mark.parametrize("S", [77, 300, 5000])
def test_calls_without_the_module(dev, without_the_module, S):
    q, k, v = (x.to(dev) for x in small_case(1, 4, 2, S, seed=S))
    with pytest.warns(UserWarning, match="through Python"):
        out = P.permuted_block_sparse_attn_fwd(q, k, v, 128, 256, 0.9, True)
    assert torch.equal(out, ops.prefill_attn_fwd(q, k, v, 128, 256, 0.9))


def test_tensors_on_the_host_are_not_taken():
    if not os.path.exists(_lib.HOST_PATH):
        from pbs_attn_amd.build import build_host_module
        build_host_module()
    q, k, v = small_case(1, 4, 2, 77)
    native = _lib.one_segment()
    assert native(q, k, v, 128, 256, 0.9, True, True, "mean", "mean") is None
    assert native(None, "k", 3, 128, 256, 0.9, True, True, "mean", "mean") is None
    with pytest.raises(TypeError):
        native(q, k, v)


def test_an_interrupt_is_not_swallowed():
    """Attributes are read through the modes that are on; what one raises there is met again by the general path, unless it ends the program."""
    from torch.overrides import TorchFunctionMode

    class Raising(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            raise self.error

    q, k, v = small_case(1, 4, 2, 77)
    native = _lib.one_segment()
    for error in (KeyboardInterrupt, RuntimeError("no")):
        with Raising() as mode:
            mode.error = error
            if error is KeyboardInterrupt:
                with pytest.raises(KeyboardInterrupt):
                    native(q, k, v, 128, 256, 0.9, True, True, "mean", "mean")
            else:
                assert native(q, k, v, 128, 256, 0.9, True, True, "mean", "mean") is None


class _Subclass(torch.Tensor):
    pass


def _with_rows_off_by(x, n):
    """`x` in memory whose rows start `n` elements further on."""
    wide = torch.zeros(*x.shape[:-1], x.shape[-1] + 8, dtype=x.dtype, device=x.device)
    wide[..., n:n + x.shape[-1]] = x
    return wide[..., n:n + x.shape[-1]]


@pytest.mark.gpu
def test_against_the_general_path(dev):
    """What is taken and what is not; both ways the result of the general path."""
    native = _lib.one_segment()
    plain = dict(block_size=128, segment_size=256, threshold=0.9, causal=True, use_triton=True, query_pool_mode="mean", key_pool_mode="mean")

    def check(q, k, v, taken, **kw):
        a = {**plain, **kw}
        out = native(q, k, v, *a.values())
        assert (out is not None) == taken, (q.shape, kw)
        want = ops.prefill_attn_fwd(q, k, v, a["block_size"], a["segment_size"], a["threshold"], True, a["query_pool_mode"], a["key_pool_mode"])
        whole = P.permuted_block_sparse_attn_fwd(q, k, v, **a)
        assert torch.equal(whole, want) and whole.is_contiguous() and (out is None or torch.equal(out, want))

    def case(B, Hq, Hkv, S):
        return [x.to(dev) for x in small_case(B, Hq, Hkv, S, seed=S)]

    for B, Hq, Hkv, S in [(1, 32, 8, 77), (1, 1, 1, 1), (2, 6, 2, 256), (1, 128, 8, 256), (3, 4, 1, 129)]:
        check(*case(B, Hq, Hkv, S), True)
    check(*case(1, 2, 1, 128 * 128), True, segment_size=128 * 128)             # 256 blocks, the last
    check(*case(1, 2, 1, 128 * 128 + 1), False, segment_size=129 * 128)
    check(*case(1, 257, 1, 100), False)
    check(*case(1, 4, 2, 257), False)                                          # longer than its segment
    check(*case(1, 4, 2, 257), True, segment_size=1 << 30)
    q, k, v = case(2, 4, 2, 200)
    for kw in (dict(threshold=1), dict(threshold=torch.full((2, 4), 0.9, device=dev))):
        check(q, k, v, False, **kw)
    check(q, k, v, True, query_pool_mode="max", key_pool_mode="max")
    check(q.as_subclass(_Subclass), k, v, False)
    check(*(x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v)), True)
    for n in (4, 8):                                                           # rows of 8-byte, of 16-byte alignment
        check(q, _with_rows_off_by(k, n), v, n == 8)
        check(_with_rows_off_by(q, n), k, v, n == 8)
    check(q, k, v.transpose(-1, -2).contiguous().transpose(-1, -2), False)     # no unit stride
    for bad in (dict(segment_size=200), dict(causal=False)):
        assert native(q, k, v, *{**plain, **bad}.values()) is None
        with pytest.raises(AssertionError):
            P.permuted_block_sparse_attn_fwd(q, k, v, **{**plain, **bad})
    for bad in ((q, k[:, :, :-1], v), (q, k[:, :1], v), (q[0], k[0], v[0]), (q.float(), k, v), (q[..., :64], k, v), (q[:, :3], k, v)):
        assert native(*bad, *plain.values()) is None
        with pytest.raises((AssertionError, ValueError, _lib.PbsHipError)):
            P.permuted_block_sparse_attn_fwd(*bad, **plain)
    assert native(q, k, v, *{**plain, "key_pool_mode": "median"}.values()) is None
    with pytest.raises(ValueError):
        P.permuted_block_sparse_attn_fwd(q, k, v, **{**plain, "key_pool_mode": "median"})


@pytest.mark.gpu
def test_under_capture_and_on_another_stream(dev):
    q, k, v = (x.to(dev) for x in small_case(1, 8, 2, 200, seed=9))
    want = ops.prefill_attn_fwd(q, k, v, 128, 256, 0.9)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        stream.wait_stream(torch.cuda.default_stream())
        assert torch.equal(P.permuted_block_sparse_attn_fwd(q, k, v, 128, 256, 0.9, True), want)
        with torch.cuda.graph(graph, stream=stream):
            out = P.permuted_block_sparse_attn_fwd(q, k, v, 128, 256, 0.9, True)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
