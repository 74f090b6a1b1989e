"""The workloads that PBS-Attn's prefill path is timed on, through its public entry points.

A case is one attention layer of a prompt: the factories that the Hugging Face patch installs
(``get_permuted_block_sparse_attn_fwd``, ``get_meanpooling_prefill``) build the prefill function once, and a pass calls
it on the layer's Q, K and V.  ``op``:

``pbs``          the permuted block-sparse attention call alone
``meanpooling``  the un-permuted MeanPooling mode on the same tensors
``rope_pbs``     what the patched forward does between the projections and the output projection: rotary embedding
                 of Q and K, then the attention call

Values come from the repository's own generators (``pbs_attn_amd/synth.py``): ``uniform_heavy``, ``span_heavy`` and
``local_window`` give near-uniform attention (most blocks are visited, the matrix cores are the bound);
``strong_heavy`` and ``strong_uniform`` give attention with few heavy keys (few blocks are visited, and the scoring,
sorting, pooling and selection weigh as much as the attention kernel).
"""
import math

import torch

from pbs_attn_amd import ops, synth
from pbs_attn_amd.patch.huggingface import get_meanpooling_prefill, get_permuted_block_sparse_attn_fwd

BLOCK = 128
HEAD_DIM = 128
NEAR_UNIFORM = ("uniform_heavy", "span_heavy", "local_window")
STRONG = ("strong_heavy", "strong_uniform")


def _case(**kw):
    c = dict(op="pbs", B=1, Hq=32, Hkv=8, S=4096, kind="uniform_heavy", segment=256, threshold=0.9,
             query_pool="mean", key_pool="mean", layout="bhsd")
    c.update(kw)
    return c


def listed():
    return [
        # a chat turn of a few dozen tokens: the patched model sends every prompt through the path, and one that fits
        # in a segment is plain causal attention; Q, K and V as the projections produce them (batch, token, head, d)
        _case(name="chat_77", S=77, layout="bshd"),
        # a short prompt of a 28 / 4 head model, just past the first permuted segments, ragged
        _case(name="prompt_1000", S=1000, Hq=28, Hkv=4, layout="bshd"),
        # a page or two of text: the 4k correctness workload of the repository
        _case(name="prompt_4k", S=4096),
        # two ragged prompts padded to one length, per-head thresholds (a float32 tensor), max pooling of both sides,
        # heavy keys scattered through the text
        _case(name="ragged_13333_max", B=2, S=13333, kind="strong_uniform", segment=512, threshold="per_head",
              query_pool="max", key_pool="max", layout="bshd"),
        # a batch of four 16k documents on a 28 / 4 head model with local attention
        _case(name="batch4_16k", B=4, Hq=28, Hkv=4, S=16384, kind="local_window"),
        # the un-permuted ablation at 16k: candidates up to the diagonal, one block per segment
        _case(name="meanpooling_16k", op="meanpooling", S=16384, segment=1024),
        # the 32k workload: a document that fills a common context window
        _case(name="prompt_32k", S=32768),
        # the same length where attention is concentrated
        _case(name="prompt_32k_sparse", S=32768, kind="strong_heavy", segment=1024),
        # one layer of the time-to-first-token workload (64k prompt), rotary embedding included
        _case(name="rope_layer_64k", op="rope_pbs", S=65536, layout="bshd"),
        # a long repository or book, near-uniform attention: the largest dense-regime pass
        _case(name="prompt_128k", S=131072, kind="span_heavy", segment=1024),
        # the same length with concentrated attention
        _case(name="prompt_128k_sparse", S=131072, kind="strong_heavy", segment=1024),
        # one GPU's heads of a 256k prompt under four-way tensor parallelism: more than 1024 blocks per row
        _case(name="shard_256k", Hq=8, Hkv=2, S=262144, kind="strong_uniform", segment=1024),
    ]


def draw(rng):
    """One more case: any length from a few dozen tokens to 128k (a head shard up to 256k), any of the head groupings, segment sizes,
    thresholds, pooling modes and value generators in use; never more work than the 128k dense listed case."""
    Hq, Hkv = rng.choice([(32, 8), (32, 8), (28, 4), (8, 2), (4, 1), (16, 16)])
    kind = rng.choice(NEAR_UNIFORM + STRONG)
    op = rng.choices(["pbs", "rope_pbs", "meanpooling"], [6, 2, 1])[0]
    S = int(math.exp(rng.uniform(math.log(33), math.log(262144))))
    if rng.random() < 0.4:
        S = max(BLOCK, S // BLOCK * BLOCK)
    B = rng.choice([1, 1, 1, 2, 4])
    most = 32 * 131072.0 ** 2 * 0.7      # (heads x length^2) of the largest listed case, less for the odd block counts
    while B * Hq * float(S) ** 2 > most:
        if B > 1:
            B //= 2
        else:
            S = int(S * 0.71)
    return _case(op=op, B=B, Hq=Hq, Hkv=Hkv, S=S, kind=kind,
                 segment=rng.choice([128, 256, 256, 512, 1024, 1024, 2048]),
                 threshold=rng.choice([0.8, 0.9, 0.9, 0.95, "per_head", 1]) if op != "meanpooling" else rng.choice([0.8, 0.9]),
                 query_pool=rng.choice(["mean", "mean", "max"]), key_pool=rng.choice(["mean", "mean", "max"]),
                 layout=rng.choice(["bhsd", "bshd"]))


def _project_layout(x):
    """The memory order of a projection's output: (batch, token, head, d), seen as (batch, head, token, d)."""
    return x.transpose(1, 2).contiguous().transpose(1, 2)


def prepare(case, seed):
    B, Hq, Hkv, S = case["B"], case["Hq"], case["Hkv"], case["S"]
    q, k, v = synth.make_qkv(B, Hq, Hkv, S, HEAD_DIM, case["kind"], seed, "cuda")
    if case["layout"] == "bshd":
        q, k, v = _project_layout(q), _project_layout(k), _project_layout(v)
    threshold = case["threshold"]
    if threshold == "per_head":
        threshold = torch.linspace(0.8, 0.95, B * Hq, device="cuda").view(B, Hq)
    if case["op"] == "meanpooling":
        prefill = get_meanpooling_prefill(block_size=BLOCK, segment_size=case["segment"], threshold=threshold)
    else:
        prefill = get_permuted_block_sparse_attn_fwd(block_size=BLOCK, segment_size=case["segment"], threshold=threshold,
                                                     query_pool_mode=case["query_pool"], key_pool_mode=case["key_pool"])
    state = dict(q=q, k=k, v=v, prefill=prefill, rope=None)
    if case["op"] == "rope_pbs":
        inv_freq = 1.0 / (500000.0 ** (torch.arange(0, HEAD_DIM, 2, device="cuda").float() / HEAD_DIM))
        angle = torch.arange(S, device="cuda").float()[:, None] * inv_freq[None, :]
        angle = torch.cat((angle, angle), dim=-1)[None]
        state["rope"] = (angle.cos().to(torch.bfloat16), angle.sin().to(torch.bfloat16))
    return state


def run(state):
    q, k, v = state["q"], state["k"], state["v"]
    if state["rope"] is None:
        return state["prefill"](q, k, v)
    q, k = ops.rope_qk(q, k, *state["rope"])
    return {"q": q, "k": k, "out": state["prefill"](q, k, v)}


def work(case):
    """Q, K, V in and the output out once (with the rotary embedding also the embedded Q and K), and the matrix
    products of the tokens a pass has to visit: the causal part of each query's own segment and, of the earlier
    segments, about the threshold's share where attention is near-uniform and next to nothing where it is
    concentrated (the first block only; with the threshold 1 everything), plus one product of the last 128 queries with all keys."""
    B, Hq, Hkv, S = case["B"], case["Hq"], case["Hkv"], case["S"]
    thr = 0.875 if case["threshold"] == "per_head" else float(case["threshold"])
    seg = BLOCK if case["op"] == "meanpooling" else case["segment"]
    whole, rest = divmod(S, seg)
    own = whole * seg * (seg + 1) / 2 + rest * (rest + 1) / 2
    earlier = S * (S + 1) / 2 - own
    if case["kind"] in NEAR_UNIFORM or thr >= 1:
        earlier *= thr
    else:
        earlier = min(earlier, float(max(S - seg, 0)) * BLOCK)
    flops = 4.0 * HEAD_DIM * B * Hq * (own + earlier)
    if S > seg and thr < 1:
        flops += 2.0 * HEAD_DIM * BLOCK * B * Hq * S
    rows = (2 * Hq + 2 * Hkv) + ((Hq + Hkv) if case["op"] == "rope_pbs" else 0)
    return {"bytes": float(B * rows * S * HEAD_DIM * 2), "flops": flops}


def tolerance(case):
    """Measured against the same path with its scores, pools and block probabilities from float32 products in another
    order and its attention in float32 on the resulting mask: 1.8e-3 .. 2.3e-3 (the rounding of the probabilities and of
    the output to bf16) and 3.2e-3 where a near tie at a block's threshold fell the other way.  Stated: about three times the latter."""
    return {"rel": 1e-2}
