// Whole PBS prefill attention in one call: every stage enqueued on one stream out of one caller-provided
// workspace (no allocation, no synchronisation, one host round trip instead of ten).
#include "pbs_lists.h"

#include "../../include/pbs_hip.h"   // the stage entry points, type-checked against the public ABI

namespace {

__global__ void identity_indices_kernel(int32_t* idx, int S_pad, int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < total) idx[i] = (int32_t)(i % S_pad);
}

// Passes of few, short rows gather every block at once, in the launch that pools: a launch and a read of K less.  Whole pass, filtered gather
// after the selection -> this, us: 32 / 8 heads x 512 54.3 -> 51.1, x 1024 68.9 -> 64.4, x 4096 181 -> 175, x 8192 499 -> 488, on
// concentrated inputs 64.0 -> 59.8, 141 -> 139, 339 -> 333; 28 / 4 x 8192 218 -> 216.5.  Longer rows leave more of the blocks unvisited: 8 / 2
// heads x 16384, concentrated, 154.9 against 156.7, x 32768 263 against 279.
// (The same passes take estimate and selection in one launch: see estimate_select_kernel.)
constexpr int SHORT_PASS_BLOCKS = 2048, SHORT_PASS_ROW = PBS_ESTIMATE_SELECT_MAX_BLOCKS;
bool short_pass(int rows, int nb) { return nb <= SHORT_PASS_ROW && rows * nb <= SHORT_PASS_BLOCKS; }

// Short passes whose gather sorts its blocks' segments.
// Up to 256 keys, which a workgroup ranks.  Whole pass, sort kernel -> this, us: 28 / 4 heads x 1000 in segments of 256 61.0 -> 52.9, 32 / 8 x 1500
// 73.8 -> 67.5, x 8192 472.1 -> 468.7, of 128 474.5 -> 471.8, 28 / 4 x 300 41.7 -> 37.2, 8 x 16 / 16 x 600 84.2 -> 82.9.  From 256 heads on the other
// routes win: 32 x 8 / 2 x 300 79.5 against 80.6, 16 x 32 / 8 x 200 of 128 88.7 against 91.4.  Where the final scoring pass could sort: 28 / 4 x 3400 of 256
// 124.2 -> 121.3, 32 / 8 x 4096 162.4 -> 160.6, but not where a segment is less than what its workgroups take otherwise, so that it gains workgroups by
// sorting (4 / 1 x 6000 of 128 106.9 against 109.6).
// Longer ones, by the first wave, as long as the sorting workgroups are in flight at once: a segment's blocks all sort it, so that a second round of them is another
// sort behind the first.  Three run on a CU, twenty-four on a shader engine of eight, and the launch deals them to the engines in a fixed order, which short rows fill
// unevenly (pbs_sorts_of_an_engine).  Up to 24 on the fullest, us: 28 / 4 x 1100 of 512 66.7 -> 62.7; 32 / 8 x 2200 of 1024 110.7 -> 105.4, x 3000 133.8 -> 129.1; 365 shapes of up to
// 768 blocks 1.00 to 1.08 times as fast.  27 and more: 28 / 4 x 2139 of 640 104.6 against 112.4, 2 x 32 / 8 x 1115 of 1024 96.2 against 105.2, 4 x 16 / 16 x 1115 of 512 94.3
// against 97.2; 116 shapes 0.90 to 1.00.  Thirty-two keys a lane: 28 / 4 x 2500 of 2048 126 against 147.
constexpr int SORT_IN_GATHER_BLOCKS = 3 * 256, SORTS_OF_AN_ENGINE = 3 * 8, RANK_IN_GATHER_HEADS = 255;
bool sorts_in_gather(int B, int Hq, int Hkv, int S, int block_size, int segment_size, int score_sort_chunk) {
  if (segment_size <= PBS_RANKED_KEYS) return B * Hq <= RANK_IN_GATHER_HEADS && score_sort_chunk <= segment_size;
  const int nb = (S + block_size - 1) / block_size;
  return segment_size <= PBS_SORT_IN_GATHER_KEYS && B * Hq * nb <= SORT_IN_GATHER_BLOCKS &&
         pbs_sorts_of_an_engine(B, Hq, Hkv, nb, S / segment_size * (segment_size / block_size)) <= SORTS_OF_AN_ENGINE;
}

// Sort with the query pooling + key pooling, against sort + both poolings, us: 32768 tokens, 32 / 8 heads 52 + 23 against 20 + 60; 13333 tokens twice
// 51 + 19 against 13 + 57; 131072 tokens 208 + 91 against 36 + 247, where the key pooling alone has too little to do while it waits for its rows.
constexpr int RIDE_BLOCKS = 16384;

struct Layout {
  size_t scores, score_ws, idx, perm_k, perm_vt, pooled_k, pooled_q, probs, cols, cnt, needed, select_ws, attn_ws, total;
};

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

Layout make_layout(int B, int Hq, int Hkv, int S, int D, int block_size, int segment_size) {
  Layout L;
  const size_t rows = (size_t)B * Hq;
  const size_t nb = (size_t)(S + block_size - 1) / block_size, s_pad = nb * block_size;
  const size_t sc = (size_t)(S / segment_size) * segment_size;
  // one segment over the whole sequence: every tile comes from the caller's K and V, only the visit lists are needed
  const bool own_tiles_only = (size_t)segment_size >= s_pad;
  size_t off = 0;
  auto take = [&](size_t bytes) { const size_t o = off; off = align256(off + (own_tiles_only ? 0 : bytes)); return o; };
  L.scores = take(rows * sc * 4);
  L.score_ws = take(pbs_score_keys_workspace_bound(B, Hq, Hkv, S, segment_size));
  L.idx = take(rows * s_pad * 4);
  L.perm_k = take(rows * s_pad * D * 2);
  L.perm_vt = take(rows * s_pad * D * 2);
  L.pooled_k = take(rows * nb * D * 2);
  L.pooled_q = take(rows * nb * D * 2);
  L.probs = take(rows * nb * nb * 4);
  const bool csr = nb > PBS_PAIR_SELECT_MAX_BLOCKS;   // shorter rows: the selection writes the attention kernel's lists itself
  L.cols = take(csr ? rows * nb * nb * 4 : 0);
  L.cnt = take(csr ? rows * nb * 4 : 0);
  L.needed = take(rows * nb);
  L.select_ws = take(pbs_select_blocks_workspace_bytes((int)rows));
  L.attn_ws = off;
  L.total = align256(off + pbs_sparse_attn_workspace_bytes(B, Hq, S, segment_size));
  return L;
}

// A sequence that fits inside one segment is plain causal attention (pbs_attn/src/pbs.py:175-182): identity key
// order, every causal block visited.  With that order and every candidate selected the result does not depend on the
// segment size, so the kernels run with one segment spanning the sequence or, beyond the attention kernel's 511
// blocks per segment, with segments of 256 blocks.  Returns the segment size to run with.
int one_segment_size(int S, int block_size) {
  const int nb = (S + block_size - 1) / block_size;
  return (nb <= 511 ? nb : 256) * block_size;
}

}  // namespace

extern "C" int pbs_identity_indices(int32_t* key_indices, int rows, int S_pad, void* stream) {
  PBS_REQUIRE(key_indices && rows > 0 && S_pad > 0, "pbs_identity_indices: bad arguments");
  const int64_t total = (int64_t)rows * S_pad;
  hipLaunchKernelGGL(identity_indices_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     key_indices, S_pad, total);
  return pbs_check_launch("pbs_identity_indices");
}

extern "C" size_t pbs_prefill_attn_workspace_bytes(int B, int Hq, int Hkv, int S, int head_dim, int block_size, int segment_size) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || S <= 0 || head_dim <= 0 || block_size <= 0 || segment_size <= 0) return 0;
  if (S <= segment_size) segment_size = one_segment_size(S, block_size);   // as pbs_prefill_attn_fwd
  return make_layout(B, Hq, Hkv, S, head_dim, block_size, segment_size).total;
}

extern "C" int pbs_one_segment_attn_fwd(const void* q, const void* k, const void* v, void* out, int B, int Hq, int Hkv, int S,
                                        int head_dim, int block_size, int segment_size, int64_t q_sb, int64_t q_sh, int64_t q_ss,
                                        int64_t k_sb, int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss,
                                        int64_t o_sb, int64_t o_sh, int64_t o_ss, float softmax_scale, void* stream) {
  PBS_REQUIRE(q && k && v && out, "pbs_one_segment_attn_fwd: null tensor pointer");
  PBS_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && S > 0, "pbs_one_segment_attn_fwd: bad shape");
  PBS_REQUIRE(block_size > 0 && segment_size > 0 && segment_size % block_size == 0,
              "pbs_one_segment_attn_fwd: segment_size must be a multiple of block_size");
  if (S > segment_size || (S + block_size - 1) / block_size > 511 || !pbs_sparse_attn_forms_lists(B, Hq, S, block_size))
    return PBS_NOT_ONE_LAUNCH;
  // (permuted tiles: none is listed, any aligned address will do)
  return pbs_sparse_attn_launch(q, q, q, k, v, nullptr, nullptr, false, out, B, Hq, Hkv, S, head_dim, block_size,
                                one_segment_size(S, block_size), q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss,
                                softmax_scale, nullptr, nullptr, stream);
}

extern "C" int pbs_prefill_attn_fwd(const void* q, const void* k, const void* v, void* out, int B, int Hq, int Hkv, int S,
                                    int head_dim, int block_size, int segment_size, int64_t q_sb, int64_t q_sh,
                                    int64_t q_ss, int64_t k_sb, int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh,
                                    int64_t v_ss, int64_t o_sb, int64_t o_sh, int64_t o_ss, float threshold,
                                    const float* threshold_per_row, int threshold_is_int_one,
                                    int force_select_first_block, int query_pool_max, int key_pool_max,
                                    float softmax_scale, void* workspace, size_t workspace_bytes, void* stream) {
  PBS_REQUIRE(q && k && v && out, "pbs_prefill_attn_fwd: null tensor pointer");
  PBS_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && S > 0, "pbs_prefill_attn_fwd: bad shape");
  PBS_REQUIRE(block_size > 0 && segment_size > 0 && segment_size % block_size == 0,
              "pbs_prefill_attn_fwd: segment_size must be a multiple of block_size");
  // sequences that fit one segment: plain causal attention = one segment spanning the sequence,
  // identity order, every causal block visited
  const bool one_segment = S <= segment_size;
  if (one_segment) {
    segment_size = one_segment_size(S, block_size);
    threshold_is_int_one = 1;
  }
  // checked here, before anything is enqueued (the attention kernel holds one segment's blocks in its list)
  PBS_REQUIRE(segment_size / block_size <= 511,
              "pbs_prefill_attn_fwd: a segment of %d blocks exceeds the limit of 511 (use a smaller segment_size)",
              segment_size / block_size);
  const Layout L = make_layout(B, Hq, Hkv, S, head_dim, block_size, segment_size);
  PBS_REQUIRE(workspace && workspace_bytes >= L.total, "pbs_prefill_attn_fwd: workspace too small (%zu < %zu bytes)",
              workspace_bytes, L.total);
  PBS_REQUIRE(((uintptr_t)workspace % 256) == 0, "pbs_prefill_attn_fwd: workspace must be 256-byte aligned");
  uint8_t* w = (uint8_t*)workspace;
  const int rows = B * Hq, nb = (S + block_size - 1) / block_size, s_pad = nb * block_size;
  const int nseg = S / segment_size, rem = S % segment_size;
  // the launch limits of the stages, whether or not this call needs them all
  PBS_REQUIRE(rows <= 65535, "pbs_prefill_attn_fwd: too many heads (%d)", rows);
  PBS_REQUIRE(Hq / Hkv * 8 <= 65535 && ((int64_t)B * Hkv * ((nb + 7) / 8) + 7) / 8 <= 65535,
              "pbs_prefill_attn_fwd: too many heads or blocks");
  int rc;
  // A sequence inside one segment of the kernel's size needs no permuted tile, hence no order, no gather and no
  // selection: the attention launch, behind the list kernel's where there are more items than workgroups (32 / 8 heads x 77 tokens,
  // before one block had a kernel of its own: six launches 32.2 us, two 20.7, one 17.1).  (Permuted tiles: none is listed, any aligned address will do.)
  const bool own_tiles_only = segment_size >= s_pad;
  if (own_tiles_only)
    return pbs_sparse_attn_launch(q, w, w, k, v, nullptr, nullptr, false, out, B, Hq, Hkv, S, head_dim, block_size, segment_size, q_sb,
                                  q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss, softmax_scale, nullptr,
                                  w + L.attn_ws, stream);
  const bool is_short = !threshold_is_int_one && short_pass(rows, nb);
  SegmentScores scores = {};   // of a gather that sorts
  bool q_pooled = false;   // the query blocks' pooling is under way
  if (one_segment || nseg == 0 || (nseg == 1 && rem == 0)) {
    if ((rc = pbs_identity_indices((int32_t*)(w + L.idx), rows, s_pad, stream))) return rc;
  } else if (is_short && sorts_in_gather(B, Hq, Hkv, S, block_size, segment_size, pbs_score_sort_chunk(B, Hq, Hkv, S, segment_size))) {
    scores = {(const float*)(w + L.scores), (int32_t*)(w + L.select_ws), nseg * segment_size, segment_size};
    if ((rc = pbs_score_keys(q, k, (float*)(w + L.scores), B, Hq, Hkv, S, head_dim, block_size, segment_size, q_sb, q_sh,
                             q_ss, k_sb, k_sh, k_ss, w + L.score_ws, L.idx - L.score_ws, stream))) return rc;
  } else if (pbs_score_sort_chunk(B, Hq, Hkv, S, segment_size)) {
    if ((rc = pbs_score_sort_launch(q, k, (int32_t*)(w + L.idx), (int32_t*)(w + L.select_ws), B, Hq, Hkv, S, s_pad, head_dim, block_size,
                                    segment_size, q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, w + L.score_ws, L.idx - L.score_ws, stream))) return rc;
  } else {
    if ((rc = pbs_score_keys(q, k, (float*)(w + L.scores), B, Hq, Hkv, S, head_dim, block_size, segment_size, q_sb, q_sh,
                             q_ss, k_sb, k_sh, k_ss, w + L.score_ws, L.idx - L.score_ws, stream))) return rc;
    // the query pooling rides with the sort, which leaves the memory idle (see RIDE_BLOCKS)
    const bool ride = !threshold_is_int_one && !is_short && rows * nb <= RIDE_BLOCKS && pbs_segment_argsort_takes_ride(segment_size);
    const PoolQ pooling = {(const uint16_t*)q, (uint16_t*)(w + L.pooled_q), q_sb, q_sh, q_ss, query_pool_max, Hq, S, nb};
    if ((rc = pbs_segment_argsort_launch((const float*)(w + L.scores), (int32_t*)(w + L.idx), (int32_t*)(w + L.select_ws), block_size,
                                         rows, S, s_pad, segment_size, stream, ride ? pooling : PoolQ{}))) return rc;
    q_pooled = ride;
  }
  // With a real threshold the permuted K / V are gathered AFTER the selection, and only the blocks some query
  // block visits: the estimate needs no more than the pooled permuted key blocks, which come straight from K.
  // (Short passes: see short_pass.)
  // (Every candidate selected: everything is visited, one full gather.)
  uint8_t* needed = threshold_is_int_one || is_short ? nullptr : w + L.needed;
  const bool pair_lists = !threshold_is_int_one && nb <= PBS_PAIR_SELECT_MAX_BLOCKS;
  if (threshold_is_int_one) {
    if ((rc = pbs_gather_kv(k, v, (const int32_t*)(w + L.idx), w + L.perm_k, w + L.perm_vt, nullptr, B, Hq, Hkv,
                            S, head_dim, block_size, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, key_pool_max, nullptr, stream))) return rc;
  } else {
    if (is_short) {
      if ((rc = pbs_gather_pool_launch(q, k, v, (const int32_t*)(w + L.idx), w + L.pooled_q, w + L.pooled_k, w + L.perm_k, w + L.perm_vt, B, Hq,
                                       Hkv, S, head_dim, block_size, q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss,
                                       query_pool_max, key_pool_max, stream, scores))) return rc;
    } else if (q_pooled) {
      if ((rc = pbs_pool_k_permuted(k, (const int32_t*)(w + L.idx), w + L.pooled_k, needed, B, Hq, Hkv, S, head_dim, block_size, k_sb, k_sh,
                                    k_ss, key_pool_max, stream))) return rc;
    } else if ((rc = pbs_pool_blocks(q, k, (const int32_t*)(w + L.idx), w + L.pooled_q, w + L.pooled_k, needed, B, Hq, Hkv, S,
                                     head_dim, block_size, q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, query_pool_max, key_pool_max,
                                     stream))) return rc;
    if (is_short) {
      if ((rc = pbs_estimate_select_pair_lists(w + L.pooled_q, w + L.pooled_k, Candidates::EARLIER_SEGMENTS, threshold_per_row, threshold,
                                               force_select_first_block != 0, (const int32_t*)(w + L.select_ws), rows, S, head_dim,
                                               block_size, segment_size, needed,
                                               pbs_pair_lists(B, Hq, Hkv, S, block_size, segment_size, w + L.attn_ws), stream))) return rc;
    // (the selection into pair lists reads a row's candidate entries only: the others are not written)
    } else if (pair_lists) {
      if ((rc = pbs_block_logits_softmax_candidates_only(w + L.pooled_q, w + L.pooled_k, (float*)(w + L.probs), rows, nb,
                                                         head_dim, segment_size / block_size, stream))) return rc;
      if ((rc = pbs_select_pair_lists((const float*)(w + L.probs), Candidates::EARLIER_SEGMENTS, threshold_per_row, threshold,
                                      force_select_first_block != 0, (const int32_t*)(w + L.select_ws), rows, S, block_size,
                                      segment_size, needed,
                                      pbs_pair_lists(B, Hq, Hkv, S, block_size, segment_size, w + L.attn_ws), stream))) return rc;
    } else {
      if ((rc = pbs_block_logits_softmax(w + L.pooled_q, w + L.pooled_k, (float*)(w + L.probs), rows, nb, head_dim,
                                         segment_size / block_size, stream))) return rc;
      if ((rc = pbs_select_blocks((const float*)(w + L.probs), threshold_per_row, threshold, /*threshold_is_int_one=*/0,
                                  force_select_first_block, /*candidate_rule=*/1, (const int32_t*)(w + L.idx), rows, S, block_size,
                                  segment_size, nullptr, nullptr, (int32_t*)(w + L.cols), (int32_t*)(w + L.cnt), needed,
                                  w + L.select_ws, L.attn_ws - L.select_ws, stream))) return rc;
    }
    if (!is_short)
      if ((rc = pbs_gather_kv(k, v, (const int32_t*)(w + L.idx), w + L.perm_k, w + L.perm_vt, nullptr, B, Hq, Hkv,
                              S, head_dim, block_size, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, key_pool_max, needed, stream))) return rc;
  }
  // (every candidate selected: the lists follow from the block numbers)
  const int32_t* cols = threshold_is_int_one || pair_lists ? nullptr : (const int32_t*)(w + L.cols);
  return pbs_sparse_attn_launch(q, w + L.perm_k, w + L.perm_vt, k, v, cols, (const int32_t*)(w + L.cnt), pair_lists, out, B, Hq, Hkv, S,
                                head_dim, block_size, segment_size, q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb,
                                o_sh, o_ss, softmax_scale, nullptr, w + L.attn_ws, stream);
}

// ---- the un-permuted MeanPooling mode (pbs_attn/baselines/MeanPooling.py) in one call: pooled blocks in their own order, every block up to
// the diagonal one a candidate, all tiles read in place from K and V
namespace {

struct MeanPoolingLayout {
  size_t pooled_k, pooled_q, probs, attn_ws, total;
};
MeanPoolingLayout meanpooling_layout(int B, int Hq, int S, int D, int block_size) {
  MeanPoolingLayout L;
  const size_t rows = (size_t)B * Hq, nb = (size_t)(S + block_size - 1) / block_size;
  size_t off = 0;
  auto take = [&](size_t bytes) { const size_t o = off; off = align256(off + bytes); return o; };
  L.pooled_k = take(rows * nb * D * 2);
  L.pooled_q = take(rows * nb * D * 2);
  L.probs = take(short_pass((int)rows, (int)nb) ? 0 : rows * nb * nb * 4);
  L.attn_ws = off;
  L.total = align256(off + pbs_sparse_attn_workspace_bytes(B, Hq, S, block_size));
  return L;
}

}  // namespace

extern "C" size_t pbs_meanpooling_attn_workspace_bytes(int B, int Hq, int Hkv, int S, int head_dim, int block_size) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || S <= 0 || head_dim <= 0 || block_size <= 0) return 0;
  return meanpooling_layout(B, Hq, S, head_dim, block_size).total;
}

extern "C" int pbs_meanpooling_attn_fwd(const void* q, const void* k, const void* v, void* out, int B, int Hq, int Hkv, int S,
                                        int head_dim, int block_size, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t k_sb,
                                        int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss, int64_t o_sb,
                                        int64_t o_sh, int64_t o_ss, float threshold, const float* threshold_per_row,
                                        int force_select_first_block, float softmax_scale, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  PBS_REQUIRE(q && k && v && out, "pbs_meanpooling_attn_fwd: null tensor pointer");
  PBS_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && S > 0 && block_size > 0, "pbs_meanpooling_attn_fwd: bad shape");
  const int rows = B * Hq, nb = (S + block_size - 1) / block_size;
  PBS_REQUIRE(rows <= 65535, "pbs_meanpooling_attn_fwd: too many heads (%d)", rows);
  // the launch limit of the pooling, whether or not this call needs it
  PBS_REQUIRE(Hq / Hkv * 16 <= 65535, "pbs_meanpooling_attn_fwd: too many heads or blocks");
  PBS_REQUIRE(nb <= PBS_PAIR_SELECT_MAX_BLOCKS, "pbs_meanpooling_attn_fwd: more than %d blocks per sequence (%d)", PBS_PAIR_SELECT_MAX_BLOCKS, nb);
  const MeanPoolingLayout L = meanpooling_layout(B, Hq, S, head_dim, block_size);
  PBS_REQUIRE(workspace && workspace_bytes >= L.total && ((uintptr_t)workspace % 256) == 0,
              "pbs_meanpooling_attn_fwd: workspace must be a 256-byte aligned device buffer of %zu bytes", L.total);
  uint8_t* w = (uint8_t*)workspace;
  // one block a row: its own, always selected (32 / 8 heads x 100 tokens 20.6 -> 5.3 us, 16 x 32 / 8 x 128 42.9 -> 20.8)
  if (nb == 1)
    return pbs_sparse_attn_launch(q, q, q, k, v, nullptr, nullptr, false, out, B, Hq, Hkv, S, head_dim, block_size, block_size, q_sb, q_sh, q_ss,
                                  k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss, softmax_scale, nullptr, w + L.attn_ws, stream);
  int rc;
  if ((rc = pbs_pool_blocks_launch(q, k, nullptr, w + L.pooled_q, w + L.pooled_k, nullptr, B, Hq, Hkv, S, head_dim, block_size, q_sb, q_sh,
                                   q_ss, k_sb, k_sh, k_ss, 0, 0, stream))) return rc;
  const PairLists lists = pbs_pair_lists(B, Hq, Hkv, S, block_size, block_size, w + L.attn_ws);
  if (short_pass(rows, nb)) {
    if ((rc = pbs_estimate_select_pair_lists(w + L.pooled_q, w + L.pooled_k, Candidates::UP_TO_DIAGONAL, threshold_per_row, threshold,
                                             force_select_first_block != 0, nullptr, rows, S, head_dim, block_size, block_size, nullptr,
                                             lists, stream))) return rc;
  } else {
    if ((rc = pbs_block_logits_softmax_causal_candidates(w + L.pooled_q, w + L.pooled_k, (float*)(w + L.probs), rows, nb, head_dim, stream))) return rc;
    if ((rc = pbs_select_pair_lists((const float*)(w + L.probs), Candidates::UP_TO_DIAGONAL, threshold_per_row, threshold,
                                    force_select_first_block != 0, nullptr, rows, S, block_size, block_size, nullptr, lists, stream))) return rc;
  }
  // (permuted tiles: none is listed, any aligned address will do)
  return pbs_sparse_attn_launch(q, q, q, k, v, nullptr, nullptr, true, out, B, Hq, Hkv, S, head_dim, block_size, block_size, q_sb, q_sh, q_ss,
                                k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss, softmax_scale, nullptr, w + L.attn_ws, stream);
}
