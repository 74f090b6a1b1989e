// Block-importance estimation: softmax over strictly-earlier-segment key blocks of
// the pooled-Q x pooled-K logits.
//
//   logit[qb, kb] = bf16( bf16(<Pq[qb], Pk[kb]>) / sqrt(D) )      kb < first block of qb's segment
//   P[qb, :]      = softmax_fp32(logit[qb, :])                     (0 outside the candidates)
// Rows with no candidate (query blocks of segment 0) are NaN, as a softmax over an
// all -inf row is.  One workgroup owns 32 query blocks of one head; its four
// waves split the key-block tiles, first to find each row's (max, sum), then to
// recompute the logits and write P with 128-byte row segments per store.
#include "pbs_estimate.h"
#include "pbs_lists.h"
#include "../../include/pbs_hip.h"   // the definitions below are checked against the public declarations

namespace {

constexpr int D = ESTIMATE_D;

// CANDIDATES_ONLY: only the candidate entries of a row are written (the selection that follows on the single-call path
// reads no others); otherwise all nb columns, zeros outside the candidates and NaN rows where there are none.
template <bool CAUSAL, bool CANDIDATES_ONLY>
__global__ __launch_bounds__(256) void block_logits_softmax_kernel(const uint16_t* pooled_q, const uint16_t* pooled_k,
                                                                   float* P, int nb, int bps, Divisor sqrt_d) {
  __shared__ EstimateStats st;
  const int qt = (int)gridDim.x - 1 - (int)blockIdx.x, bh = blockIdx.y;   // the tiles with the most candidates start first
  float* out = P + ((int64_t)bh * nb + 32 * qt) * nb;
  estimate_tile<CAUSAL, CANDIDATES_ONLY>(pooled_q + (int64_t)bh * nb * D, pooled_k + (int64_t)bh * nb * D, nb, bps, sqrt_d, qt, st,
                                         [&](int ql, int kb, float p) __attribute__((always_inline)) { out[(int64_t)ql * nb + kb] = p; });
}

}  // namespace

namespace {
int launch_block_logits(const char* who, bool causal, bool candidates_only, const void* pooled_q, const void* pooled_k, float* block_attn_scores,
                        int rows, int nb, int head_dim, int blocks_per_segment, void* stream) {
  PBS_REQUIRE(pooled_q && pooled_k && block_attn_scores, "%s: null tensor pointer", who);
  PBS_REQUIRE(head_dim == D, "%s: head_dim must be 128, got %d", who, head_dim);
  PBS_REQUIRE(rows > 0 && rows <= 65535 && nb > 0 && blocks_per_segment > 0, "%s: bad shape", who);
  const dim3 grid((nb + 31) / 32, rows);
  const Divisor sqrt_d = pbs_sqrt_divisor(head_dim);
  if (candidates_only && causal)
    hipLaunchKernelGGL((block_logits_softmax_kernel<true, true>), grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)pooled_q,
                       (const uint16_t*)pooled_k, block_attn_scores, nb, blocks_per_segment, sqrt_d);
  else if (candidates_only)
    hipLaunchKernelGGL((block_logits_softmax_kernel<false, true>), grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)pooled_q,
                       (const uint16_t*)pooled_k, block_attn_scores, nb, blocks_per_segment, sqrt_d);
  else if (causal)
    hipLaunchKernelGGL((block_logits_softmax_kernel<true, false>), grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)pooled_q,
                       (const uint16_t*)pooled_k, block_attn_scores, nb, blocks_per_segment, sqrt_d);
  else
    hipLaunchKernelGGL((block_logits_softmax_kernel<false, false>), grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)pooled_q,
                       (const uint16_t*)pooled_k, block_attn_scores, nb, blocks_per_segment, sqrt_d);
  return pbs_check_launch(who);
}
}  // namespace

extern "C" int pbs_block_logits_softmax(const void* pooled_q, const void* pooled_k, float* block_attn_scores, int rows,
                                        int nb, int head_dim, int blocks_per_segment, void* stream) {
  return launch_block_logits("pbs_block_logits_softmax", false, false, pooled_q, pooled_k, block_attn_scores, rows, nb, head_dim,
                             blocks_per_segment, stream);
}

extern "C" int pbs_block_logits_softmax_causal(const void* pooled_q, const void* pooled_k, float* block_attn_scores,
                                               int rows, int nb, int head_dim, void* stream) {
  return launch_block_logits("pbs_block_logits_softmax_causal", true, false, pooled_q, pooled_k, block_attn_scores, rows, nb,
                             head_dim, 1, stream);
}

int pbs_block_logits_softmax_causal_candidates(const void* pooled_q, const void* pooled_k, float* block_attn_scores, int rows, int nb,
                                               int head_dim, void* stream) {
  return launch_block_logits("pbs_block_logits_softmax_causal", true, true, pooled_q, pooled_k, block_attn_scores, rows, nb, head_dim, 1, stream);
}

extern "C" int pbs_block_logits_softmax_candidates_only(const void* pooled_q, const void* pooled_k, float* block_attn_scores, int rows,
                                             int nb, int head_dim, int blocks_per_segment, void* stream) {
  return launch_block_logits("pbs_block_logits_softmax", false, true, pooled_q, pooled_k, block_attn_scores, rows, nb, head_dim,
                             blocks_per_segment, stream);
}
