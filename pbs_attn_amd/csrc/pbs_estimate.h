// The block estimate of 32 query blocks of one head by a workgroup of four waves: see pbs_estimate.hip.
#pragma once
#include "pbs_common.h"
#include "pbs_div.h"

namespace {

constexpr int ESTIMATE_D = 128;

__device__ __forceinline__ bf16x8 load_frag(const uint16_t* row_ptr, int t, int half) {
  return *reinterpret_cast<const bf16x8*>(row_ptr + 16 * t + 8 * half);
}
// two accumulators -> the logits a bf16 matmul followed by a bf16 division by sqrt(D) yields: round to bf16, divide
// (the exact quotient, see pbs_div.h), round to bf16
struct Divisor {
  float b, y;   // sqrt(D) and its correctly rounded reciprocal
};
inline Divisor pbs_sqrt_divisor(int head_dim) {
  const float b = (float)__builtin_sqrt((double)head_dim);
  return {b, (float)(1.0 / (double)b)};   // the correctly rounded reciprocal for head_dim 128 (tests/c_abi/div_check.c)
}
__device__ __forceinline__ f32x2 logit_round2(float acc0, float acc1, Divisor d) {
  const f32x2 r = hw_round_bf16x2((f32x2){acc0, acc1});
  return hw_round_bf16x2((f32x2){pbs_div_by_const(r.x, d.b, d.y), pbs_div_by_const(r.y, d.b, d.y)});
}

// number of candidate key blocks of query block qb (its candidates are key blocks 0 .. count - 1): the blocks
// of strictly earlier segments, or -- CAUSAL, the rule of the reference's un-permuted MeanPooling baseline --
// every block up to and including the diagonal one
template <bool CAUSAL>
__device__ __forceinline__ int candidate_count(int qb, int bps) {
  return CAUSAL ? qb + 1 : (qb / bps) * bps;
}

struct EstimateStats {   // in LDS
  float m[4][32], l[4][32];
  float max[32], inv[32];
};
// The probabilities of query blocks 32 qt .. 32 qt + 31, one after the other to sink(query block in the tile, key block, probability).
// CANDIDATES_ONLY: only those of candidates; otherwise of all nb key blocks, zeros outside the candidates and NaN rows where
// there are none.  pq, pk: the head's pooled query and key blocks.  ONE_TILE: up to 128 key blocks, a tile of 32 a wave, whose fragments
// serve both passes.
template <bool CAUSAL, bool CANDIDATES_ONLY, bool ONE_TILE = false, class Sink>
__device__ __forceinline__ void estimate_tile(const uint16_t* pq, const uint16_t* pk, int nb, int bps, Divisor sqrt_d, int qt,
                                              EstimateStats& st, Sink sink) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = lane & 31, half = lane >> 5;
  const int q_last = min(32 * qt + 31, nb - 1);
  const int cand_max = candidate_count<CAUSAL>(q_last, bps);   // candidates of the tile's last row
  const int n_kt_cand = (cand_max + 31) / 32;
  const int n_kt_all = (nb + 31) / 32;

  bf16x8 qf[8], kf[8];
  auto load_keys = [&](int kt) __attribute__((always_inline)) {
    const uint16_t* row = pk + (int64_t)min(32 * kt + j, nb - 1) * ESTIMATE_D;
#pragma unroll
    for (int t = 0; t < 8; ++t) kf[t] = load_frag(row, t, half);
  };
  {
    const uint16_t* row = pq + (int64_t)min(32 * qt + j, nb - 1) * ESTIMATE_D;
#pragma unroll
    for (int t = 0; t < 8; ++t) qf[t] = load_frag(row, t, half);
  }

  // ---- pass A: per query block (column j) running max / sum over its candidates
  const int qb_col = 32 * qt + j;
  const int cand_col = qb_col < nb ? candidate_count<CAUSAL>(qb_col, bps) : 0;
  float m_run = -INFINITY, l_run = 0.f;
  for (int kt = wave; kt < n_kt_cand; kt += 4) {
    load_keys(kt);
    f32x16 acc = {0};
#pragma unroll
    for (int t = 0; t < 8; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[t], qf[t], acc, 0, 0, 0);
    float v[16], mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      const int kb = 32 * kt + 8 * (r >> 2) + 4 * half + (r & 3);
      const f32x2 l2 = logit_round2(acc[r], acc[r + 1], sqrt_d);
      v[r] = kb < cand_col ? l2.x : -INFINITY;
      v[r + 1] = kb + 1 < cand_col ? l2.y : -INFINITY;
      mx = fmaxf(mx, fmaxf(v[r], v[r + 1]));
    }
    if (mx > -INFINITY) {
      const float m_new = fmaxf(m_run, mx);
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) sum += __expf(v[r] - m_new);
      l_run = l_run * __expf(m_run - m_new) + sum;
      m_run = m_new;
    }
  }
  {
    const float m_o = xhalf_f32(m_run), l_o = xhalf_f32(l_run);
    const float m_new = fmaxf(m_run, m_o);
    float l_new = 0.f;
    if (m_new > -INFINITY) l_new = l_run * __expf(m_run - m_new) + l_o * __expf(m_o - m_new);
    if (half == 0) {
      st.m[wave][j] = m_new;
      st.l[wave][j] = l_new;
    }
  }
  __syncthreads();
  if (threadIdx.x < 32) {
    float m = -INFINITY, l = 0.f;
    for (int w = 0; w < 4; ++w) m = fmaxf(m, st.m[w][threadIdx.x]);
    if (m > -INFINITY)
      for (int w = 0; w < 4; ++w) l += st.l[w][threadIdx.x] * __expf(st.m[w][threadIdx.x] - m);
    st.max[threadIdx.x] = m;
    st.inv[threadIdx.x] = 1.0f / l;
  }
  __syncthreads();

  // ---- pass B: rows = query blocks, column = key block j of tile kt
  for (int kt = wave; kt < (CANDIDATES_ONLY ? n_kt_cand : n_kt_all); kt += 4) {
    const int kb = 32 * kt + j;
    f32x16 acc = {0};
    if (kt < n_kt_cand) {
      if (!ONE_TILE) load_keys(kt);
#pragma unroll
      for (int t = 0; t < 8; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[t], kf[t], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      const f32x2 l2 = logit_round2(acc[r], acc[r + 1], sqrt_d);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int ql = 8 * (r >> 2) + 4 * half + (r & 3) + u;
        const int qb = 32 * qt + ql;
        if (qb < nb && kb < nb) {
          const int cand = candidate_count<CAUSAL>(qb, bps);
          float p;
          if (cand == 0) p = __uint_as_float(0x7fc00000u);
          else if (kb < cand) p = __expf((u ? l2.y : l2.x) - st.max[ql]) * st.inv[ql];
          else p = 0.f;
          if (!CANDIDATES_ONLY || kb < cand) sink(ql, kb, p);
        }
      }
    }
  }
}

}  // namespace
