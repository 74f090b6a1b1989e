// Cumulative-threshold block selection and CSR emission.
//
// One workgroup per (head, query block) row of the block-probability matrix:
//   * NaN -> 0, stable descending sort of the row in LDS (64-bit composite keys),
//   * running sum in the order torch's CPU cumsum uses: sequential, accumulated in
//     float64, every prefix rounded to float32 and compared with float32(threshold),
//   * keep ranks <= the first prefix that reaches the threshold (none if never),
//   * OR in the block holding original key 0 (optional) and the row's own segment,
//   * emit the dense byte masks and the visit list: the ascending selected key blocks of
//     strictly earlier segments (the attention kernel adds the causal part of the row's
//     own segment itself, in original key order).
// Rows of up to 1024 blocks (2048 on the single-call path, which writes the attention kernel's merged lists instead of
// CSR rows) take the wave-level variant further down (one wave per row, the row in registers).
#include "pbs_lists.h"
#include "pbs_estimate.h"
#include "pbs_wave.h"
#include <utility>
#include "../../include/pbs_hip.h"   // the definitions below are checked against the public declarations
#include <float.h>

namespace {

struct SelectArgs {
  const float* P;          // (rows, nb, nb) or null when threshold_is_int_one
  const float* thr_rows;   // per-head thresholds (rows) or null
  float thr;
  int thr_is_int_one;
  int force_first;
  const int32_t* idx;      // (rows, nb*bs)
  int32_t* first_blk;      // (rows) workspace
  int nb, bs, bps, S, n_pow2;
  uint8_t* sel_mask;       // (rows, nb, nb) or null: selected | first-token
  uint8_t* final_mask;     // (rows, nb, nb) or null: sel | own segment
  int32_t* csr_cols;       // (rows, nb, nb) or null
  int32_t* csr_cnt;        // (rows, nb)
  uint8_t* needed;         // (rows, nb) or null: set to 1 for every key block on some query block's visit list
  int cand_rule;           // which entries of a row can be non-zero: 0 any, 1 kb < first block of qb's segment, 2 kb <= qb
  int qb_lo, qb_hi;        // wave kernel: the query blocks this launch covers
  int in_place;            // merged lists of un-permuted blocks up to the diagonal one, which is always visited
};

// Block that holds original key 0.  A segment-wise permutation keeps it inside the first segment, so that
// part of the row is searched first; the rest only if it is not there (any index layout stays correct).
__global__ __launch_bounds__(1024) void first_token_block_kernel(const int32_t* idx, int32_t* first_blk, int S_pad, int bs,
                                                                 int first_span) {
  __shared__ int found;
  if (threadIdx.x == 0) found = -1;
  __syncthreads();
  const int32_t* row = idx + (int64_t)blockIdx.x * S_pad;
  for (int i = threadIdx.x; i < first_span; i += blockDim.x)
    if (row[i] == 0) atomicMax(&found, i / bs);
  __syncthreads();
  if (found < 0) {
    for (int i = first_span + threadIdx.x; i < S_pad; i += blockDim.x)
      if (row[i] == 0) atomicMax(&found, i / bs);
  }
  __syncthreads();
  if (threadIdx.x == 0) first_blk[blockIdx.x] = found;
}

__device__ __forceinline__ double shfl_up_f64(double v, int delta) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __shfl_up((uint32_t)u, delta, 64), hi = __shfl_up((uint32_t)(u >> 32), delta, 64);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double readlane_f64(double v, int lane) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)u, lane), hi = __builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// ---- sums over the lanes of a wave without LDS: a shuffle is a trip through it, and what follows waits for it; a row's decision had 24 of
// them in a chain (whole pass, with them -> this and the key fragments and the threshold read once, ahead: 32 / 8 heads x 600 40.9 -> 39.4 us, 28 / 4 x 1000
// 52.5 -> 51.5, 8 / 2 x 8192 110.0 -> 108.7).
// the lane above's value of an inclusive prefix, zero for the first lane; and the prefix itself: inside rows of sixteen lanes, then
// rows 0 and 2 to the next, then the first two rows to the others
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_or_zero_f64(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, ROWS, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, ROWS, 0xf, false);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double wave_prefix_f64(double v) {
  v += dpp_or_zero_f64<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8
  v += dpp_or_zero_f64<0x112, 0xf>(v);
  v += dpp_or_zero_f64<0x114, 0xf>(v);
  v += dpp_or_zero_f64<0x118, 0xf>(v);
  v += dpp_or_zero_f64<0x142, 0xa>(v);   // row_bcast 15 into rows 1 and 3
  v += dpp_or_zero_f64<0x143, 0xc>(v);   // row_bcast 31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ double lane_before_f64(double v) { return dpp_or_zero_f64<0x138, 0xf>(v); }   // wave_shr 1
// numbers of up to `BITS` bits: their sum over the wave, and over the lanes before
template <int BITS>
__device__ __forceinline__ int wave_sum_of(int n, uint64_t lanes = ~0ull) {
  int sum = 0;
#pragma unroll
  for (int b = 0; b < BITS; ++b) sum += __popcll(__ballot(n >> b & 1) & lanes) << b;
  return sum;
}

__global__ __launch_bounds__(256) void select_blocks_kernel(SelectArgs a) {
  extern __shared__ uint64_t keys[];
  uint8_t* flag = reinterpret_cast<uint8_t*>(keys + a.n_pow2);
  __shared__ int s_first;
  __shared__ int s_scan[256];
  const int qb = blockIdx.x, row = blockIdx.y;
  const int nb = a.nb;
  const int seg_first = (qb / a.bps) * a.bps;
  const int seg_end = min(seg_first + a.bps, nb);
  const int64_t row_off = ((int64_t)row * nb + qb) * nb;

  for (int kb = threadIdx.x; kb < nb; kb += blockDim.x) flag[kb] = 0;

  if (a.thr_is_int_one) {
    __syncthreads();
    for (int kb = threadIdx.x; kb < seg_first; kb += blockDim.x) flag[kb] = 1;
  } else {
    const float* p = a.P + row_off;
    for (int i = threadIdx.x; i < a.n_pow2; i += blockDim.x) {
      uint64_t key = ~0ull;
      if (i < nb) {
        float v = p[i];
        if (v != v) v = 0.f;
        else if (v == INFINITY) v = FLT_MAX;
        else if (v == -INFINITY) v = -FLT_MAX;
        key = desc_stable_key(v, (uint32_t)i);
      }
      keys[i] = key;
    }
    bitonic_sort_lds(keys, a.n_pow2);
    if (threadIdx.x < 64) {
      // Running sum of the sorted row by ONE wave: lane l owns the `per` consecutive ranks from l * per.  The
      // sum is first taken as a parallel float64 prefix (local sums + wave scan), which differs from the
      // sequential float64 sum torch's CPU cumsum forms by < 1e-12; "float32(prefix) >= threshold" is decided
      // from it unless a prefix up to the first hit lies within 1e-11 of the float32 rounding boundary of the
      // threshold -- only then the exact sequential sum is evaluated, lane after lane.  Either way the decision
      // is the sequential sum's.
      const int lane = threadIdx.x;
      const int per = a.n_pow2 / 64;   // n_pow2 >= 2048 here
      const float thr = a.thr_rows ? a.thr_rows[row] : a.thr;
      const int r_lo = lane * per;
      double c = 0.0;
      for (int u = 0; u < per; ++u) {
        const int r = r_lo + u;
        c += r < nb ? (double)desc_key_value(keys[r]) : 0.0;
      }
      double incl = c;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const double t = shfl_up_f64(incl, d);
        if (lane >= d) incl += t;
      }
      double excl = shfl_up_f64(incl, 1);
      if (lane == 0) excl = 0.0;
      const double mid = 0.5 * ((double)thr + (double)nextafterf(thr, -INFINITY));
      const double tol = 1e-11 * fmax(1.0, fabs(mid));
      int my_first = INT_MAX, my_amb = INT_MAX;   // first reaching rank / first ambiguous rank of this lane
      {
        double cp = excl;
        for (int u = 0; u < per; ++u) {
          const int r = r_lo + u;
          if (r >= nb) break;
          cp += (double)desc_key_value(keys[r]);
          if (my_first == INT_MAX && (float)cp >= thr) my_first = r;
          if (my_amb == INT_MAX && fabs(cp - mid) <= tol) my_amb = r;
        }
      }
      int first = my_first, amb = my_amb;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        first = min(first, __shfl_xor(first, off, 64));
        amb = min(amb, __shfl_xor(amb, off, 64));
      }
      if (amb <= first && amb != INT_MAX) {
        // exact sequential sum: lane after lane, each continuing from the lane before
        double carry = 0.0;
        first = INT_MAX;
        for (int L = 0; L < 64 && first == INT_MAX; ++L) {
          double cs = carry;
          int hit = INT_MAX;
          if (lane == L) {
            for (int u = 0; u < per; ++u) {
              const int r = r_lo + u;
              if (r >= nb) break;
              cs += (double)desc_key_value(keys[r]);
              if (hit == INT_MAX && (float)cs >= thr) hit = r;
            }
          }
          carry = readlane_f64(cs, L);
          first = __builtin_amdgcn_readlane(hit, L);
        }
      }
      if (lane == 0) s_first = (first == INT_MAX || first >= nb) ? -1 : first;
    }
    __syncthreads();
    const int first = s_first;
    for (int r = threadIdx.x; r <= first; r += blockDim.x) flag[(uint32_t)keys[r]] = 1;
  }
  __syncthreads();
  if (a.force_first && threadIdx.x == 0) {
    const int fb = a.first_blk[row];
    if (fb >= 0 && fb < nb) flag[fb] = 1;
  }
  __syncthreads();

  // visit list: the selected blocks of strictly earlier segments (the attention kernel adds the query
  // block's own segment itself)
  const int per = (nb + 255) / 256;
  const int k0 = threadIdx.x * per, k1 = min(k0 + per, nb);
  int cnt = 0;
  for (int kb = k0; kb < k1; ++kb) {
    const bool own = kb >= seg_first && kb < seg_end;
    const uint8_t s = flag[kb];
    if (a.sel_mask) a.sel_mask[row_off + kb] = s;
    if (a.final_mask) a.final_mask[row_off + kb] = s | (own ? 1 : 0);
    cnt += (s && kb < seg_first) ? 1 : 0;
  }
  s_scan[threadIdx.x] = cnt;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    int v = 0;
    if ((int)threadIdx.x >= off) v = s_scan[threadIdx.x - off];
    __syncthreads();
    s_scan[threadIdx.x] += v;
    __syncthreads();
  }
  int w = s_scan[threadIdx.x] - cnt;
  if (a.csr_cols) {
    for (int kb = k0; kb < k1; ++kb) {
      if (flag[kb] && kb < seg_first) a.csr_cols[row_off + w++] = kb;
    }
  }
  if (a.needed) {
    for (int kb = k0; kb < k1; ++kb)
      if (flag[kb] && kb < seg_first) a.needed[(int64_t)row * nb + kb] = 1;   // every writer stores the same value
  }
  if (threadIdx.x == 255) a.csr_cnt[(int64_t)row * nb + qb] = s_scan[255];
}


// ---------------------------------------------------------------------------------------------
// Wave-level variant (rows of up to 2048 blocks): ONE wave per row, the row lives in registers.
//   * bitonic network on the 32-bit value keys, NPL keys per lane, no barriers and no LDS: strides below NPL are register
//     compare-exchanges, larger strides exchange with lane ^ (stride / NPL) by row moves of the vector unit; the stable
//     order's tie-break by index is applied only where it matters, at the value where the threshold is reached;
//   * the running sum is first taken as a parallel float64 prefix (local prefixes + wave scan).  It
//     differs from the sequential sum by < 1e-12, so "float32(prefix) >= threshold" is decided from it
//     unless some prefix up to the first hit lies within 1e-11 of the float32 rounding boundary of the
//     threshold; only then the exact sequential sum is evaluated (lane after lane).  Either way the
//     decision is the one the sequential float64 sum gives;
//   * flags, own-segment minima, masks and the compacted visit list as in the block-level kernel.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
  TwoOf t = with_lane_xor<1>(v);
  v = min(t.a, t.b);
  t = with_lane_xor<2>(v);
  v = min(t.a, t.b);
  t = with_lane_xor<4>(v);
  v = min(t.a, t.b);
  t = with_lane_xor<8>(v);
  v = min(t.a, t.b);
  t = with_lane_xor<16>(v);
  v = min(t.a, t.b);
  t = with_lane_xor<32>(v);
  return min(t.a, t.b);
}
// the median of three: the minimum of a and b where c is 0, their maximum where it is ~0
__device__ __forceinline__ uint32_t med3_u32(uint32_t a, uint32_t b, uint32_t c) { return max(min(a, b), min(max(a, b), c)); }

// one stage of the network: LS is the lane distance
template <int NPL, int LS>
__device__ __forceinline__ void cross_lane_stage(uint32_t (&k)[NPL], int lane) {
  uint32_t side = lane & LS ? ~0u : 0u;   // the upper lane keeps the maximum
  asm("" : "+v"(side));                   // (a value, not a condition: one median per key instead of two compares and a select)
#pragma unroll
  for (int r = 0; r < NPL; ++r) {
    const TwoOf t = with_lane_xor<LS>(k[r]);
    k[r] = med3_u32(t.a, t.b, side);
  }
}
// the stages of strides 2^n - 1 .. 1 inside a lane's keys, ascending or, for `size` < NPL, by the register's place
template <int NPL>
__device__ __forceinline__ void local_stages(uint32_t (&k)[NPL], int size) {
#pragma unroll
  for (int stride = min(size, NPL) >> 1; stride > 0; stride >>= 1) {
#pragma unroll
    for (int r = 0; r < NPL; ++r) {
      if ((r & stride) == 0) {
        const int p = r | stride;
        const bool up = size >= NPL || (r & size) == 0;
        const uint32_t lo = min(k[r], k[p]), hi = max(k[r], k[p]);
        k[r] = up ? lo : hi;
        k[p] = up ? hi : lo;
      }
    }
  }
}
// a phase: runs of NPL * LANES / 2 keys become runs of NPL * LANES (LANES 1: a lane's own keys).  Where the direction depends
// on the lane, the keys of the descending lanes are complemented for the phase, so that every exchange is a plain minimum
// and maximum; `flipped` is the complement the keys carry from the phase before.
template <int NPL>
__device__ __forceinline__ void begin_phase(uint32_t (&k)[NPL], int lanes, int lane, uint32_t& flipped) {
  const uint32_t flip = (lane & lanes) ? ~0u : 0u, change = flip ^ flipped;
#pragma unroll
  for (int r = 0; r < NPL; ++r) k[r] ^= change;
  flipped = flip;
}
template <int NPL, int LANES>
__device__ __forceinline__ void phase(uint32_t (&k)[NPL], int lane, uint32_t& flipped) {
  begin_phase<NPL>(k, LANES, lane, flipped);
  if constexpr (LANES >= 64) cross_lane_stage<NPL, 32>(k, lane);
  if constexpr (LANES >= 32) cross_lane_stage<NPL, 16>(k, lane);
  if constexpr (LANES >= 16) cross_lane_stage<NPL, 8>(k, lane);
  if constexpr (LANES >= 8) cross_lane_stage<NPL, 4>(k, lane);
  if constexpr (LANES >= 4) cross_lane_stage<NPL, 2>(k, lane);
  if constexpr (LANES >= 2) cross_lane_stage<NPL, 1>(k, lane);
  local_stages<NPL>(k, NPL);
}
// The bitonic network on 32-bit keys, NPL per lane.  Short rows have it unrolled.  With 32 keys per lane the phases that
// reach across lanes are a loop over one copy of each stage: unrolled, the compiler gave the long rows twice the time
// (rows of 1025 .. 2048 blocks of a 256k head shard: 361 us unrolled, 169 us as a loop; the short rows of a 4k prompt: 6.2
// unrolled against 7.5 us).
template <int NPL>
__device__ __forceinline__ void wave_bitonic_sort_u32(uint32_t (&k)[NPL], int lane) {
#pragma unroll
  for (int size = 2; size < NPL; size <<= 1) local_stages<NPL>(k, size);
  uint32_t flipped = 0;
  if constexpr (NPL < 32) {
    phase<NPL, 1>(k, lane, flipped);
    phase<NPL, 2>(k, lane, flipped);
    phase<NPL, 4>(k, lane, flipped);
    phase<NPL, 8>(k, lane, flipped);
    phase<NPL, 16>(k, lane, flipped);
    phase<NPL, 32>(k, lane, flipped);
    phase<NPL, 64>(k, lane, flipped);
  } else {
#pragma nounroll
    for (int lanes = 1; lanes <= 64; lanes <<= 1) {
      begin_phase<NPL>(k, lanes, lane, flipped);
      switch (lanes) {   // strides from lanes / 2 lanes down to one
        case 64: cross_lane_stage<NPL, 32>(k, lane); [[fallthrough]];
        case 32: cross_lane_stage<NPL, 16>(k, lane); [[fallthrough]];
        case 16: cross_lane_stage<NPL, 8>(k, lane); [[fallthrough]];
        case 8: cross_lane_stage<NPL, 4>(k, lane); [[fallthrough]];
        case 4: cross_lane_stage<NPL, 2>(k, lane); [[fallthrough]];
        case 2: cross_lane_stage<NPL, 1>(k, lane); [[fallthrough]];
        default: local_stages<NPL>(k, NPL); break;
      }
    }
  }
}

// what a row's decision reads besides its probabilities: the threshold, and the block to be selected in any case (-1: none)
struct RowRule {
  float thr;
  int first_blk;
};
__device__ __forceinline__ RowRule row_rule(const SelectArgs& a, int row) {
  return {a.thr_rows ? a.thr_rows[row] : a.thr, a.force_first ? (a.first_blk ? a.first_blk[row] : 0) : -1};
}
// One wave decides a head's row of query block qb with the probabilities p[0 .. nb): flag[0 .. nb) (this wave's, in LDS) becomes the selection.
template <int NPL>
__device__ __forceinline__ void decide_row(const SelectArgs& a, RowRule rule, int qb, const float* p, uint8_t* flag) {
  const int lane = threadIdx.x & 63;
  const int nb = a.nb;
  const float thr = rule.thr;
  const int seg_first = (qb / a.bps) * a.bps;

  for (int kb = lane; kb < nb; kb += 64) flag[kb] = 0;

  if (a.thr_is_int_one) {
    for (int kb = lane; kb < seg_first; kb += 64) flag[kb] = 1;
  } else {
    // entries that are zero by construction sort behind every candidate (ties keep index order) and add nothing
    // to the running sum: the row is sorted up to its last candidate only (the launch is sized for that)
    const int count = a.cand_rule == 1 ? seg_first : a.cand_rule == 2 ? min(qb + 1, nb) : nb;
    // value keys, ascending key = descending value; lane l holds entries l * NPL .. l * NPL + NPL - 1, so that the order of
    // (lane, register) is the order of the indices.  No entry has the key ~0, which stands for "none".
    uint32_t k0v[NPL];
    float raw[NPL];
    if (NPL >= 4 && (nb & 3) == 0 && ((uintptr_t)a.P & 15) == 0) {   // (p is a row of a.P)
      // whole 16-byte pieces: the one that holds the last candidate ends inside the row (nb is a multiple of four)
#pragma unroll
      for (int r = 0; r < NPL; r += 4) {
        const int i = lane * NPL + r;
        f32x4 x = {0.f, 0.f, 0.f, 0.f};
        if (i < count) x = *reinterpret_cast<const f32x4*>(p + i);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (r + e < NPL) raw[r + e] = x[e];
      }
    } else {
#pragma unroll
      for (int r = 0; r < NPL; ++r) {
        const int i = lane * NPL + r;
        raw[r] = i < count ? p[i] : 0.f;
      }
    }
#pragma unroll
    for (int r = 0; r < NPL; ++r) {
      float v = raw[r];
      if (v != v) v = 0.f;
      else if (v == INFINITY) v = FLT_MAX;
      else if (v == -INFINITY) v = -FLT_MAX;
      k0v[r] = lane * NPL + r < count ? ~f32_orderable(v) : ~0u;
    }
    // Rows whose mass sits in a few blocks need no sort: the largest remaining entry is taken out of the row
    // (value descending, ties by index -- the order of the sort) and added to the
    // sequential float64 sum until float32(sum) reaches the threshold: the reference's decision, term by term.
    // Tried only when EXTRACT_MAX times the row's largest value can reach the threshold; a row that does not
    // get there in EXTRACT_MAX steps is sorted whole like any other.
    bool decided = false;
    if (NPL > 1) {
      constexpr int EXTRACT_MAX = 16;
      uint32_t mine = k0v[0];   // the smallest key of this lane
#pragma unroll
      for (int r = 1; r < NPL; ++r) mine = min(mine, k0v[r]);
      uint32_t best = wave_min_u32(mine);
      if (best != ~0u && (float)((double)f32_from_orderable(~best) * EXTRACT_MAX) >= thr) {
        uint32_t w[NPL];
#pragma unroll
        for (int r = 0; r < NPL; ++r) w[r] = k0v[r];
        double cum = 0.0;
        int my_idx = 0;
        int taken = 0;
        for (int it = 0; it < EXTRACT_MAX; ++it) {
          if (best == ~0u) break;   // the row has no further entry: not reached, let the sort path say so
          // the lowest lane that holds the key, and its lowest register that does
          const int owner = __builtin_ctzll(__ballot(mine == best));
          int at = 0;
#pragma unroll
          for (int r = NPL - 1; r >= 0; --r) at = w[r] == best ? r : at;
          const int gone = lane == owner ? at : NPL;
          mine = ~0u;
#pragma unroll
          for (int r = 0; r < NPL; ++r) {
            w[r] = r == gone ? ~0u : w[r];
            mine = min(mine, w[r]);
          }
          const int idx = owner * NPL + __builtin_amdgcn_readlane(at, owner);
          if (lane == it) my_idx = idx;
          cum += (double)f32_from_orderable(~best);
          taken = it + 1;
          if ((float)cum >= thr) {
            decided = true;
            break;
          }
          best = wave_min_u32(mine);
        }
        if (decided && lane < taken) flag[my_idx] = 1;
      }
    }
    if (!decided) {
    // The sort runs on the 32-bit value keys alone (ascending key = descending value).  Entries of equal value are
    // interchangeable in the running sum; which of them the stable order takes first matters only for the value at
    // which the threshold is reached, and is settled there by index (below).
    uint32_t kv[NPL];
#pragma unroll
    for (int r = 0; r < NPL; ++r) kv[r] = k0v[r];
    wave_bitonic_sort_u32<NPL>(kv, lane);

    auto value = [&](int r) __attribute__((always_inline)) { return lane * NPL + r < count ? f32_from_orderable(~kv[r]) : 0.f; };
    // parallel float64 prefix
    double c = 0.0;
#pragma unroll
    for (int r = 0; r < NPL; ++r) c += (double)value(r);
    const double excl = lane_before_f64(wave_prefix_f64(c));
    // float32 rounding boundary of the threshold (midpoint to its predecessor), as a double
    const double mid = 0.5 * ((double)thr + (double)nextafterf(thr, -INFINITY));
    const double tol = 1e-11 * fmax(1.0, fabs(mid));
    uint32_t reach = 0, amb = 0;
    c = 0.0;
#pragma unroll
    for (int r = 0; r < NPL; ++r) {
      c += (double)value(r);
      const double cp = excl + c;
      reach |= ((float)cp >= thr ? 1u : 0u) << r;
      amb |= (fabs(cp - mid) <= tol ? 1u : 0u) << r;
    }
    const uint64_t reached = __ballot(reach != 0);   // the first rank is the lowest lane's lowest
    int first = INT_MAX;
    if (reached) {
      const int owner = __builtin_ctzll(reached);
      first = owner * NPL + __builtin_ctz((uint32_t)__builtin_amdgcn_readlane((int)reach, owner));
    }
    // ambiguous prefixes at or before the first hit?
    bool my_amb = false;
#pragma unroll
    for (int r = 0; r < NPL; ++r) my_amb |= ((amb >> r) & 1u) && (lane * NPL + r <= first) && (lane * NPL + r < nb);
    if (__any(my_amb)) {
      // exact sequential sum, lane after lane
      double carry = 0.0;
      first = INT_MAX;
      for (int L = 0; L < 64; ++L) {
        double cs = carry;
        uint32_t rch = 0;
#pragma unroll
        for (int r = 0; r < NPL; ++r) {
          cs += (double)value(r);
          rch |= ((float)cs >= thr ? 1u : 0u) << r;
        }
        const uint32_t rl = (uint32_t)__builtin_amdgcn_readlane((int)rch, L);
        carry = readlane_f64(cs, L);
        if (rl) {
          first = L * NPL + __builtin_ctz(rl);
          break;
        }
      }
    }
    if (first >= count) first = -1;   // never reached (padding ranks cannot qualify: they add zero)
    if (first >= 0) {
      // the selection is ranks 0 .. first of the stable order: every entry above the value at rank `first`, and of
      // the entries equal to it the m lowest indices, m = first + 1 - (number of entries above it)
      uint32_t at_first = 0;
#pragma unroll
      for (int r = 0; r < NPL; ++r) at_first = (r == first % NPL) ? kv[r] : at_first;
      const uint32_t kstar = (uint32_t)__builtin_amdgcn_readlane((int)at_first, first / NPL);
      int above = 0, ties = 0;
#pragma unroll
      for (int r = 0; r < NPL; ++r) {
        above += k0v[r] < kstar ? 1 : 0;
        ties += k0v[r] == kstar ? 1 : 0;
      }
      constexpr int BITS = NPL == 1 ? 1 : NPL <= 2 ? 2 : NPL <= 4 ? 3 : NPL <= 8 ? 4 : NPL <= 16 ? 5 : 6;   // of 0 .. NPL
      const int m = first + 1 - wave_sum_of<BITS>(above);
      int tie_rank = wave_sum_of<BITS>(ties, (1ull << lane) - 1ull);   // ties at lower indices
#pragma unroll
      for (int r = 0; r < NPL; ++r) {
        const bool tie = k0v[r] == kstar;
        if (k0v[r] < kstar || (tie && tie_rank < m)) flag[lane * NPL + r] = 1;
        tie_rank += tie ? 1 : 0;
      }
    }
    }   // !decided
    // a row without candidates is all zeros: sorted whole, its first entry is block 0 and the running sum is 0
    if (count == 0 && 0.0f >= thr && lane == 0) flag[0] = 1;
  }
  __builtin_amdgcn_wave_barrier();
  if (lane == 0 && rule.first_blk >= 0 && rule.first_blk < nb) flag[rule.first_blk] = 1;
  if (a.in_place && lane == 0) flag[qb] = 1;
}

// one wave decides row `rq` ((row, qb - qb_lo) flattened) of the group of rows [qb_lo, qb_hi) x all heads
template <int NPL>
__device__ __forceinline__ void select_row_by_wave(const SelectArgs& a, int64_t rq, int total_rows, uint8_t* smem_w) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nb = a.nb;
  const int nb_pad = (nb + 15) & ~15;
  uint8_t* flag = smem_w + wave * nb_pad;
  if (rq >= total_rows) return;
  const int nqb = a.qb_hi - a.qb_lo;
  const int row = (int)(rq / nqb), qb = a.qb_lo + (int)(rq % nqb);
  const int seg_first = (qb / a.bps) * a.bps;
  const int seg_end = min(seg_first + a.bps, nb);
  const int64_t row_off = ((int64_t)row * nb + qb) * nb;
  decide_row<NPL>(a, row_rule(a, row), qb, a.P + row_off, flag);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  int base = 0;
  // without mask outputs only the blocks of earlier segments matter: they are what the visit list and the gather's
  // filter hold
  const int kb_end = (a.sel_mask || a.final_mask) ? nb : seg_first;
  for (int kb0 = 0; kb0 < kb_end; kb0 += 64) {
    const int kb = kb0 + lane;
    bool visit = false;
    if (kb < kb_end) {
      const bool own = kb >= seg_first && kb < seg_end;
      const uint8_t sf = flag[kb];
      if (a.sel_mask) a.sel_mask[row_off + kb] = sf;
      if (a.final_mask) a.final_mask[row_off + kb] = sf | (own ? 1 : 0);
      visit = sf && kb < seg_first;   // own-segment blocks are the attention kernel's business
    }
    const uint64_t ballot = __ballot(visit);
    if (visit && a.csr_cols) a.csr_cols[row_off + base + __popcll(ballot & ((1ull << lane) - 1ull))] = kb;
    if (visit && a.needed) a.needed[(int64_t)row * nb + kb] = 1;   // every writer stores the same value
    base += __popcll(ballot);
  }
  if (lane == 0) a.csr_cnt[(int64_t)row * nb + qb] = base;
}

template <int NPL>
__global__ __launch_bounds__(256) void select_blocks_wave_kernel(SelectArgs a, int total_rows) {
  extern __shared__ uint8_t smem_w[];
  select_row_by_wave<NPL>(a, (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), total_rows, smem_w);
}

// Up to five groups of rows of like length (see pbs_select_blocks) in ONE launch, the longest rows first: as launches
// of their own the groups run one after the other and each ends with a tail of idle CUs.
struct SelectGroups {
  int n;
  int npl[5], qb_lo[5], qb_hi[5];
  int wg_end[5];   // workgroups of groups 0 .. g
};
__global__ __launch_bounds__(256) void select_blocks_groups_kernel(SelectArgs a, SelectGroups gr, int rows) {
  extern __shared__ uint8_t smem_w[];
  int g = 0;
  while (g + 1 < gr.n && (int)blockIdx.x >= gr.wg_end[g]) ++g;
  const int wg0 = g == 0 ? 0 : gr.wg_end[g - 1];
  a.qb_lo = gr.qb_lo[g];
  a.qb_hi = gr.qb_hi[g];
  const int total = rows * (a.qb_hi - a.qb_lo);
  const int64_t rq = (int64_t)((int)blockIdx.x - wg0) * 4 + (threadIdx.x >> 6);
  switch (gr.npl[g]) {
    case 1: select_row_by_wave<1>(a, rq, total, smem_w); break;
    case 2: select_row_by_wave<2>(a, rq, total, smem_w); break;
    case 4: select_row_by_wave<4>(a, rq, total, smem_w); break;
    case 8: select_row_by_wave<8>(a, rq, total, smem_w); break;
    default: select_row_by_wave<16>(a, rq, total, smem_w); break;
  }
}

// Row (`row`, pair) of a workgroup whose waves have decided the rows of two pairs into `flags` (nb rounded up to 16 bytes a wave): the first wave
// of a pair writes its list, the second one the gather's flags; items of one query block: every wave both.
__device__ __forceinline__ void write_lists(const SelectArgs& a, const PairLists& l, int row, int pair, const uint8_t* flags) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int nb = a.nb, nb_pad = (nb + 15) & ~15, npair = (nb + 1) >> 1, qb0 = 2 * pair, qb = qb0 + (wave & 1);
  const bool pairs = l.span == 2;
  if (!pairs && qb >= nb) return;
  const int first = pairs ? qb0 : qb;   // of the item
  const bool second = pairs && first + 1 < nb;
  const int qb1 = second ? first + 1 : first;
  const int sf0 = (first / a.bps) * a.bps, sf1 = (qb1 / a.bps) * a.bps;
  // a row's flags count up to its own segment, or up to its own block
  const int end0 = a.in_place ? first + 1 : sf0, end1 = second ? (a.in_place ? qb1 + 1 : sf1) : 0, end = max(end0, end1);
  const uint32_t kind = a.in_place ? ENT_ORIG : 0u;
  const uint32_t* f0 = reinterpret_cast<const uint32_t*>(flags + (pairs ? wave & 2 : wave) * nb_pad);
  const uint32_t* f1 = reinterpret_cast<const uint32_t*>(flags + ((wave & 2) + 1) * nb_pad);
  // the flags of blocks 4 x .. 4 x + 3, a byte each: bit 0 visited by the first query block, bit 1 by the second
  auto visited = [&](int x) __attribute__((always_inline)) {
    auto below = [&](int n) __attribute__((always_inline)) {   // bytes of blocks below n
      const int valid = n - 4 * x;
      return valid >= 4 ? ~0u : valid <= 0 ? 0u : (1u << (8 * valid)) - 1u;
    };
    const uint32_t m0 = below(end0), m1 = below(end1);
    return (m0 ? f0[x] & m0 : 0u) | (m1 ? f1[x] & m1 : 0u) << 1;
  };
  if (!pairs || (wave & 1)) {
    if (a.needed)
      for (int x = lane; 4 * x < end; x += 64) {
        const uint32_t v = visited(x);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (v >> (8 * e) & 3u) a.needed[(int64_t)row * nb + 4 * x + e] = 1;   // every writer stores the same value
      }
    if (pairs) return;
  }
  const int n_items = pairs ? npair : nb;
  uint16_t* header = l.plist + ((int64_t)row * n_items + (n_items - 1 - (pairs ? pair : qb))) * l.cap;
  uint16_t* out = header + LIST_HEADER;
  int base = 0;
  for (int x0 = 0; 4 * x0 < end; x0 += 64) {
    const int x = x0 + lane;
    const uint32_t v = 4 * x < end ? visited(x) : 0u;
    const int n = __popc((v | v >> 1) & 0x01010101u);
    // prefix of n (0 .. 4) over the lanes, a bit of it at a time
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t b0 = __ballot(n & 1), b1 = __ballot(n & 2), b2 = __ballot(n & 4);
    int w = base + __popcll(b0 & below) + 2 * __popcll(b1 & below) + 4 * __popcll(b2 & below);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t use = v >> (8 * e) & 3u;
      if (use) out[w++] = (uint16_t)((uint32_t)(4 * x + e) | kind | use << 14);
    }
    base += __popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2);
  }
  const int n_own = a.in_place ? 0 : qb1 - sf0 + 1;
  for (int t = lane; t < n_own; t += 64) {
    const int kb = sf0 + t;
    const uint32_t use = (kb <= first ? 1u : 0u) | (second && kb >= sf1 ? 2u : 0u);
    out[base + t] = (uint16_t)((uint32_t)kb | ENT_ORIG | use << 14);
  }
  if (lane == 0) {
    header[0] = (uint16_t)(base + n_own);
    header[1] = (uint16_t)(row / l.Hq);
    header[2] = (uint16_t)(row % l.Hq);
    header[3] = (uint16_t)(row % l.Hq / l.group);
    header[4] = (uint16_t)first;
    header[5] = (uint16_t)(second ? 2 : 1);
  }
}

// ---- the single-call path: selection straight into the merged lists that the attention kernel reads (pbs_lists.h).
// A workgroup decides the rows of two pairs of query blocks, one wave each, into flags in LDS; then the first wave of a
// pair writes the pair's list and the second one the gather's flags (items of one query block: every wave those of its row).  No CSR rows (4 bytes per visited block and row, written
// here and read back) and no launch that merges them.  Groups are in pairs here: qb_lo / qb_hi are pair numbers.
// LONG: rows of 1025 .. 2048 candidates, in a kernel of their own: the register need of 32 entries per lane would cost the shorter
// rows two thirds of their waves.
// Waves per SIMD: left to itself the compiler gives the long rows one (8 / 2 heads x 262144 7.39 against 7.21 ms a pass) and the others, a register too many,
// three (32 / 8 x 131072 concentrated 2584 against 2572 us).
template <bool LONG>
__global__ __launch_bounds__(256, LONG ? 2 : 4) void select_pair_lists_kernel(SelectArgs a, PairLists l, SelectGroups gr, int rows) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_w[];
  int g = 0;
  while (g + 1 < gr.n && (int)blockIdx.x >= gr.wg_end[g]) ++g;
  const int wg0 = g == 0 ? 0 : gr.wg_end[g - 1];
  const int n_pairs = gr.qb_hi[g] - gr.qb_lo[g], total = rows * n_pairs;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int unit = ((int)blockIdx.x - wg0) * 2 + (wave >> 1);
  const bool live = unit < total;
  const int row = live ? unit / n_pairs : 0, pair = gr.qb_lo[g] + (live ? unit - row * n_pairs : 0);
  const int nb = a.nb, nb_pad = (nb + 15) & ~15, qb = 2 * pair + (wave & 1);
  uint8_t* flag = smem_w + wave * nb_pad;
  if (blockIdx.x == 0 && threadIdx.x < 8) l.queue[threadIdx.x] = l.first_tickets;
  if (live && qb < nb) {
    const float* p = a.P + ((int64_t)row * nb + qb) * nb;
    const RowRule rule = row_rule(a, row);
    if constexpr (LONG) {
      decide_row<32>(a, rule, qb, p, flag);
    } else {
      switch (gr.npl[g]) {
        case 1: decide_row<1>(a, rule, qb, p, flag); break;
        case 2: decide_row<2>(a, rule, qb, p, flag); break;
        case 4: decide_row<4>(a, rule, qb, p, flag); break;
        case 8: decide_row<8>(a, rule, qb, p, flag); break;
        default: decide_row<16>(a, rule, qb, p, flag); break;
      }
    }
  }
  __syncthreads();
  if (live) write_lists(a, l, row, pair, smem_w);
}

// Estimate and selection of four query blocks in one launch, for rows of up to 64 blocks: the workgroup forms the probabilities of
// the 32 query blocks its own are among (the products are next to nothing) and keeps its own rows in LDS.  A launch and its
// way to memory and back less: 32 / 8 heads x 512 51.8 -> 48.6 us a pass, 28 / 4 x 1000 63.1 -> 59.4, 32 / 8 x 4096 174.0 -> 169.9, x
// 8192 482 -> 477.  Above 2048 blocks the repeated products outweigh it: 128 heads x 6144 1159 against 1162, 32 / 8 x
// 12288 (two entries a lane) 962 against 970.
template <bool CAUSAL>
__global__ __launch_bounds__(256) void estimate_select_kernel(const uint16_t* pooled_q, const uint16_t* pooled_k, SelectArgs a, PairLists l, Divisor sqrt_d) {
  __shared__ EstimateStats st;
  __shared__ float probs[4][PBS_ESTIMATE_SELECT_MAX_BLOCKS];
  __shared__ __attribute__((aligned(16))) uint8_t flags[4 * PBS_ESTIMATE_SELECT_MAX_BLOCKS];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int four = (int)gridDim.x - 1 - (int)blockIdx.x, row = blockIdx.y;   // the rows with the most candidates start first
  const int nb = a.nb, nb_pad = (nb + 15) & ~15, qb = 4 * four + wave;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 8) l.queue[threadIdx.x] = l.first_tickets;
  const int64_t head = (int64_t)row * nb * ESTIMATE_D;
  const RowRule rule = row_rule(a, row);   // (on its way while the probabilities are formed)
  static_assert(PBS_ESTIMATE_SELECT_MAX_BLOCKS <= 4 * 32, "a tile of key blocks a wave");
  estimate_tile<CAUSAL, true, true>(pooled_q + head, pooled_k + head, nb, a.bps, sqrt_d, four / 8, st, [&](int ql, int kb, float p) __attribute__((always_inline)) {
    if (ql >> 2 == (four & 7)) probs[ql & 3][kb] = p;
  });
  __syncthreads();
  if (qb < nb) decide_row<1>(a, rule, qb, probs[wave], flags + wave * nb_pad);
  __syncthreads();
  const int pair = 2 * four + (wave >> 1);
  if (2 * pair < nb) write_lists(a, l, row, pair, flags);
}

// Visit lists from a given block mask: one wave per (row, query block), the set bits of strictly earlier segments
// compacted in ascending order; own_missing counts the blocks of the query block's own segment the mask leaves out
// (in permuted order any of them can hold keys the query may see).
__global__ __launch_bounds__(256) void mask_to_csr_kernel(const uint8_t* __restrict__ mask, int32_t* __restrict__ cols,
                                                          int32_t* __restrict__ cnt, int32_t* __restrict__ own_missing, int nb,
                                                          int bps, int total_rows) {
  const int lane = threadIdx.x & 63;
  const int64_t rq = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (rq >= total_rows) return;
  const int qb = (int)(rq % nb);
  const int seg_first = (qb / bps) * bps, seg_end = min(seg_first + bps, nb);
  const uint8_t* m = mask + rq * nb;
  int base = 0, missing = 0;
  for (int kb0 = 0; kb0 < seg_end; kb0 += 64) {
    const int kb = kb0 + lane;
    const bool on = kb < seg_end && m[kb] != 0;
    const bool visit = on && kb < seg_first;
    const uint64_t ballot = __ballot(visit);
    if (visit) cols[rq * nb + base + __popcll(ballot & ((1ull << lane) - 1ull))] = kb;
    base += __popcll(ballot);
    missing += __popcll(__ballot(kb >= seg_first && kb < seg_end && !on));
  }
  if (lane == 0) {
    cnt[rq] = base;
    if (missing) atomicAdd(own_missing, missing);
  }
}

}  // namespace

extern "C" int pbs_block_mask_to_csr(const uint8_t* block_mask, int32_t* csr_cols, int32_t* csr_cnt, int32_t* own_missing,
                                     int rows, int nb, int blocks_per_segment, void* stream) {
  PBS_REQUIRE(block_mask && csr_cols && csr_cnt && own_missing, "pbs_block_mask_to_csr: null pointer");
  PBS_REQUIRE(rows > 0 && nb > 0 && nb <= 4096 && blocks_per_segment > 0 && (int64_t)rows * nb < (1ll << 31),
              "pbs_block_mask_to_csr: bad shape");
  const int total = rows * nb;
  hipLaunchKernelGGL(mask_to_csr_kernel, dim3((unsigned)((total + 3) / 4)), dim3(256), 0, (hipStream_t)stream, block_mask,
                     csr_cols, csr_cnt, own_missing, nb, blocks_per_segment, total);
  return pbs_check_launch("pbs_block_mask_to_csr");
}

extern "C" size_t pbs_select_blocks_workspace_bytes(int rows) { return (size_t)rows * sizeof(int32_t); }

extern "C" int pbs_select_blocks(const float* block_attn_scores, const float* threshold_per_row, float threshold,
                                 int threshold_is_int_one, int force_select_first_block, int candidate_rule,
                                 const int32_t* key_indices, int rows, int S, int block_size, int segment_size, uint8_t* sel_mask,
                                 uint8_t* final_mask, int32_t* csr_cols, int32_t* csr_cnt, uint8_t* block_needed,
                                 void* workspace, size_t workspace_bytes, void* stream) {
  PBS_REQUIRE(key_indices && csr_cnt, "pbs_select_blocks: null index / count pointer");
  PBS_REQUIRE(threshold_is_int_one || block_attn_scores, "pbs_select_blocks: null score pointer");
  PBS_REQUIRE(rows > 0 && rows <= 65535 && S > 0, "pbs_select_blocks: bad shape");
  PBS_REQUIRE(candidate_rule >= 0 && candidate_rule <= 2, "pbs_select_blocks: candidate_rule must be 0, 1 or 2");
  PBS_REQUIRE(block_size > 0 && block_size <= 256, "pbs_select_blocks: block_size %d outside (0, 256]", block_size);
  PBS_REQUIRE(segment_size > 0 && segment_size % block_size == 0, "pbs_select_blocks: segment_size must be a multiple of block_size");
  const int nb = (S + block_size - 1) / block_size;
  const int bps = segment_size / block_size;
  PBS_REQUIRE(nb <= 4096, "pbs_select_blocks: more than 4096 blocks per sequence (%d)", nb);
  PBS_REQUIRE(workspace && workspace_bytes >= pbs_select_blocks_workspace_bytes(rows), "pbs_select_blocks: workspace too small");
  SelectArgs a;
  a.P = block_attn_scores; a.thr_rows = threshold_per_row; a.thr = threshold;
  a.thr_is_int_one = threshold_is_int_one; a.force_first = force_select_first_block;
  a.idx = key_indices; a.first_blk = (int32_t*)workspace;
  a.nb = nb; a.bs = block_size; a.bps = bps; a.S = S; a.n_pow2 = next_pow2_int(nb);
  a.sel_mask = sel_mask; a.final_mask = final_mask; a.csr_cols = csr_cols; a.csr_cnt = csr_cnt;
  a.needed = block_needed;
  a.cand_rule = candidate_rule; a.qb_lo = 0; a.qb_hi = nb;
  hipStream_t st = (hipStream_t)stream;
  if (force_select_first_block)
    hipLaunchKernelGGL(first_token_block_kernel, dim3(rows), dim3(1024), 0, st, key_indices, a.first_blk, nb * block_size, block_size,
                       min(segment_size, nb * block_size));
  if (nb <= 1024) {
    // one wave per row, four rows per workgroup.  The sort network is sized for the longest row of a launch;
    // where the number of candidates grows with the query block, the rows are launched in groups of like length
    const size_t lds_w = (size_t)4 * ((nb + 15) & ~15);
    auto launch = [&](int npl, int qb_lo, int qb_hi) {
      SelectArgs g = a;
      g.qb_lo = qb_lo; g.qb_hi = qb_hi;
      const int total = rows * (qb_hi - qb_lo);
      const dim3 grid((unsigned)((total + 3) / 4));
      switch (npl) {
        case 1: hipLaunchKernelGGL(select_blocks_wave_kernel<1>, grid, dim3(256), lds_w, st, g, total); break;
        case 2: hipLaunchKernelGGL(select_blocks_wave_kernel<2>, grid, dim3(256), lds_w, st, g, total); break;
        case 4: hipLaunchKernelGGL(select_blocks_wave_kernel<4>, grid, dim3(256), lds_w, st, g, total); break;
        case 8: hipLaunchKernelGGL(select_blocks_wave_kernel<8>, grid, dim3(256), lds_w, st, g, total); break;
        default: hipLaunchKernelGGL(select_blocks_wave_kernel<16>, grid, dim3(256), lds_w, st, g, total); break;
      }
    };
    if (candidate_rule == 0 || threshold_is_int_one) {
      launch(threshold_is_int_one || nb <= 64 ? 1 : nb <= 128 ? 2 : nb <= 256 ? 4 : nb <= 512 ? 8 : 16, 0, nb);
    } else {
      SelectGroups gr;
      gr.n = 0;
      int qb_lo = 0;
      for (int npl = 1; npl <= 16 && qb_lo < nb; npl *= 2) {
        // query blocks whose candidate count fits 64 * npl sorted entries
        const int64_t lim = 64 * npl;
        int64_t hi = candidate_rule == 1 ? (lim / bps + 1) * (int64_t)bps : lim;
        if (npl == 16 || hi > nb) hi = nb;
        if (hi > qb_lo) {
          gr.npl[gr.n] = npl; gr.qb_lo[gr.n] = qb_lo; gr.qb_hi[gr.n] = (int)hi;
          ++gr.n;
          qb_lo = (int)hi;
        }
      }
      if (gr.n == 1) {
        launch(gr.npl[0], gr.qb_lo[0], gr.qb_hi[0]);
      } else {
        // longest rows first
        for (int x = 0; x < gr.n / 2; ++x) {
          std::swap(gr.npl[x], gr.npl[gr.n - 1 - x]);
          std::swap(gr.qb_lo[x], gr.qb_lo[gr.n - 1 - x]);
          std::swap(gr.qb_hi[x], gr.qb_hi[gr.n - 1 - x]);
        }
        int wgs = 0;
        for (int x = 0; x < gr.n; ++x) {
          wgs += (rows * (gr.qb_hi[x] - gr.qb_lo[x]) + 3) / 4;
          gr.wg_end[x] = wgs;
        }
        hipLaunchKernelGGL(select_blocks_groups_kernel, dim3((unsigned)wgs), dim3(256), lds_w, st, a, gr, rows);
      }
    }
    return pbs_check_launch("pbs_select_blocks");
  }
  const size_t lds = (size_t)a.n_pow2 * sizeof(uint64_t) + (size_t)((nb + 15) / 16) * 16;
  hipLaunchKernelGGL(select_blocks_kernel, dim3(nb, rows), dim3(256), lds, st, a);
  return pbs_check_launch("pbs_select_blocks");
}

int pbs_select_pair_lists(const float* block_attn_scores, Candidates rule, const float* threshold_per_row, float threshold, bool force_first,
                          const int32_t* first_blk, int rows, int S, int block_size, int segment_size, uint8_t* block_needed, const PairLists& lists,
                          void* stream) {
  const int nb = (S + block_size - 1) / block_size, npair = (nb + 1) / 2;
  PBS_REQUIRE(rows > 0 && rows <= 65535 && nb <= PBS_PAIR_SELECT_MAX_BLOCKS, "pbs_select_pair_lists: bad shape");
  PBS_REQUIRE(block_attn_scores, "pbs_select_pair_lists: null score pointer");
  SelectArgs a = {};
  a.P = block_attn_scores; a.thr_rows = threshold_per_row; a.thr = threshold;
  a.force_first = force_first;
  a.first_blk = const_cast<int32_t*>(first_blk);
  a.nb = nb; a.bs = block_size; a.bps = segment_size / block_size; a.S = S;
  a.needed = block_needed;
  a.cand_rule = (int)rule;
  a.in_place = rule == Candidates::UP_TO_DIAGONAL;
  // groups of pairs whose second row's candidates fit 64 * npl sorted entries, longest first
  int npl[6], lo[6], hi[6], n = 0, from = 0;
  for (int x = 1; x <= 32 && from < npair; x *= 2) {
    const int64_t blocks = a.in_place ? 64 * x : (64 * x / a.bps + 1) * (int64_t)a.bps;   // query blocks with at most 64 x candidates
    const int to = blocks >= nb ? npair : (int)(blocks / 2);
    if (to > from) {
      npl[n] = x; lo[n] = from; hi[n] = to;
      ++n;
      from = to;
    }
  }
  const size_t lds = (size_t)4 * ((nb + 15) & ~15);
  SelectGroups gr;
  gr.n = 0;
  int wgs = 0;
  for (int x = n - 1; x >= 0; --x) {
    if (npl[x] == 32) {
      SelectGroups one;
      one.n = 1;
      one.npl[0] = 32; one.qb_lo[0] = lo[x]; one.qb_hi[0] = hi[x];
      one.wg_end[0] = (rows * (hi[x] - lo[x]) + 1) / 2;
      hipLaunchKernelGGL(select_pair_lists_kernel<true>, dim3((unsigned)one.wg_end[0]), dim3(256), lds, (hipStream_t)stream, a, lists, one, rows);
      continue;
    }
    gr.npl[gr.n] = npl[x]; gr.qb_lo[gr.n] = lo[x]; gr.qb_hi[gr.n] = hi[x];
    wgs += (rows * (hi[x] - lo[x]) + 1) / 2;
    gr.wg_end[gr.n++] = wgs;
  }
  if (wgs)
    hipLaunchKernelGGL(select_pair_lists_kernel<false>, dim3((unsigned)wgs), dim3(256), lds, (hipStream_t)stream, a, lists, gr, rows);
  return pbs_check_launch("pbs_select_pair_lists");
}

int pbs_estimate_select_pair_lists(const void* pooled_q, const void* pooled_k, Candidates rule, const float* threshold_per_row,
                                   float threshold, bool force_first, const int32_t* first_blk, int rows, int S, int head_dim, int block_size, int segment_size,
                                   uint8_t* block_needed, const PairLists& lists, void* stream) {
  const int nb = (S + block_size - 1) / block_size;
  PBS_REQUIRE(pooled_q && pooled_k && head_dim == ESTIMATE_D, "pbs_estimate_select: bad pooled tensors");
  PBS_REQUIRE(rows > 0 && rows <= 65535 && nb <= PBS_ESTIMATE_SELECT_MAX_BLOCKS, "pbs_estimate_select: bad shape");
  SelectArgs a = {};
  a.thr_rows = threshold_per_row; a.thr = threshold;
  a.force_first = force_first;
  a.first_blk = const_cast<int32_t*>(first_blk);
  a.nb = nb; a.bs = block_size; a.bps = segment_size / block_size; a.S = S;
  a.needed = block_needed;
  a.cand_rule = (int)rule;
  a.in_place = rule == Candidates::UP_TO_DIAGONAL;
  const dim3 grid((unsigned)((nb + 3) / 4), (unsigned)rows);
  const Divisor sqrt_d = pbs_sqrt_divisor(head_dim);
  hipLaunchKernelGGL(a.in_place ? estimate_select_kernel<true> : estimate_select_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)pooled_q, (const uint16_t*)pooled_k, a,
                     lists, sqrt_d);
  return pbs_check_launch("pbs_estimate_select");
}
