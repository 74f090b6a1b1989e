// Key scoring: mean over the last 128 queries of softmax(Q_last K^T / sqrt(D))
// over all keys of the complete segments (no causal mask).
//
// Two or three launches, K is read twice (each time once per workgroup, through LDS) and never re-materialised:
//   (all exponentials are base 2 on logits pre-multiplied by log2(e))
//   1. score_partial : per (head, key chunk) online (max, sum-exp) of every query row
//   2. score_reduce  : fold the chunk partials into row max + log2(row sum) (short sequences: part of 3)
//   3. score_final   : recompute the logits and emit the per-key mean probability
// Logits reproduce the rounding points of a bf16 matmul followed by a bf16
// divide: fp32 accumulate -> bf16 -> / sqrt(D) -> bf16.
#include "pbs_lists.h"
#include "pbs_sort.h"
#include "../../include/pbs_hip.h"   // the definitions below are checked against the public declarations
#include <algorithm>
#include <atomic>
#include <mutex>

namespace {

constexpr int D = 128;             // head dim
constexpr int NQ = 128;            // scoring queries (= block size)
constexpr int KEYS_PER_WAVE_STEP = 32;
constexpr int KEYS_PER_WG = 1024;  // keys one 4-wave workgroup walks through (256 for 1-wave groups)

struct ScoreArgs {
  const uint16_t* q;
  const uint16_t* k;
  int B, Hq, Hkv, S, Sc;
  int64_t q_sb, q_sh, q_ss;
  int64_t k_sb, k_sh, k_ss;
  float inv_sqrt_d;
  float* part;    // (B*Hq, nchunk, NQ, 2)
  float* stats;   // (B*Hq, NQ)  row max + log2(row sum)
  float* scores;  // (B*Hq, Sc)
  int nchunk;
  int chunk_keys;
  int32_t* idx;        // (SORT) order of the keys (B*Hq, S_pad) and the block that holds key 0 (B*Hq)
  int32_t* first_blk;
  int S_pad, block_size;
};

__device__ __forceinline__ bf16x8 load_frag(const uint16_t* row_ptr, int t, int half) {
  return *reinterpret_cast<const bf16x8*>(row_ptr + 16 * t + 8 * half);
}

// fp32 accumulator -> the bf16 logit a bf16 matmul followed by a bf16 divide by sqrt(D) yields: round to
// bf16, scale (multiplication by the reciprocal; it differs from the true quotient by at most one fp32 ulp,
// which survives the second bf16 rounding only for values within 2^-16 of a tie), round to bf16.
// Hardware conversions (round to nearest even), two values per conversion instruction.
__device__ __forceinline__ f32x2 logit2(float acc0, float acc1, float inv_sqrt_d) {
  const f32x2 r = hw_round_bf16x2((f32x2){acc0, acc1});
  return hw_round_bf16x2((f32x2){r.x * inv_sqrt_d, r.y * inv_sqrt_d});
}
constexpr float LOG2E = 1.4426950408889634f;

// ---- key rows through LDS: the waves of a workgroup (one per query head of the KV group) walk the same keys,
// so a stage of 64 key rows is copied once per workgroup with asynchronous global -> LDS copies (no registers),
// double-buffered, and every wave reads its MFMA fragments from there.  Rows are 16 chunks of 16 bytes with the
// chunk index XORed with (row & 15): fragment reads (row = lane % 32, one chunk) are bank-conflict free.  The copy
// instruction writes lane l at M0 + 16 l, so the swizzle is applied on the global side: lane l of copy i fetches
// chunk (l & 15) ^ (row & 15) of row 4 i + (l >> 4).
constexpr int STAGE_KEYS = 64;
constexpr uint32_t STAGE_BYTES = STAGE_KEYS * D * 2;      // 16 KB
constexpr uint32_t LDS_STATS = 2 * STAGE_BYTES;           // per wave: NQ floats (row max + log2 row sum)
constexpr uint32_t LDS_SCORE_TOTAL = LDS_STATS + 4 * NQ * 4;   // (SPLIT: NQ statistics and 4 x STAGE_KEYS sums)
constexpr int SPLIT_MAX_CHUNKS = 32;                      // the final pass of the split form folds a query's chunks itself
static_assert(STAGE_KEYS == PBS_WAVE && NQ + 4 * STAGE_KEYS <= 4 * NQ, "sums and statistics of the split form");

typedef __attribute__((address_space(3))) uint8_t lds_u8;

__device__ __forceinline__ bf16x8 lds_frag(uint32_t byte_addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>((const lds_u8*)(uintptr_t)byte_addr);
}

// copies of rows [0, STAGE_KEYS) starting at `rows` (row stride k_ss elements) into the stage buffer at LDS byte
// offset `lds_byte`; wave w of nwaves issues copies w, w + nwaves, ...
__device__ __forceinline__ void stage_keys_async(const uint16_t* rows, int64_t k_ss, uint32_t lds_byte, int wave, int nwaves, int lane) {
  const uint64_t src0 = (uint64_t)(uintptr_t)rows;
  const uint32_t src_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)src0);
  const uint32_t src_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(src0 >> 32));
  const uint64_t srcu = ((uint64_t)src_hi << 32) | (uint64_t)src_lo;
  const uint32_t row_bytes = (uint32_t)k_ss * 2u;   // < 2^29 (checked on the host)
  for (int i = wave; i < STAGE_KEYS / 4; i += nwaves) {
    const uint32_t r = (uint32_t)(lane >> 4);
    const uint32_t c = (uint32_t)(lane & 15) ^ ((4u * (uint32_t)(i & 3) + r) & 15u);
    const uint32_t voff = r * row_bytes + c * 16u;
    const uint64_t base = srcu + (uint64_t)(4 * i) * row_bytes;
    register uint32_t m0v asm("m0") = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_byte + (uint32_t)i * 1024u));
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0v), "v"(voff), "s"(base) : "memory");
  }
}

// One wave per query head of the KV group; the waves of a workgroup share the staged key rows.  SPLIT (short sequences, see
// score_plan): the four waves take 32 queries each of ONE head.
// Waves per SIMD: the final pass of the split form needs 147 registers and would spill 18 of them at four.
// SORT: a workgroup of the final split pass takes a whole segment of up to 256 keys, keeps its scores in LDS, and ranks them: no launch, and
// no way to memory and back, for the sort.
template <bool FINAL, bool SPLIT, bool SORT = false>
__global__ __launch_bounds__(256, SPLIT ? (FINAL ? 3 : 4) : 2) void score_kernel(ScoreArgs a) {
  constexpr int QT = SPLIT ? 1 : NQ / 32;   // query tiles of a wave
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];   // starts at LDS offset 0: this kernel has no static LDS
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int j = lane & 31, half = lane >> 5;
  const int G = a.Hq / a.Hkv;
  const int b = blockIdx.y / (SPLIT ? a.Hq : a.Hkv), in_batch = blockIdx.y % (SPLIT ? a.Hq : a.Hkv);
  const int kvh = SPLIT ? in_batch / G : in_batch;
  const int q_first = SPLIT ? 32 * wave : 0;
  const int chunk = blockIdx.x;
  const int key_lo = chunk * a.chunk_keys;
  const int key_hi = min(key_lo + a.chunk_keys, a.Sc);   // chunk_keys and Sc are multiples of STAGE_KEYS
  const int nwaves = (int)blockDim.x >> 6;
  const uint16_t* kbase = a.k + b * a.k_sb + kvh * a.k_sh;
  float* s_stats = reinterpret_cast<float*>(smem + LDS_STATS) + wave * (32 * QT);   // p = exp2(logit - stat)
  float* s_sums = reinterpret_cast<float*>(smem + LDS_STATS) + NQ;   // SPLIT: a wave's sums of the stage's keys
  double* s_keys = reinterpret_cast<double*>(smem + LDS_SCORE_TOTAL);   // SORT: the segment's sort keys
  // LDS byte offset of fragment 0 of key row j inside a stage buffer; fragment t lies at frag0 ^ (t << 5),
  // rows 32 .. 63 of the stage 8 KB further on
  const uint32_t frag0 = (uint32_t)(j * 256 + ((half ^ (j & 15)) * 16));
  const int n_stages = (key_hi - key_lo) / STAGE_KEYS;

  for (int g0 = 0; g0 < (SPLIT ? 1 : G); g0 += nwaves) {
    const int g = SPLIT ? in_batch - kvh * G : g0 + wave;
    const bool active = g < G;
    const int h = kvh * G + (active ? g : 0);
    const int bh = b * a.Hq + h;
    const uint16_t* qbase = a.q + b * a.q_sb + h * a.q_sh + (int64_t)(a.S - NQ) * a.q_ss;

    __syncthreads();   // every wave is done with the stage buffers (and the statistics) of the previous group of heads
    stage_keys_async(kbase + (int64_t)key_lo * a.k_ss, a.k_ss, 0u, wave, nwaves, lane);

    // the wave's scoring queries, resident for the whole chunk
    bf16x8 qf[QT][8];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int t = 0; t < 8; ++t) qf[qt][t] = load_frag(qbase + (int64_t)(q_first + 32 * qt + j) * a.q_ss, t, half);

    if (FINAL && SPLIT) {
      // a query's chunks are few enough to be folded here: two lanes a query, all loads in flight
      const float* p = a.part + ((int64_t)bh * a.nchunk * NQ + q_first + j) * 2;
      float2 ml[SPLIT_MAX_CHUNKS / 2];
#pragma unroll
      for (int c = 0; c < SPLIT_MAX_CHUNKS / 2; ++c)
        ml[c] = *reinterpret_cast<const float2*>(p + (int64_t)min(2 * c + half, a.nchunk - 1) * NQ * 2);
      float m = ml[0].x, l = 0.f;   // (a chunk read twice does not move the maximum)
#pragma unroll
      for (int c = 1; c < SPLIT_MAX_CHUNKS / 2; ++c) m = fmaxf(m, ml[c].x);
      m = fmaxf(m, xhalf_f32(m));
#pragma unroll
      for (int c = 0; c < SPLIT_MAX_CHUNKS / 2; ++c)
        l += 2 * c + half < a.nchunk ? ml[c].y * __builtin_amdgcn_exp2f(ml[c].x - m) : 0.f;
      l += xhalf_f32(l);
      if (half == 0) s_stats[j] = m + __builtin_amdgcn_logf(l);   // log base 2
    } else if (FINAL && active) {
      for (int i = lane; i < NQ; i += 64) s_stats[i] = a.stats[(int64_t)bh * NQ + i];
    }

    float m_run[QT], l_run[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      m_run[qt] = -INFINITY;
      l_run[qt] = 0.f;
    }

    for (int st = 0; st < n_stages; ++st) {
      const uint32_t buf = (uint32_t)(st & 1) * STAGE_BYTES;
      __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's copies of stage st have landed
      __syncthreads();                      // every wave's have; everyone is done with the other buffer
      if (st + 1 < n_stages)
        stage_keys_async(kbase + (int64_t)(key_lo + (st + 1) * STAGE_KEYS) * a.k_ss, a.k_ss, buf ^ STAGE_BYTES, wave, nwaves, lane);
      if (!active) continue;
      // Eight logit tiles (32 keys x 32 queries) per stage (SPLIT: two), one ahead: the matrix instructions of tile i + 1 go out among the
      // vector work of tile i (left to itself the compiler issues a tile's eight in a row, each waiting for the one
      // before).  What bounds the pass is the vector unit: per pair of logits 4 conversions, 2 multiplications, 2 multiply-adds,
      // 2 exponentials (two slots each), 2 additions and, here, a maximum.  Both passes together: 256k head shard
      // 210 -> 193 us, 128k 418 -> 397 us, 32k 111 -> 107 us (with the one-instruction rounding of pbs_common.h).
      constexpr int TILES = QT * STAGE_KEYS / KEYS_PER_WAVE_STEP;
      bf16x8 kf[8];
      f32x16 acc_next = {0};
      auto load_keys = [&](int sub) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 8; ++t) kf[t] = lds_frag(buf + (uint32_t)sub * 8192u + (frag0 ^ (uint32_t)(t << 5)));
      };
      auto multiply = [&](int qt) __attribute__((always_inline)) {
        acc_next = (f32x16){0};
#pragma unroll
        for (int t = 0; t < 8; ++t)   // rows = keys and columns = queries, or (FINAL) the other way round
          acc_next = FINAL ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[qt][t], kf[t], acc_next, 0, 0, 0)
                           : __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[t], qf[qt][t], acc_next, 0, 0, 0);
      };
      load_keys(0);
      multiply(0);
      __builtin_amdgcn_sched_barrier(0);
      float accp = 0.f;
#pragma unroll
      for (int i = 0; i < TILES; ++i) {
        const int sub = i / QT, qt = i % QT;
        const f32x16 acc = acc_next;
        if (qt == QT - 1 && i + 1 < TILES) load_keys(sub + 1);
        if (i + 1 < TILES) multiply((i + 1) % QT);
        if (!FINAL) {
          float v[16], mx = -INFINITY;   // logits before the log2(e) factor
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            const f32x2 l2 = logit2(acc[r], acc[r + 1], a.inv_sqrt_d);
            v[r] = l2.x;
            v[r + 1] = l2.y;
            mx = fmaxf(fmaxf(mx, l2.x), l2.y);
          }
          const float m_new = fmaxf(m_run[qt], mx * LOG2E);
          float sum = 0.f;
#pragma unroll
          for (int r = 0; r < 16; ++r) sum += __builtin_amdgcn_exp2f(__builtin_fmaf(v[r], LOG2E, -m_new));
          l_run[qt] = l_run[qt] * __builtin_amdgcn_exp2f(m_run[qt] - m_new) + sum;
          m_run[qt] = m_new;
        } else {
#pragma unroll
          for (int r4 = 0; r4 < 4; ++r4) {
            const float4 st4 = *reinterpret_cast<const float4*>(&s_stats[32 * qt + 8 * r4 + 4 * half]);
            const f32x2 la = logit2(acc[4 * r4 + 0], acc[4 * r4 + 1], a.inv_sqrt_d);
            const f32x2 lb = logit2(acc[4 * r4 + 2], acc[4 * r4 + 3], a.inv_sqrt_d);
            accp += __builtin_amdgcn_exp2f(__builtin_fmaf(la.x, LOG2E, -st4.x));
            accp += __builtin_amdgcn_exp2f(__builtin_fmaf(la.y, LOG2E, -st4.y));
            accp += __builtin_amdgcn_exp2f(__builtin_fmaf(lb.x, LOG2E, -st4.z));
            accp += __builtin_amdgcn_exp2f(__builtin_fmaf(lb.y, LOG2E, -st4.w));
          }
        }
        if (i + 1 < TILES) {
#pragma unroll
          for (int t = 0; t < 8; ++t) {
            if (qt == QT - 1 && t == 0) {   // the next keys, and time for them to arrive
              __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
              __builtin_amdgcn_sched_group_barrier(0x2, 30, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x2, 11, 0);                           // vector instructions
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                            // a matrix instruction
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (FINAL && qt == QT - 1) {
          const float total = accp + xhalf_f32(accp);
          accp = 0.f;
          const int in_stage = sub * KEYS_PER_WAVE_STEP + j;
          const int key = key_lo + st * STAGE_KEYS + in_stage;   // always < Sc
          if (half == 0) {
            if (SPLIT) s_sums[wave * STAGE_KEYS + in_stage] = total;
            else a.scores[(int64_t)bh * a.Sc + key] = total * (1.0f / NQ);
          }
        }
      }
      if (FINAL && SPLIT) {
        __syncthreads();   // (the next stage's sums are written behind its first barrier)
        if (wave == 0) {
          const float* s = s_sums + lane;
          const float score = ((s[0] + s[STAGE_KEYS]) + (s[2 * STAGE_KEYS] + s[3 * STAGE_KEYS])) * (1.0f / NQ);
          if (SORT) s_keys[st * STAGE_KEYS + lane] = sort_key(score, (uint32_t)(st * STAGE_KEYS + lane));
          else a.scores[(int64_t)bh * a.Sc + key_lo + st * STAGE_KEYS + lane] = score;
        }
      }
    }
    if constexpr (SORT) {
      int32_t* row = a.idx + (int64_t)bh * a.S_pad;
      __syncthreads();
      const int i = threadIdx.x;
      if (i < a.chunk_keys) {
        const int rank = rank_of(s_keys[i], s_keys, a.chunk_keys);
        row[key_lo + rank] = key_lo + i;
        if (chunk == 0 && i == 0 && a.first_blk) a.first_blk[bh] = rank / a.block_size;
      }
      if (chunk == 0) {   // the remainder of the sequence and the block padding keep their places
        for (int i = a.Sc + (int)threadIdx.x; i < a.S_pad; i += 256) row[i] = i;
      }
    }
    if (!FINAL && active) {
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        const float m_o = xhalf_f32(m_run[qt]), l_o = xhalf_f32(l_run[qt]);
        const float m_new = fmaxf(m_run[qt], m_o);
        const float l_new = l_run[qt] * __builtin_amdgcn_exp2f(m_run[qt] - m_new) + l_o * __builtin_amdgcn_exp2f(m_o - m_new);
        if (half == 0) {
          float* p = a.part + (((int64_t)bh * a.nchunk + chunk) * NQ + q_first + 32 * qt + j) * 2;
          p[0] = m_new;
          p[1] = l_new;
        }
      }
    }
  }
}

// Folds the chunk partials of one head into row max + log2(row sum).  A row's chunks are spread over REDUCE_LANES
// threads and taken in two passes -- the maximum over all chunks, then the sum of the chunk sums scaled to it -- so
// that no term waits for the one before it: folded one after the other with a running maximum, a row is a chain of
// `nchunk` dependent loads and exponentials (19 us for 64 chunks, as long as the two scoring passes of a short
// sequence together).  The order of the additions is fixed: per thread ascending chunks, then ascending threads.
constexpr int REDUCE_LANES = 8;

__global__ __launch_bounds__(NQ * REDUCE_LANES) void score_reduce_kernel(ScoreArgs a) {
  __shared__ float part[REDUCE_LANES][NQ];
  const int bh = blockIdx.x, qrow = threadIdx.x % NQ, cl = threadIdx.x / NQ;
  const float* p = a.part + (int64_t)bh * a.nchunk * NQ * 2 + qrow * 2;
  float m = -INFINITY;
#pragma unroll 8
  for (int c = cl; c < a.nchunk; c += REDUCE_LANES) m = fmaxf(m, p[(int64_t)c * NQ * 2]);
  part[cl][qrow] = m;
  __syncthreads();
#pragma unroll
  for (int x = 0; x < REDUCE_LANES; ++x) m = fmaxf(m, part[x][qrow]);
  __syncthreads();
  float l = 0.f;
#pragma unroll 8
  for (int c = cl; c < a.nchunk; c += REDUCE_LANES) {
    const float2 ml = *reinterpret_cast<const float2*>(p + (int64_t)c * NQ * 2);
    l += ml.y * __builtin_amdgcn_exp2f(ml.x - m);
  }
  part[cl][qrow] = l;
  __syncthreads();
  if (cl == 0) {
    l = 0.f;
#pragma unroll
    for (int x = 0; x < REDUCE_LANES; ++x) l += part[x][qrow];
    a.stats[(int64_t)bh * NQ + qrow] = m + __builtin_amdgcn_logf(l);   // log base 2
  }
}

int chunks_for(int Sc, int chunk_keys) { return (Sc + chunk_keys - 1) / chunk_keys; }

// Keys per workgroup.  With one query head per KV head a workgroup is a single wave and starts from a
// quarter of the keys; short sequences get shorter chunks until the launch has enough workgroups to
// fill the chip (each workgroup re-reads its heads' 128 queries, so chunks stay >= 64 keys).
//
// The split form (a workgroup's waves share one head's queries) has 4 G workgroups for every 4 query heads of a KV head, a
// quarter of the serial work and registers per wave, and folds the chunk partials without a launch of its own, but it stages each
// key row once per query head.  It takes:
//   * short sequences, where the grouped form leaves the chip idle or waiting.  Whole pass, grouped -> split, us: 28 / 4 heads x
//     1000 keys 93.9 -> 72.9 (the three launches 37.4 -> 14.2, two launches), 32 / 8 x 600 66.7 -> 57.4, x 4096 191.9 -> 184.0, x 6000
//     338 -> 328, 16 / 4 x 12000 526 -> 516; equal at 32 / 8 x 8192 (501, 504) and 4 / 1 x 30000, slower at 4 / 1 x 40000 (654 -> 681:
//     SPLIT_MAX_CHUNKS workgroups a head no longer fill the chip), hence the two limits;
//   * groups that leave waves of the grouped form idle: 28 / 4 x 9000 601 -> 567, 16 / 16 x 20000 783 -> 763 and x 131072 1485 ->
//     1409, 8 / 8 x 131072 790 -> 760, 16 / 8 x 32768 460 -> 430, 14 / 2 x 65536 632 -> 624; at 28 / 4 x 65536, where an eighth is
//     idle, the two are equal (1193, 1196), hence the limit for groups with less than a quarter idle.
// A short sequence's workgroups all run at once, three a CU: one more round costs more than the longer chunk (a stage of 64 keys 1.2 us a
// pass).  Whole pass: 32 / 8 heads x 2048, 1024 workgroups of 64 keys -> 512 of 128, 93.9 -> 90.7 us; x 4096, 1024 of 128 -> 512 of 256,
// 167.5 -> 165.8; 28 / 4 x 4096 153.3 -> 151.5; fewer than they have to be: 16 / 16 x 2048, 512 -> 256, 65.5 -> 69.4.  More heads than
// that do not run at once even with one chunk each: theirs stay short (and the doubling would have no end).
constexpr int SPLIT_WORKGROUPS = 3 * 256;
// The final pass sorts where a segment is at most two chunks long, so that a workgroup's serial part hardly grows, and its workgroups still
// run at once (and the gather does not: short passes mostly leave it to that).  Whole pass, sort kernel -> this, us: segments of 128, 4 / 1 heads x 6000 109.7 -> 102.0, x 16384 267.6 ->
// 257.8, 32 x 8 / 2 x 300 81.7 -> 78.0, 16 x 32 / 8 x 200 91.7 -> 88.1; of 256, 4 / 1 x 16384 269.2 -> 259.0, 8 / 2 x 12000 195.5 -> 189.0, 16 / 16 x 12000
// 518 -> 512; everything selected, 28 / 4 x 1019 of 128 52.1 -> 48.0, 32 / 8 x 4096 of 256 164.0 -> 158.8.  Past the limits, measured
// where everything is selected, there is little left in it: segments of four chunks, 8 / 2 x 2048 61.7 -> 60.6; 1024 workgroups, 32 / 8 x 4096 of 128 162.2 -> 161.4; 1536, 24 / 8 x
// 8192 386.5 -> 385.7.
constexpr int SORT_IN_PASS_KEYS = 256;
struct ScorePlan {
  bool split, small;
  int chunk_keys, nchunk;
};
int longest_chunk(bool grouped) { return grouped ? KEYS_PER_WG : KEYS_PER_WG / 4; }
int64_t workgroups_wanted(bool grouped) { return grouped ? 512 : 2048; }
ScorePlan score_plan(int B, int Hq, int Hkv, int Sc) {
  const bool grouped = Hq / Hkv > 1;
  int chunk = longest_chunk(grouped);
  const int64_t want = workgroups_wanted(grouped);
  while (chunk > 64 && (int64_t)chunks_for(Sc, chunk) * B * Hkv < want) chunk /= 2;
  const int64_t heads = (int64_t)B * Hq, keys = heads * Sc;
  const int G = Hq / Hkv, slots = (G + 3) / 4 * 4, idle = slots - G;
  const bool small = keys <= 3 << 16 && Sc <= 16384;
  const bool uneven = idle > 0 && heads >= 8 && (4 * idle >= slots || keys <= 1 << 20);
  const bool split = (small || uneven) && heads <= 65535;
  const bool at_once = small && heads <= SPLIT_WORKGROUPS;
  if (split)
    while (chunks_for(Sc, chunk) > SPLIT_MAX_CHUNKS || (at_once && chunks_for(Sc, chunk) * heads > SPLIT_WORKGROUPS)) chunk *= 2;
  return {split, small, chunk, chunks_for(Sc, chunk)};
}

}  // namespace

extern "C" size_t pbs_score_keys_workspace_bytes(int B, int Hq, int Hkv, int S, int segment_size) {
  if (segment_size <= 0 || B <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv) return 0;
  const int Sc = (S / segment_size) * segment_size;
  if (Sc == 0) return 0;
  return (size_t)B * Hq * ((size_t)score_plan(B, Hq, Hkv, Sc).nchunk + 1) * NQ * 2 * sizeof(float);
}

size_t pbs_score_keys_workspace_bound(int B, int Hq, int Hkv, int S, int segment_size) {
  const int Sc = (S / segment_size) * segment_size;
  if (Sc == 0) return 0;
  // A chunk is the longest one, or half of one that gave fewer workgroups than wanted, or longer (score_plan); 64 keys and more.
  const bool grouped = Hq / Hkv > 1;
  const int64_t halved = 2 * ((workgroups_wanted(grouped) - 1) / ((int64_t)B * Hkv));
  const int64_t chunks = std::min<int64_t>(chunks_for(Sc, 64), std::max<int64_t>(chunks_for(Sc, longest_chunk(grouped)), halved));
  return (size_t)B * Hq * ((size_t)chunks + 1) * NQ * 2 * sizeof(float);
}

namespace {

// Argument checks and the three launches shared by the two entry points; `workspace` holds the chunk
// partials and the folded row statistics.
int score_keys_launch(const char* who, const void* q, const void* k, float* scores, int B, int Hq, int Hkv, int S,
                      int head_dim, int block_size, int segment_size, int64_t q_sb, int64_t q_sh, int64_t q_ss,
                      int64_t k_sb, int64_t k_sh, int64_t k_ss, void* workspace, size_t workspace_bytes, void* stream,
                      int32_t* idx = nullptr, int32_t* first_blk = nullptr, int S_pad = 0) {
  PBS_REQUIRE(q && k && (scores || idx), "%s: null tensor pointer", who);
  PBS_REQUIRE(head_dim == D, "%s: head_dim must be 128, got %d", who, head_dim);
  PBS_REQUIRE(block_size == NQ, "%s: block_size must be 128, got %d", who, block_size);
  PBS_REQUIRE(B > 0 && Hkv > 0 && Hq > 0 && Hq % Hkv == 0, "%s: bad head counts Hq=%d Hkv=%d", who, Hq, Hkv);
  PBS_REQUIRE(segment_size > 0 && segment_size % block_size == 0, "%s: segment_size %d not a multiple of block_size", who, segment_size);
  PBS_REQUIRE(S >= NQ, "%s: sequence shorter than one block", who);
  PBS_REQUIRE(q_ss % 8 == 0 && k_ss % 8 == 0 && q_sh % 8 == 0 && k_sh % 8 == 0 && q_sb % 8 == 0 && k_sb % 8 == 0,
              "%s: strides must keep rows 16-byte aligned", who);
  PBS_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0, "%s: pointers must be 16-byte aligned", who);
  PBS_REQUIRE(k_ss >= D && k_ss < (1 << 28), "%s: key row stride %lld outside [128, 2^28)", who, (long long)k_ss);
  PBS_REQUIRE((int64_t)B * Hkv <= 65535, "%s: too many KV heads (%lld)", who, (long long)B * Hkv);
  const int Sc = (S / segment_size) * segment_size;
  if (Sc == 0) return 0;
  PBS_REQUIRE(workspace && workspace_bytes >= pbs_score_keys_workspace_bytes(B, Hq, Hkv, S, segment_size),
              "%s: workspace too small (%zu < %zu bytes)", who, workspace_bytes,
              pbs_score_keys_workspace_bytes(B, Hq, Hkv, S, segment_size));
  ScoreArgs a;
  a.q = (const uint16_t*)q;
  a.k = (const uint16_t*)k;
  a.B = B; a.Hq = Hq; a.Hkv = Hkv; a.S = S; a.Sc = Sc;
  a.q_sb = q_sb; a.q_sh = q_sh; a.q_ss = q_ss;
  a.k_sb = k_sb; a.k_sh = k_sh; a.k_ss = k_ss;
  a.inv_sqrt_d = (float)(1.0 / sqrt((double)head_dim));
  const ScorePlan plan = score_plan(B, Hq, Hkv, Sc);
  a.chunk_keys = plan.chunk_keys;
  a.nchunk = plan.nchunk;
  a.part = (float*)workspace;
  a.stats = a.part + (size_t)B * Hq * a.nchunk * NQ * 2;
  a.scores = scores;
  a.idx = idx; a.first_blk = first_blk; a.S_pad = S_pad; a.block_size = block_size;
  static std::atomic<bool> lds_checked{false};   // once per process: a property of the code object
  if (!lds_checked.load(std::memory_order_acquire)) {
    if (const int rc = pbs_require_no_static_lds((const void*)score_kernel<false, false>, who)) return rc;
    if (const int rc = pbs_require_no_static_lds((const void*)score_kernel<true, false>, who)) return rc;
    if (const int rc = pbs_require_no_static_lds((const void*)score_kernel<false, true>, who)) return rc;
    if (const int rc = pbs_require_no_static_lds((const void*)score_kernel<true, true>, who)) return rc;
    if (const int rc = pbs_require_no_static_lds((const void*)score_kernel<true, true, true>, who)) return rc;
    lds_checked.store(true, std::memory_order_release);
  }
  hipStream_t st = (hipStream_t)stream;
  if (plan.split) {
    const dim3 grid(a.nchunk, B * Hq);
    hipLaunchKernelGGL((score_kernel<false, true>), grid, dim3(256), LDS_SCORE_TOTAL, st, a);
    if (idx) {
      a.chunk_keys = segment_size;
      const dim3 segments(Sc / segment_size, B * Hq);
      hipLaunchKernelGGL((score_kernel<true, true, true>), segments, dim3(256), LDS_SCORE_TOTAL + segment_size * sizeof(double), st, a);
      return pbs_check_launch(who);
    }
    hipLaunchKernelGGL((score_kernel<true, true>), grid, dim3(256), LDS_SCORE_TOTAL, st, a);
    return pbs_check_launch(who);
  }
  dim3 grid(a.nchunk, B * Hkv);
  const dim3 block(Hq / Hkv > 1 ? 256 : 64);
  hipLaunchKernelGGL((score_kernel<false, false>), grid, block, LDS_SCORE_TOTAL, st, a);
  hipLaunchKernelGGL(score_reduce_kernel, dim3(B * Hq), dim3(NQ * REDUCE_LANES), 0, st, a);
  hipLaunchKernelGGL((score_kernel<true, false>), grid, block, LDS_SCORE_TOTAL, st, a);
  return pbs_check_launch(who);
}

}  // namespace

int pbs_score_sort_chunk(int B, int Hq, int Hkv, int S, int segment_size) {
  const int Sc = (S / segment_size) * segment_size;
  if (Sc == 0 || segment_size > SORT_IN_PASS_KEYS || segment_size % STAGE_KEYS) return 0;
  const ScorePlan plan = score_plan(B, Hq, Hkv, Sc);
  const bool sorts = plan.split && plan.small && segment_size <= 2 * plan.chunk_keys && (int64_t)B * Hq * (Sc / segment_size) <= SPLIT_WORKGROUPS;
  return sorts ? plan.chunk_keys : 0;
}

int pbs_score_sort_launch(const void* q, const void* k, int32_t* key_indices, int32_t* first_blk, int B, int Hq, int Hkv, int S, int S_pad,
                          int head_dim, int block_size, int segment_size, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t k_sb,
                          int64_t k_sh, int64_t k_ss, void* workspace, size_t workspace_bytes, void* stream) {
  PBS_REQUIRE(key_indices && pbs_score_sort_chunk(B, Hq, Hkv, S, segment_size), "pbs_score_sort: bad arguments");
  return score_keys_launch("pbs_score_keys", q, k, nullptr, B, Hq, Hkv, S, head_dim, block_size, segment_size, q_sb, q_sh, q_ss, k_sb,
                           k_sh, k_ss, workspace, workspace_bytes, stream, key_indices, first_blk, S_pad);
}

extern "C" int pbs_score_keys(const void* q, const void* k, float* scores, int B, int Hq, int Hkv, int S, int head_dim,
                              int block_size, int segment_size, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t k_sb,
                              int64_t k_sh, int64_t k_ss, void* workspace, size_t workspace_bytes, void* stream) {
  return score_keys_launch("pbs_score_keys", q, k, scores, B, Hq, Hkv, S, head_dim, block_size, segment_size, q_sb, q_sh,
                           q_ss, k_sb, k_sh, k_ss, workspace, workspace_bytes, stream);
}

// ---- the variant that allocates nothing: chunk partials and row statistics live in a library-owned
// device array.  Every GPU holds its own copy of the array at its own address; the address is looked up
// once per device, on that device's first call, and only that pointer is ever handed to kernels.
namespace {

constexpr size_t SCRATCH_BYTES = PBS_SCORE_KEYS_STATIC_SCRATCH_BYTES;   // 8 MiB per GPU, held until the process ends
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_lock;
void* g_scratch_ptr[MAX_DEVICES] = {};

// device pointer of `scratch` on the current device (null + error message on failure)
void* scratch_on_current_device(const char* who) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
    pbs_set_error("%s: cannot identify the current device (%s, device %d)", who, hipGetErrorString(e), dev);
    return nullptr;
  }
  std::lock_guard<std::mutex> hold(g_scratch_lock);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      pbs_set_error("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", who, dev, hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}

}  // namespace

extern "C" int pbs_score_keys_static(const void* q, const void* k, float* scores, int B, int Hq, int Hkv, int S,
                                     int head_dim, int block_size, int segment_size, int64_t q_sb, int64_t q_sh,
                                     int64_t q_ss, int64_t k_sb, int64_t k_sh, int64_t k_ss, void* stream) {
  PBS_REQUIRE(B > 0 && Hkv > 0 && Hq > 0 && Hq % Hkv == 0 && S > 0 && segment_size > 0,
              "pbs_score_keys_static: bad shape B=%d Hq=%d Hkv=%d S=%d segment_size=%d", B, Hq, Hkv, S, segment_size);
  const size_t need = pbs_score_keys_workspace_bytes(B, Hq, Hkv, S, segment_size);
  PBS_REQUIRE(need <= SCRATCH_BYTES,
              "pbs_score_keys_static: this shape needs %zu bytes of scratch memory, the library-owned buffer holds %zu; "
              "use pbs_score_keys with a caller-provided workspace", need, SCRATCH_BYTES);
  void* ws = scratch_on_current_device("pbs_score_keys_static");
  if (!ws) return -2;
  // every partial and statistic the later launches read is written by the earlier ones of this call:
  // nothing needs clearing between calls
  return score_keys_launch("pbs_score_keys_static", q, k, scores, B, Hq, Hkv, S, head_dim, block_size, segment_size,
                           q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, ws, SCRATCH_BYTES, stream);
}
