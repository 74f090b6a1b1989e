// Causal attention of sequences of up to 128 tokens: one key block, one tile.
//
// What bounds it is latency, the chain from the launch to the last store, on a chip that is nearly idle.  The persistent kernel
// (pbs_attn.hip) spends 21 000 cycles on such an item, 3 800 of them on the tile: its list and hand-over to a next item, both tiles through
// LDS for one wave a SIMD, four sub-tiles one after the other in each.  Here a workgroup takes 32 queries of a head, so that a head has up to four, and the
// chain is: queries and keys straight into registers as fragments, 32 keys a wave; the maxima of the four
// sub-tiles exchanged through LDS; the probabilities likewise; then each wave 32 columns of the output over all keys.  V's rows
// come into LDS meanwhile and are read transposed.  32 / 8 heads x 77 tokens: 9.6 -> 4.7 us a launch.
//
// The arithmetic is that of the persistent kernel's first diagonal tile, operation by operation (online softmax over sub-tiles
// of 32 keys, ascending, those behind the workgroup's queries left out): the same bits.
#include "pbs_attn_block.h"
#include "pbs_attn_tile.h"

namespace {

constexpr int ROWS = 32;             // queries of a workgroup, and keys of a sub-tile
constexpr int SUBS = BS / ROWS;

__global__ __launch_bounds__(THREADS) void one_block_attn_kernel(OneBlockArgs a) {
  __shared__ __attribute__((aligned(1024))) uint8_t v_tile[TILE_BYTES];
  __shared__ bf16x8 probs[SUBS][2][PBS_WAVE];
  __shared__ float maxima[SUBS][ROWS], sums[SUBS][ROWS];
  const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int i16 = lane & 15, g4 = lane >> 4;
  const int h = blockIdx.x, b = blockIdx.z, part = (int)(gridDim.y - 1 - blockIdx.y);   // (the workgroups with the most sub-tiles first)
  const int kvh = a.group_magic ? (int)(((uint64_t)(uint32_t)h * a.group_magic) >> 32) : h;
  const int last = a.S - 1;
  const float c_log2 = a.scale_log2;
  const bool has_keys = wave <= part;   // sub-tile `wave` has keys that the workgroup's queries see

  // Rows past the end of the sequence read its last one: such keys lie after every query, such queries are not stored.
  bf16x8 qf[2][4], kf[2][4];
  if (has_keys) {
    const uint16_t* const q = a.q + b * a.q_sb + h * a.q_sh + 8 * g4;
    const uint16_t* const k = a.k + b * a.k_sb + kvh * a.k_sh + 8 * g4;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const uint16_t* const qrow = q + (int64_t)min(ROWS * part + 16 * n + i16, last) * a.q_ss;
      const uint16_t* const krow = k + (int64_t)min(ROWS * wave + 8 * (i16 >> 2) + 4 * n + (i16 & 3), last) * a.k_ss;
#pragma unroll
      for (int kd = 0; kd < 4; ++kd) {
        qf[n][kd] = *reinterpret_cast<const bf16x8*>(qrow + 32 * kd);
        kf[n][kd] = *reinterpret_cast<const bf16x8*>(krow + 32 * kd);
      }
    }
    // V rows into the layout of the transposing reads (see pbs_attn_tile.h)
    const uint16_t* const v = a.v + b * a.v_sb + kvh * a.v_sh + 8 * (2 * (lane >> 3) + (lane & 1));
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const uint16_t* const vrow = v + (int64_t)min(ROWS * wave + 4 * n + ((lane >> 1) & 3), last) * a.v_ss;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)vrow,
                                       (__attribute__((address_space(3))) void*)(v_tile + wave * 8192 + n * 1024), 16, 0, 0);
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  f32x4 s[2][2];   // [row tile][column group]
  if (has_keys) {
#pragma unroll
    for (int T = 0; T < 2; ++T)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        s[T][q] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kd = 0; kd < 4; ++kd) s[T][q] = PBS_MFMA(kf[T][kd], qf[q][kd], s[T][q]);
      }
    if (wave == part) {   // keys after the query
      const int qrel8 = i16 - 8 * g4;
#pragma unroll
      for (int T = 0; T < 2; ++T)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (4 * T + r - 16 * q > qrel8) s[T][q][r] = -INFINITY;
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      float mx = max3(s[0][q][0], s[0][q][1], s[0][q][2]);
      mx = max3(mx, s[0][q][3], s[1][q][0]);
      mx = max3(mx, s[1][q][1], s[1][q][2]);
      mx = max_over_lane_groups(max3(mx, mx, s[1][q][3])) * c_log2;
      if (g4 == 0) maxima[wave][16 * q + i16] = mx;
    }
  }
  __syncthreads();

  // the running maxima, by every wave: what earlier sums are scaled by at each sub-tile, and this wave's own reference
  float alpha[SUBS][2], m_own[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float m = -INFINITY;
#pragma unroll
    for (int ks = 0; ks < SUBS; ++ks) {
      if (ks > part) break;
      const float m_new = fmaxf(m, maxima[ks][16 * q + i16]);
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
      alpha[ks][q] = __builtin_amdgcn_exp2f(m - m_use);
      if (ks == wave) m_own[q] = m_use;
      m = m_new;
    }
  }
  if (has_keys) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      float rs = 0.f;
      bf16x8 pf;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float pe = __builtin_amdgcn_exp2f(s[e >> 2][q][e & 3] * c_log2 - m_own[q]);
        rs += pe;
        pf[e] = (__bf16)pe;
      }
      probs[wave][q][lane] = pf;
      rs = sum_over_lane_groups(rs);
      if (g4 == 0) sums[wave][16 * q + i16] = rs;
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's rows of V have landed
  __syncthreads();

  const uint32_t vr = vrow_lane_addr((uint32_t)(uintptr_t)(lds_u8*)v_tile, lane) + (uint32_t)wave * 256u;   // d tiles 2 wave, 2 wave + 1
  f32x4 o[2][2];   // [d tile][column group]
  float l[2] = {0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < SUBS; ++ks) {
    if (ks > part) break;
#pragma unroll
    for (int q = 0; q < 2; ++q) l[q] = l[q] * alpha[ks][q] + sums[ks][16 * q + i16];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const bf16x8 fv = ldsf_transposed(vr + t * 128 + ks * 8192);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (ks == 0) {
          o[t][q] = (f32x4){0.f, 0.f, 0.f, 0.f};
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) o[t][q][r] *= alpha[ks][q];
        }
        o[t][q] = PBS_MFMA(fv, probs[ks][q][lane], o[t][q]);
      }
    }
  }

  // normalise and store: 16 bytes a lane once the odd and even lane groups have exchanged between the two d tiles
  uint16_t* const orow = a.o + b * a.o_sb + h * a.o_sh + 32 * wave + 16 * (g4 & 1) + 8 * (g4 >> 1);
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const float inv = l[q] == 0.f ? 0.f : 1.0f / l[q];
    uint32_t two[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 2; ++e)
        two[t][e] = __builtin_bit_cast(uint32_t, (bf16x2){(__bf16)(o[t][q][2 * e] * inv), (__bf16)(o[t][q][2 * e + 1] * inv)});
    const auto lo = __builtin_amdgcn_permlane16_swap(two[0][0], two[1][0], false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(two[0][1], two[1][1], false, false);
    const int row = ROWS * part + 16 * q + i16;
    if (row < a.S) *reinterpret_cast<u32x4*>(orow + row * a.o_ss) = (u32x4){lo[0], hi[0], lo[1], hi[1]};
  }
}

}  // namespace

int pbs_one_block_attn_launch(OneBlockArgs a, int B, int Hq, int Hkv, void* stream) {
  const int group = Hq / Hkv;
  a.group_magic = group == 1 ? 0u : (uint32_t)((1ull << 32) / group + 1);   // exact for heads and groups below 65536
  hipLaunchKernelGGL(one_block_attn_kernel, dim3((unsigned)Hq, (unsigned)((a.S + ROWS - 1) / ROWS), (unsigned)B), dim3(THREADS), 0,
                     (hipStream_t)stream, a);
  return pbs_check_launch("pbs_sparse_attn_fwd");
}
