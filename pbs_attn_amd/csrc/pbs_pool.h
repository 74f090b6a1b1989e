// The pooling of query blocks: a workgroup of 256 threads per block.  Shared by the launches it rides in: the pooling of key blocks, or the
// segment sort, which leaves the memory idle.
#pragma once
#include "pbs_lists.h"

namespace {

constexpr int POOL_D = 128, POOL_BS = 128;

// Mean / max pooling of Q blocks (rows past S count as zeros, the divisor stays 128).
__device__ __forceinline__ void pool_q_block(float (&pool)[16][POOL_D], const PoolQ& p, int qb, int bh) {
  const uint16_t* q = p.q;
  const int Hq = p.Hq, S = p.S, nb = p.nb, pool_max = p.pool_max;
  const int b = bh / Hq, h = bh % Hq;
  const int rg = threadIdx.x >> 4, c = threadIdx.x & 15;
  const uint16_t* src = q + b * p.q_sb + h * p.q_sh;
  // all eight loads in flight before the first is used; rows past the end read the last row and count as zeros
  u32x4 x[8];
#pragma unroll
  for (int pass = 0; pass < 8; ++pass) {
    const int pos = qb * POOL_BS + pass * 16 + rg;
    x[pass] = *reinterpret_cast<const u32x4*>(src + (int64_t)min(pos, S - 1) * p.q_ss + c * 8);
  }
#pragma unroll
  for (int pass = 0; pass < 8; ++pass)
    if (qb * POOL_BS + pass * 16 + rg >= S) x[pass] = (u32x4){0, 0, 0, 0};
  float acc[8];
  if (pool_max) {
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = -INFINITY;
#pragma unroll
    for (int pass = 0; pass < 8; ++pass)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[2 * e] = fmaxf(acc[2 * e], bf16_bits_to_f32(x[pass][e] & 0xffffu));
        acc[2 * e + 1] = fmaxf(acc[2 * e + 1], bf16_bits_to_f32(x[pass][e] >> 16));
      }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
#pragma unroll
    for (int pass = 0; pass < 8; ++pass)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[2 * e] += bf16_bits_to_f32(x[pass][e] & 0xffffu);
        acc[2 * e + 1] += bf16_bits_to_f32(x[pass][e] >> 16);
      }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) pool[rg][c * 8 + e] = acc[e];
  __syncthreads();
  if (threadIdx.x < POOL_D) {
    float s = pool[0][threadIdx.x];
    for (int r = 1; r < 16; ++r) s = pool_max ? fmaxf(s, pool[r][threadIdx.x]) : s + pool[r][threadIdx.x];
    if (!pool_max) s = s / (float)POOL_BS;
    p.pooled_q[((int64_t)bh * nb + qb) * POOL_D + threadIdx.x] = (uint16_t)f32_to_bf16_bits(s);
  }
}

}  // namespace
