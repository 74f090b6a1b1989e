// The order of a segment's keys: by one wave in registers (the sort kernel, and the gather of short passes for longer segments), and by ranks in a
// workgroup (that gather and the final scoring pass, segments of up to 256 keys).
#pragma once
#include "pbs_wave.h"

namespace {

// ---- one wave per segment, NPL keys per lane in registers.
// The 32 score bits and an 11-bit index make a 43-bit integer.  As the mantissa of a double in [1, 2) it keeps its order, and
// a compare-exchange inside a lane is one minimum and one maximum of doubles (64-bit integers take a comparison and four
// selects); descending runs carry the keys negated.  Between lanes: two moves, a comparison, two selects, no LDS.
// Segments of 1024, 32 heads x 128k keys: 87 -> 37 us (the LDS network moved each key through memory in all 55 stages);
// segments of 256 at 4k: 10.2 -> 7.2 us.
__device__ __forceinline__ double sort_key(float score, uint32_t index) {
  const uint64_t u = (uint64_t)(~f32_orderable(score)) << 11 | index;
  return __builtin_bit_cast(double, 0x3ff0000000000000ull | u);
}
__device__ __forceinline__ uint32_t sort_key_index(double key) { return (uint32_t)__builtin_bit_cast(uint64_t, key) & 2047u; }

// lane distance LS: the lower lane keeps the smaller key
template <int NPL, int LS>
__device__ __forceinline__ void cross_lane_sort_stage(double (&k)[NPL], int lane) {
  const bool upper = (lane & LS) != 0;
#pragma unroll
  for (int r = 0; r < NPL; ++r) {
    const uint64_t u = __builtin_bit_cast(uint64_t, k[r]);
    const TwoOf lo = with_lane_xor<LS>((uint32_t)u), hi = with_lane_xor<LS>((uint32_t)(u >> 32));
    const double a = __builtin_bit_cast(double, (uint64_t)hi.a << 32 | lo.a), b = __builtin_bit_cast(double, (uint64_t)hi.b << 32 | lo.b);
    const bool first = (a < b) != upper;
    const uint32_t rl = first ? lo.a : lo.b, rh = first ? hi.a : hi.b;
    k[r] = __builtin_bit_cast(double, (uint64_t)rh << 32 | rl);
  }
}
template <int NPL>
__device__ __forceinline__ void local_sort_stages(double (&k)[NPL], int size) {
#pragma unroll
  for (int stride = min(size, NPL) >> 1; stride > 0; stride >>= 1) {
#pragma unroll
    for (int r = 0; r < NPL; ++r) {
      if ((r & stride) == 0) {
        const int p = r | stride;
        const bool up = size >= NPL || (r & size) == 0;
        const double lo = fmin(k[r], k[p]), hi = fmax(k[r], k[p]);
        k[r] = up ? lo : hi;
        k[p] = up ? hi : lo;
      }
    }
  }
}
// ascending; the result's element lane * NPL + r is in register r.  The phases that reach across lanes are a loop over one
// copy of each stage (the unrolled network of a long segment does not fit the instruction cache).
template <int NPL>
__device__ __forceinline__ void wave_sort(double (&k)[NPL], int lane) {
#pragma unroll
  for (int size = 2; size < NPL; size <<= 1) local_sort_stages<NPL>(k, size);
  double sign = 1.0;   // what the keys are multiplied with
#pragma nounroll
  for (int lanes = 1; lanes <= 64; lanes <<= 1) {   // runs of NPL * lanes keys
    const double want = (lane & lanes) ? -1.0 : 1.0, change = want * sign;
#pragma unroll
    for (int r = 0; r < NPL; ++r) k[r] *= change;
    sign = want;
    switch (lanes) {   // strides from lanes / 2 lanes down to one
      case 64: cross_lane_sort_stage<NPL, 32>(k, lane); [[fallthrough]];
      case 32: cross_lane_sort_stage<NPL, 16>(k, lane); [[fallthrough]];
      case 16: cross_lane_sort_stage<NPL, 8>(k, lane); [[fallthrough]];
      case 8: cross_lane_sort_stage<NPL, 4>(k, lane); [[fallthrough]];
      case 4: cross_lane_sort_stage<NPL, 2>(k, lane); [[fallthrough]];
      case 2: cross_lane_sort_stage<NPL, 1>(k, lane); [[fallthrough]];
      default: local_sort_stages<NPL>(k, NPL); break;
    }
  }
}

// ---- a workgroup ranks the keys of a segment of up to 256: `keys` (LDS, 16-byte aligned) are its sort keys, and the place of the one
// that is `own` is the number of smaller ones.  Quadratic, a comparison and an addition with carry per pair, and yet the shorter chain where
// a workgroup waits for its order (a segment of 256 by one wave's network -> this, whole pass: 28 / 4 heads x 1000 55.8 -> 52.9 us, 32 / 8 x 4096
// 160.8 -> 159.4, 4 / 1 x 16384 164.8 -> 162.2; of 512, two keys a thread, 28 / 4 x 1100 60.8 -> 61.4); launches of nothing but
// sorts, which are bound by the instructions, keep the network.
__device__ __forceinline__ int rank_of(double own, const double* keys, int seg) {
  typedef __attribute__((ext_vector_type(2))) double f64x2;
  constexpr int AT_ONCE = 16;   // pairs of keys requested before the first is looked at
  int n = 0;
  for (int j = 0; j < seg; j += 2 * AT_ONCE) {   // a segment is a multiple of 64
    f64x2 k[AT_ONCE];
#pragma unroll
    for (int x = 0; x < AT_ONCE; ++x) k[x] = *reinterpret_cast<const f64x2*>(keys + j + 2 * x);
#pragma unroll
    for (int x = 0; x < AT_ONCE; x += 2) {
      uint64_t m0, m1, m2, m3;   // (a comparison's mask may be read two instructions later)
      asm("v_cmp_lt_f64_e64 %1, %5, %9\n\tv_cmp_lt_f64_e64 %2, %6, %9\n\tv_cmp_lt_f64_e64 %3, %7, %9\n\tv_cmp_lt_f64_e64 %4, %8, %9\n\t"
          "v_addc_co_u32_e64 %0, %1, %0, 0, %1\n\tv_addc_co_u32_e64 %0, %2, %0, 0, %2\n\tv_addc_co_u32_e64 %0, %3, %0, 0, %3\n\t"
          "v_addc_co_u32_e64 %0, %4, %0, 0, %4"
          : "+v"(n), "=&s"(m0), "=&s"(m1), "=&s"(m2), "=&s"(m3)
          : "v"(k[x].x), "v"(k[x].y), "v"(k[x + 1].x), "v"(k[x + 1].y), "v"(own));
    }
  }
  return n;
}

template <int NPL>
__device__ __forceinline__ double sort_key_of(const float* scores, int i, int seg) {
  const double none = __builtin_bit_cast(double, 0x3ff0000000000000ull | (uint64_t)0xffffffffu << 11 | (uint32_t)i);
  return i < seg ? sort_key(scores[i], (uint32_t)i) : none;
}

}  // namespace
