// Per-segment stable descending argsort of the key scores.
//
// A bitonic network over composite keys (inverted order-preserving score bits, then the local index), so
// equal scores keep ascending index order whatever the network does.  The
// trailing partial segment and the padding up to a whole block keep identity order.
// Segments of up to 2048 keys are sorted by one wave in registers, longer ones by a workgroup in LDS.
#include "pbs_lists.h"
#include "pbs_wave.h"
#include "../../include/pbs_hip.h"   // the definitions below are checked against the public declarations
#include <algorithm>

namespace {

__global__ __launch_bounds__(256) void segment_argsort_kernel(const float* scores, int32_t* idx, int S, int Sc,
                                                              int S_pad, int seg, int n_pow2, int32_t* first_blk, int block_size) {
  extern __shared__ uint64_t keys[];
  const int row = blockIdx.y;
  const int nseg = Sc / seg;
  int32_t* out = idx + (int64_t)row * S_pad;
  if ((int)blockIdx.x >= nseg) {
    // identity tail: remainder of the sequence and the block padding
    for (int i = Sc + (blockIdx.x - nseg) * seg + threadIdx.x; i < min(S_pad, Sc + ((int)blockIdx.x - nseg + 1) * seg); i += blockDim.x)
      out[i] = i;
    return;
  }
  const int base = blockIdx.x * seg;
  const float* src = scores + (int64_t)row * Sc + base;
  for (int i = threadIdx.x; i < n_pow2; i += blockDim.x)
    keys[i] = i < seg ? desc_stable_key(src[i], (uint32_t)i) : ~0ull;
  bitonic_sort_lds(keys, n_pow2);
  for (int i = threadIdx.x; i < seg; i += blockDim.x) out[base + i] = base + (int32_t)(uint32_t)keys[i];
  if (first_blk && blockIdx.x == 0)
    for (int i = threadIdx.x; i < seg; i += blockDim.x)
      if ((uint32_t)keys[i] == 0) first_blk[row] = i / block_size;
}

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

template <int NPL>
__global__ __launch_bounds__(256) void segment_argsort_wave_kernel(const float* scores, int32_t* idx, int Sc, int S_pad, int seg, int n_units,
                                                                   int rows, int32_t* first_blk, int block_size) {
  const int lane = threadIdx.x & 63;
  // a segment of a row, or a piece of its identity tail
  const int64_t unit = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int row = (int)(unit / n_units), s = (int)(unit - (int64_t)row * n_units);
  if (row >= rows) return;
  const int base = s * seg;
  int32_t* out = idx + (int64_t)row * S_pad + base;
  if (base >= Sc) {
    for (int i = lane; i < min(seg, S_pad - base); i += 64) out[i] = base + i;
    return;
  }
  const float* src = scores + (int64_t)row * Sc + base;
  double k[NPL];
#pragma unroll
  for (int r = 0; r < NPL; ++r) {
    const int i = 64 * r + lane;   // (where a key starts does not matter: its index goes with it)
    const double none = __builtin_bit_cast(double, 0x3ff0000000000000ull | (uint64_t)0xffffffffu << 11 | (uint32_t)i);
    k[r] = i < seg ? sort_key(src[i], (uint32_t)i) : none;
  }
  wave_sort<NPL>(k, lane);
  const int at = lane * NPL;   // a segment is a multiple of the block size or not: the last lanes may hold padding
  int32_t o[NPL];
  int zero_at = -1;
#pragma unroll
  for (int r = 0; r < NPL; ++r) {
    const uint32_t i = sort_key_index(k[r]);
    zero_at = i == 0 ? at + r : zero_at;
    o[r] = base + (int32_t)i;
  }
  if (first_blk && s == 0 && zero_at >= 0) first_blk[row] = zero_at / block_size;
  if (NPL >= 4 && (seg & 3) == 0 && ((uintptr_t)out & 15) == 0) {
    typedef __attribute__((ext_vector_type(4))) int32_t i32x4;
#pragma unroll
    for (int r = 0; r < NPL; r += 4)
      if (at + r < seg) *reinterpret_cast<i32x4*>(out + at + r) = (i32x4){o[r], o[(r + 1) % NPL], o[(r + 2) % NPL], o[(r + 3) % NPL]};
  } else {
#pragma unroll
    for (int r = 0; r < NPL; ++r)
      if (at + r < seg) out[at + r] = o[r];
  }
}

}  // namespace

int pbs_segment_argsort_launch(const float* scores, int32_t* key_indices, int32_t* first_blk, int block_size, int rows, int S,
                               int S_pad, int segment_size, void* stream) {
  PBS_REQUIRE(key_indices, "pbs_segment_argsort: null index pointer");
  PBS_REQUIRE(rows > 0 && S > 0 && S_pad >= S, "pbs_segment_argsort: bad shape rows=%d S=%d S_pad=%d", rows, S, S_pad);
  PBS_REQUIRE(segment_size > 0 && segment_size <= 8192, "pbs_segment_argsort: segment_size %d outside (0, 8192]", segment_size);
  const int Sc = (S / segment_size) * segment_size;
  PBS_REQUIRE(Sc == 0 || scores, "pbs_segment_argsort: null score pointer");
  const int nseg = Sc / segment_size;
  const int tail_blocks = (S_pad - Sc + segment_size - 1) / segment_size;
  const int n_pow2 = next_pow2_int(segment_size);
  PBS_REQUIRE(rows <= 65535, "pbs_segment_argsort: too many rows (%d)", rows);
  if (segment_size <= 2048) {
    const int n_units = nseg + tail_blocks;
    // a launch holds fewer than 2^32 work-items along a dimension: rows of very many segments go on along y
    const int64_t wgs = ((int64_t)rows * n_units + 3) / 4, gx = std::min<int64_t>(wgs, 1 << 23);
    const int64_t gy = (wgs + gx - 1) / gx;
    PBS_REQUIRE(gy <= 65535, "pbs_segment_argsort: launch too large");
    const dim3 grid((unsigned)gx, (unsigned)gy);
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, scores, key_indices, Sc, S_pad, segment_size, n_units, rows,
                         first_blk, block_size);
    };
    if (segment_size <= 128) launch(segment_argsort_wave_kernel<2>);
    else if (segment_size <= 256) launch(segment_argsort_wave_kernel<4>);
    else if (segment_size <= 512) launch(segment_argsort_wave_kernel<8>);
    else if (segment_size <= 1024) launch(segment_argsort_wave_kernel<16>);
    else launch(segment_argsort_wave_kernel<32>);
    return pbs_check_launch("pbs_segment_argsort");
  }
  hipLaunchKernelGGL(segment_argsort_kernel, dim3(nseg + tail_blocks, rows), dim3(256), (size_t)n_pow2 * sizeof(uint64_t),
                     (hipStream_t)stream, scores, key_indices, S, Sc, S_pad, segment_size, n_pow2,
                     first_blk, block_size);
  return pbs_check_launch("pbs_segment_argsort");
}

extern "C" int pbs_segment_argsort(const float* scores, int32_t* key_indices, int rows, int S, int S_pad,
                                   int segment_size, void* stream) {
  return pbs_segment_argsort_launch(scores, key_indices, nullptr, 1, rows, S, S_pad, segment_size, stream);
}
