// Per-segment stable descending argsort of the key scores.
//
// A bitonic network over composite keys (inverted order-preserving score bits, then the local index), so
// equal scores keep ascending index order whatever the network does.  The
// trailing partial segment and the padding up to a whole block keep identity order.
// Segments of up to 2048 keys are sorted by one wave in registers, longer ones by a workgroup in LDS.
#include "pbs_lists.h"
#include "pbs_pool.h"
#include "pbs_sort.h"
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

// Sorts the wave's keys of segment `s` of a row (`seg` of them; register r of lane l starts with that of local index 64 r + l) and writes
// their order, as positions `base` and on, and, of segment 0, the block that holds key 0.
template <int NPL>
__device__ __forceinline__ void sort_and_store(double (&k)[NPL], int lane, int seg, int base, int s, int32_t* out, int32_t* first_blk, int block_size) {
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
  if (first_blk && s == 0 && zero_at >= 0) *first_blk = zero_at / block_size;
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

// The workgroups behind the first `sort_wgs` do the ride's pooling: the sort waits on its lanes and leaves the memory idle.
// Whole pass, pooling with the key blocks -> here, us: 32 / 8 heads x 20000 in segments of 2048 671 -> 654, 16 / 16 x 60000 875 -> 868, 28 / 4 x
// 13333 twice 778 -> 776.  (In the first pass of the split scoring, which leaves half of a CU free, it took more than it saved: 16 / 16 x
// 60000 854 -> 880, 32 / 8 x 2048 88.7 -> 91.1.)
template <int NPL>
__global__ __launch_bounds__(256) void segment_argsort_wave_kernel(const float* scores, int32_t* idx, int Sc, int S_pad, int seg, int n_units,
                                                                   int rows, int32_t* first_blk, int block_size, int64_t sort_wgs, PoolQ ride) {
  __shared__ float pool[16][POOL_D];
  const int lane = threadIdx.x & 63;
  const int64_t wg = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
  if (wg >= sort_wgs) {
    const int64_t blk = wg - sort_wgs;
    if (blk < (int64_t)rows * ride.nb) pool_q_block(pool, ride, (int)(blk % ride.nb), (int)(blk / ride.nb));
    return;
  }
  // a segment of a row, or a piece of its identity tail
  const int64_t unit = wg * 4 + (threadIdx.x >> 6);
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
  for (int r = 0; r < NPL; ++r) k[r] = sort_key_of<NPL>(src, 64 * r + lane, seg);   // (where a key starts does not matter: its index goes with it)
  sort_and_store<NPL>(k, lane, seg, base, s, out, first_blk ? first_blk + row : nullptr, block_size);
}

}  // namespace

bool pbs_segment_argsort_takes_ride(int segment_size) { return segment_size <= 2048; }

int pbs_segment_argsort_launch(const float* scores, int32_t* key_indices, int32_t* first_blk, int block_size, int rows, int S,
                               int S_pad, int segment_size, void* stream, const PoolQ& ride) {
  PBS_REQUIRE(!ride.nb || pbs_segment_argsort_takes_ride(segment_size), "pbs_segment_argsort: no pooling with segments of %d", segment_size);
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
    const int64_t sort_wgs = ((int64_t)rows * n_units + 3) / 4, wgs = sort_wgs + (int64_t)rows * ride.nb, gx = std::min<int64_t>(wgs, 1 << 23);
    const int64_t gy = (wgs + gx - 1) / gx;
    PBS_REQUIRE(gy <= 65535, "pbs_segment_argsort: launch too large");
    const dim3 grid((unsigned)gx, (unsigned)gy);
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, scores, key_indices, Sc, S_pad, segment_size, n_units, rows,
                         first_blk, block_size, sort_wgs, ride);
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
