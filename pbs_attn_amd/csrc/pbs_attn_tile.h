// The tile pipeline of the PBS block-sparse attention kernel: LDS layout constants, the asynchronous global -> LDS
// tile copies, MFMA fragment reads and the software pipeline over one 128 x 128 tile (fast_tile).  Shared by the
// attention kernel and by the bench-only probe that times this pipeline by itself.
#pragma once
#include "pbs_lists.h"
#include <type_traits>
#include <utility>

// branch hints: they decide which side of a branch is laid out as the fall-through.  A taken branch refills the
// wave's instruction buffer, and in the tile loop all four waves of a workgroup take it at about the same time with
// the matrix pipes idle, so the common path of that loop has to be the straight one.
#define PBS_LIKELY(x) __builtin_expect(!!(x), 1)
#define PBS_UNLIKELY(x) __builtin_expect(!!(x), 0)

namespace {


constexpr int D = 128;
constexpr int BS = 128;
constexpr int TILE_BYTES = BS * D * 2;            // 32 KB
constexpr uint32_t LDS_V0 = 2 * TILE_BYTES;       // K buffers at 0 / 32 KB, V buffers at 64 / 96 KB
constexpr uint32_t LDS_LIST = 4 * TILE_BYTES;     // two merged visit lists (current item, next item), uint16 entries
constexpr uint32_t LIST_BYTES = 9728;             // header + at most 4096 + 511 + 1 entries, rounded up
constexpr uint32_t LDS_MISC = LDS_LIST + 2 * LIST_BYTES;   // ints: [1] redo flag, [4] next work item, [5] ranges with items left
constexpr uint32_t LDS_TOTAL = LDS_MISC + 1024;   // 151 552 bytes of the CU's 160 KB
constexpr int THREADS = 256;                      // four waves, one per SIMD
constexpr int QG = 4;                             // query column groups of 16 per wave: 64 queries

typedef __attribute__((address_space(3))) uint8_t lds_u8;

// lane id formed where it is asked for: as a plain intrinsic it is computed once at the top of the kernel and
// everything derived from it holds registers from there on
__device__ __forceinline__ int lane_id_here() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

// ---- operand geometry of a wave (64 queries = four column groups qg of 16: groups 0 and 1 are queries 32 w .. 32 w + 31
// of the pair's first query block, groups 2 and 3 those of its second; lane l: i = l % 16, g = l / 16)
//   S^T = K Q^T per 32-key sub-tile ks: two 16-key row tiles T, four d-steps kd of 32:
//       A = K[key(T, i)][32 kd + 8 g + 0..7],  key(T, i) = 32 ks + 8 (i / 4) + 4 T + i % 4
//       B = Q[16 qg + i][32 kd + 8 g + 0..7]
//       D: lane holds query 16 qg + i, keys 32 ks + 8 g + 4 T + 0..3
//     so the eight values of (T = 0, T = 1) are keys 32 ks + 8 g + 0..7: converted to bf16 they ARE the B operand of
//   O^T += V^T P^T per sub-tile: eight 16-row d tiles dt:
//       A = V^T[16 dt + i][32 ks + 8 g + 0..7],  B = P[keys 32 ks + 8 g + 0..7][16 qg + i]
//       D: lane holds query 16 qg + i, d = 16 dt + 4 g + 0..3
// LDS tiles are 128 rows x 16 chunks of 16 bytes, chunk index XOR hash(row): rows of a K tile are keys and the 16
// lanes of a fragment read take keys 8 (i / 4) + i % 4 (+ 4 T), so the hash is (row & 3) | ((row >> 3) & 3) << 2
// (= i: sixteen chunks, no bank conflict); rows of a V^T tile are d and the lanes take consecutive rows: row & 15.
__device__ __forceinline__ int k_row_hash(int row) { return (row & 3) | (((row >> 3) & 3) << 2); }

// A tile of V rows taken from the caller's tensor (a query block's own segment) is not transposed on the way in.  Its
// fragments are read with the transposing LDS read (ds_read_b64_tr_b16: lane l of a group of 16 hands in the address of
// four consecutive d of key (l / 4), and receives, for d = l, the four keys), two reads per fragment.  Four rows (keys
// 4 m + 0..3) share 1024 bytes of LDS, 32-byte piece p (d = 16 p .. 16 p + 15) of row 4 m + e at m * 1024 + p * 128 +
// e * 32: a group's four keys x 32 bytes are 128 consecutive bytes (no bank conflict), the d tile, the sub-tile and the
// key half of a read are constant offsets from one address per lane, and one copy instruction (1024 bytes of LDS)
// reads four whole rows.
// ---- asynchronous global -> LDS copy of a tile pair (K and V, 32 KB each) by four waves ----
// global_load_lds_dwordx4 writes lane l at M0 + offset + 16 l, so one instruction fills 1 KB = 4 consecutive LDS rows
// and the chunk swizzle is applied on the GLOBAL side.  Wave w copies rows 32 w .. 32 w + 31 of both tiles: pieces
// n = 0..7 of K, then of V, piece n being rows 32 w + 4 n + 0..3.  The immediate offset 1024 (n & 3) of a piece counts
// on both sides, so M0 changes every fourth piece only.  The sixteen source offsets are held per lane: with them the
// same sixteen instructions copy a permuted tile (32 KB contiguous), rows of the caller's tensor at their stride, or
// the last, partial block of a sequence, and only the two base addresses change from tile to tile.
// The pieces go out one by one between the matrix instructions of the current tile (fast_tile): issued together behind
// the tile's barrier they hold up a SIMD that has only one wave by 44 cycles each (5882 cycles per tile step against
// 5143 with a piece after every eighth matrix instruction).
// They are issued from inline assembly so that the compiler does not order later LDS reads of the OTHER buffer behind
// them; M0 is handed over as a register operand (the compiler writes it and knows it is in use; the s_nop is the wait
// state between that write and the copy); completion is awaited with s_waitcnt vmcnt(0) before the barrier that
// publishes the tile.
struct TileCopy {
  uint64_t k, v;               // source addresses less COPY_BIAS (wave-uniform)
  uint32_t lds;                // LDS byte offset of this wave's first piece of the destination K buffer
  uint32_t ko[8], vo[8];       // this lane's source offset of piece n of K / V, plus COPY_BIAS, less 1024 (n & 3)
};
constexpr uint32_t COPY_BIAS = 3072;   // keeps the offsets non-negative: the hardware adds them unsigned

template <int I>
__device__ __forceinline__ void copy_piece(const TileCopy& c) {
  constexpr int n = I & 7;
  const uint32_t voff = I < 8 ? c.ko[n] : c.vo[n];
  const uint64_t base = I < 8 ? c.k : c.v;
  register uint32_t m0v asm("m0") = c.lds + (I < 8 ? 0u : LDS_V0) + (n >> 2) * 4096;
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3" ::"s"(m0v), "v"(voff), "s"(base), "n"((n & 3) * 1024) : "memory");
}

__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
  // readfirstlane returns int: widen through uint32_t or the low half would be sign-extended
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32));
  return ((uint64_t)hi << 32) | (uint64_t)lo;
}

// source offsets for permuted tiles: lane l of piece n fetches chunk (l & 15) ^ hash(row) of row 32 w + 4 n + (l >> 4)
__device__ __forceinline__ void copy_offsets_perm(TileCopy& c, int wave, int lane) {
  const uint32_t r = (uint32_t)(lane >> 4), l16 = (uint32_t)(lane & 15);
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const uint32_t rows = COPY_BIAS + (uint32_t)wave * 8192u + (uint32_t)(n >> 2) * 4096u + r * 256u;
    c.ko[n] = rows + (l16 ^ (r | (uint32_t)(n >> 1) << 2)) * 16u;   // k_row_hash(32 w + 4 n + r)
    c.vo[n] = rows + (l16 ^ (4u * (uint32_t)(n & 3) + r)) * 16u;    // (32 w + 4 n + r) & 15
  }
}

// source offsets for a block of the caller's tensors (row strides in elements, < 2^22: offsets fit 32 bits).  K as above.
// V in the layout above: lane l takes row (l >> 1) & 3 of the piece and its 16-byte chunk 2 (l >> 3) + (l & 1).  Rows past
// the end of the sequence re-read the last valid row: their keys lie after every query and are masked.
__device__ __forceinline__ void copy_offsets_rows(TileCopy& c, uint32_t k_ss, uint32_t v_ss, int rows_valid, int wave, int lane) {
  const uint32_t r = (uint32_t)(lane >> 4), l16 = (uint32_t)(lane & 15);
  const int last = min(rows_valid, BS) - 1;
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const uint32_t bias = COPY_BIAS - 1024u * (uint32_t)(n & 3);
    const uint32_t krow = (uint32_t)min(32 * wave + 4 * n + (int)r, last);
    const uint32_t vrow = (uint32_t)min(32 * wave + 4 * n + ((lane >> 1) & 3), last);
    c.ko[n] = bias + krow * k_ss * 2u + (l16 ^ (r | (uint32_t)(n >> 1) << 2)) * 16u;
    c.vo[n] = bias + vrow * v_ss * 2u + (uint32_t)(2 * (lane >> 3) + (lane & 1)) * 16u;
  }
}

template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// all sixteen pieces at once: where no matrix instructions of this wave are there to hide them.  (The s_nop: an address that
// a vector instruction has just put into scalar registers, by readfirstlane, may be read by a memory instruction five wait
// states later, and the compiler does not look for that hazard inside inline assembly.)
__device__ __forceinline__ void copy_tile_now(const TileCopy& c) {
  asm volatile("s_nop 4");
  static_for<16>([&](auto ic) __attribute__((always_inline)) { copy_piece<decltype(ic)::value>(c); });
}

__device__ __forceinline__ bf16x8 ldsf(uint32_t byte_addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>((const lds_u8*)(uintptr_t)byte_addr);
}

// v_mfma_f32_16x16x32_bf16: D (16 x 16) += A (16 x 32) B (32 x 16).  Lane l holds row l % 16 of A and column l % 16 of
// B, each with k = 8 (l / 16) + 0..7, and of D column l % 16, rows 4 (l / 16) + 0..3.  On normally distributed
// operands the chip sustains about 11 % more FLOP/s with this shape than with 32x32x16 (it moves half the
// accumulator registers per FLOP and holds a higher clock inside its power limit).
// V^T fragment (16 d x 32 keys of a sub-tile) out of a tile of V rows: addr = this lane's address
// for the fragment's d tile and sub-tile; keys 8 g + 0..3 at addr, 8 g + 4..7 in the next four rows (1024 bytes further)
typedef __attribute__((ext_vector_type(4))) short s16x4;
__device__ __forceinline__ bf16x8 ldsf_transposed(uint32_t addr) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(lds_u8*)(uintptr_t)addr);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(lds_u8*)(uintptr_t)(addr + 1024));
  typedef __attribute__((ext_vector_type(8))) short s16x8;
  const s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(bf16x8, both);
}
// this lane's address of the fragment of sub-tile 0, d tile 0 in the tile whose buffer starts at LDS byte offset
// v_buf; d tile dt: + dt * 128, sub-tile ks: + ks * 8192
__device__ __forceinline__ uint32_t vrow_lane_addr(uint32_t v_buf, int lane) {
  const int l16 = lane & 15, g = lane >> 4;
  return v_buf + (uint32_t)(g * 2048 + (l16 >> 2) * 32 + (l16 & 3) * 8);
}

#define PBS_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0)

// the largest of three logits (a NaN only if all are), one instruction: the compiler puts one more per operand in front, to quieten
// signalling NaNs, of which matrix instructions have none
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// over the four lanes l, l ^ 16, l ^ 32, l ^ 48 that share a query column, by row exchanges of the vector unit (a shuffle
// goes through LDS)
template <class F>
__device__ __forceinline__ float fold_lane_groups(float v, F f) {
  const uint32_t u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const uint32_t w = __float_as_uint(f(__uint_as_float(a[0]), __uint_as_float(a[1])));
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float max_over_lane_groups(float v) {
  return fold_lane_groups(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float sum_over_lane_groups(float v) {
  return fold_lane_groups(v, [](float a, float b) { return a + b; });
}

// ---- accumulation registers.  The kernels that use this header keep O^T (a0 .. a127) and the wave's Q^T fragments
// (a128 .. a191; the next item's on their way in a192 .. a255) there by name; nothing of theirs is handed to the compiler, which has no use for accumulation
// registers of its own in these kernels (they need fewer than 256 vector registers;
// tests/test_attention_registers.py looks at the compiled code).  RESERVE_ACC_REGS makes them part of the kernels' register count.
constexpr int o_reg(int dt, int qg) { return (dt * QG + qg) * 4; }               // O^T: d tile dt, column group qg
constexpr int q_reg(int qg, int kd) { return 8 * QG * 4 + (qg * 4 + kd) * 4; }   // Q^T: column group qg, d-step kd
constexpr int Q_NEXT = 64;                                                        // the next item's Q^T: this much further on
#define PBS_ACC8(a, b) "a" #a #b "0", "a" #a #b "1", "a" #a #b "2", "a" #a #b "3", "a" #a #b "4", "a" #a #b "5", "a" #a #b "6", "a" #a #b "7", "a" #a #b "8", "a" #a #b "9"
#define RESERVE_ACC_REGS() asm volatile("" ::: "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", PBS_ACC8(, 1), PBS_ACC8(, 2), PBS_ACC8(, 3), \
  PBS_ACC8(, 4), PBS_ACC8(, 5), PBS_ACC8(, 6), PBS_ACC8(, 7), PBS_ACC8(, 8), PBS_ACC8(, 9), PBS_ACC8(1, 0), PBS_ACC8(1, 1), PBS_ACC8(1, 2), PBS_ACC8(1, 3), \
  PBS_ACC8(1, 4), PBS_ACC8(1, 5), PBS_ACC8(1, 6), PBS_ACC8(1, 7), PBS_ACC8(1, 8), PBS_ACC8(1, 9), PBS_ACC8(2, 0), PBS_ACC8(2, 1), PBS_ACC8(2, 2), PBS_ACC8(2, 3), PBS_ACC8(2, 4), \
  "a250", "a251", "a252", "a253", "a254", "a255")
// wait states between a matrix instruction and other accesses to its registers, either way round
#define MFMA_FENCE()                                     \
  do {                                                   \
    __builtin_amdgcn_sched_barrier(0);                   \
    asm volatile("s_nop 15" ::: "memory");               \
    __builtin_amdgcn_sched_barrier(0);                   \
  } while (0)

__device__ __forceinline__ void o_clear() {
  static_for<8 * QG * 4>([](auto ic) __attribute__((always_inline)) {
    asm volatile("v_accvgpr_write_b32 a[%0], 0" ::"n"(decltype(ic)::value));
  });
}
template <int DT, int Q>
__device__ __forceinline__ f32x4 o_get() {
  constexpr int r = o_reg(DT, Q);
  float x0, x1, x2, x3;
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x0) : "n"(r));
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x1) : "n"(r + 1));
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x2) : "n"(r + 2));
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x3) : "n"(r + 3));
  return (f32x4){x0, x1, x2, x3};
}
// the rows of column group Q times `alpha` (fences are the caller's)
template <int Q>
__device__ __forceinline__ void o_scale(float alpha) {
  static_for<8 * 4>([&](auto ic) __attribute__((always_inline)) {
    constexpr int r = o_reg(decltype(ic)::value >> 2, Q) + (decltype(ic)::value & 3);
    float x;
    asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(r));
    x *= alpha;
    asm volatile("v_accvgpr_write_b32 a[%1], %0" ::"v"(x), "n"(r));
  });
}
// this lane's 16 bytes of a Q^T fragment, straight into the accumulation registers.  They are there only once a vmcnt wait
// has covered the load, and nobody waits by himself: neither the compiler nor the hardware.
template <int Q, int KD, int SET = 0>
__device__ __forceinline__ void q_load(const uint16_t* src) {
  constexpr int r = q_reg(Q, KD) + SET;
  asm volatile("global_load_dwordx4 a[%1:%2], %0, off" ::"v"(src), "n"(r), "n"(r + 3) : "memory");
}
// the Q^T fragments that q_load<.., Q_NEXT> brought in become the current ones
__device__ __forceinline__ void q_advance() {
  static_for<QG * 16>([](auto ic) __attribute__((always_inline)) {
    constexpr int r = q_reg(0, 0) + decltype(ic)::value;
    asm volatile("v_accvgpr_mov_b32 a[%0], a[%1]" ::"n"(r), "n"(r + Q_NEXT));
  });
}
// S^T (+)= K fragment x Q^T;  O^T += V^T fragment x P^T
template <int Q, int KD, bool FROM_ZERO>
__device__ __forceinline__ void mfma_s(f32x4& d, const bf16x8& k) {
  constexpr int r = q_reg(Q, KD);
  if constexpr (FROM_ZERO) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, a[%2:%3], 0" : "=v"(d) : "v"(k), "n"(r), "n"(r + 3));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, a[%2:%3], %0" : "+v"(d) : "v"(k), "n"(r), "n"(r + 3));
}
// the same with the sums in vector registers
template <bool FROM_ZERO>
__device__ __forceinline__ void mfma_v(f32x4& d, const bf16x8& v, const bf16x8& p) {
  if constexpr (FROM_ZERO) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=v"(d) : "v"(v), "v"(p));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(v), "v"(p));
}
template <int DT, int Q>
__device__ __forceinline__ void o_set(const f32x4& x) {
  constexpr int r = o_reg(DT, Q);
  asm volatile("v_accvgpr_write_b32 a[%1], %0" ::"v"(x[0]), "n"(r));
  asm volatile("v_accvgpr_write_b32 a[%1], %0" ::"v"(x[1]), "n"(r + 1));
  asm volatile("v_accvgpr_write_b32 a[%1], %0" ::"v"(x[2]), "n"(r + 2));
  asm volatile("v_accvgpr_write_b32 a[%1], %0" ::"v"(x[3]), "n"(r + 3));
}
template <int DT, int Q>
__device__ __forceinline__ void mfma_o(const bf16x8& v, const bf16x8& p) {
  constexpr int r = o_reg(DT, Q);
  asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(v), "v"(p), "n"(r), "n"(r + 3));
}

// ---- fast tile: one 128-key tile for the wave's 64 queries, a static schedule of 272 matrix instructions ----
// The four 32-key sub-tiles k run as a software pipeline: S of sub-tile k + 1 and k + 2, the exponentials of k and P.V
// of k - 1 at the same time.  A SIMD holds ONE wave (64 queries need 128 accumulator registers for O, 64 for Q^T, 64 for
// two sub-tiles of S), which issues in order, so nothing but the order of the instructions keeps the matrix pipe fed:
// a matrix instruction occupies the pipe for 16 cycles and the issue of its wave for 8, which leaves 8 cycles per
// instruction ("gap") for vector work -- two multiply-adds, or one exponential, or two conversions.  The schedule gives
// every gap one such unit: 32 combos (sub-tile, row tile T, column group) of 7 units = 224 of the 272 gaps; scheduling
// barriers keep the compiler from moving anything.  An LDS read goes out right behind a matrix instruction, before the
// gap's vector work (behind the vector work it costs 8 cycles more), and so does the wait for a fragment (in front of
// its matrix instruction it costs 4).
// Why 64 queries per wave: half the LDS fragment reads per FLOP of 32 queries per wave and two waves per SIMD (the form
// this replaces: 5543 cycles and 3.03 us per tile step on normally distributed values, inside the chip's power limit).
// Same box, same call: 5143 cycles, 2.79 us, 1421 -> 1538 TFLOP/s; with matrix instructions and vector work in
// alternating runs of eight instead of one by one it was 8400 cycles.
//
// Matrix instructions are inline assembly, with O and Q^T in accumulation registers named here (below) and S and P in
// vector registers: left to the compiler, S goes through accumulation registers (one extra vector instruction per
// logit), and O, live across four tile loops and the rare paths between them, is copied and spilled at every seam.  The
// compiler knows the wait states around its own matrix instructions only, so the distances inside the schedule are
// checked at compile time (check_schedule), and MFMA_FENCE stands wherever other code meets these registers.
struct MfmaOp { int kind, k, T, x, q, frag; };   // kind 0: S (sub-tile k, row tile T, d-step x); 1: P.V (k, d tile x); 2: row sums (k)
constexpr int N_FRAG = 64, UNITS_PER_COMBO = 7;
constexpr int FRAG_BUFS = 6, FRAG_AHEAD = 11;   // fragment registers; how many matrix instructions ahead of its use a fragment is read
constexpr int COPY_FIRST_GAP = 2;
// A piece of the next tile's copy every so many matrix instructions: all of them are on their way before the middle of a tile, which leaves its second
// half to the memory's latency.  In a tile of two column groups pieces 8 apart end with the tile, and its wait was a round trip to L2: passes of single
// blocks, 8 apart -> 4, 4 / 1 heads x 8192 96.3 -> 92.0 us, 129.1 -> 124.3 in segments of 128, 8 / 2 x 2048 60.5 -> 59.2, 28 / 4 x 1000 53.5 -> 52.7;
// 3 apart 93.7, 127.7, 59.7 and 52.8, 2 apart no better than 8; rows of few selected blocks, 8 / 2 x 142981 in segments of 2048 2193 -> 2112.
// The second block's diagonal tile, a pair's last, keeps 8: its copies, the next item's first tile, follow that item's sixteen query loads and hold up
// what is behind them.  4 apart there -> 8: inside one segment 4 x 16 / 16 x 1152 41.0 -> 40.0 us, 2 x 32 / 8 x 1152 40.4 -> 39.5; 28 / 4 x 1000 in segments of 256 52.3 -> 51.8,
// 32 / 8 x 32768 concentrated 826.5 -> 822.5, x 131072 2668 -> 2643.
constexpr int copy_gap_step(int nq, bool ends_pair) { return nq == 2 && !ends_pair ? 4 : 8; }
// NQ: the column groups the tile is worked on for, four or (a tile that only one of the pair's blocks sees) two
template <int NQ>
struct TileSchedule {
  static constexpr int N_MFMA = 68 * NQ, N_UNITS = 8 * NQ * UNITS_PER_COMBO;
  static constexpr int FIRST_UNIT_GAP = 3 * NQ + 3;   // the exponentials start when the first row tile of S is complete
  MfmaOp op[N_MFMA];
  int first_use[N_FRAG], last_use[N_FRAG];     // matrix instructions that use fragment f (NQ each)
  int read_after[N_FRAG];                      // f is read behind this matrix instruction (-1: before the first)
  int frag_kind[N_FRAG], frag_k[N_FRAG], frag_T[N_FRAG], frag_x[N_FRAG];
  static constexpr int unit_gap(int combo, int unit) { return FIRST_UNIT_GAP + UNITS_PER_COMBO * combo + unit; }
};
template <int NQ>
constexpr TileSchedule<NQ> make_schedule() {
  TileSchedule<NQ> s{};
  int n = 0, nf = 0;
  auto frag = [&](int kind, int k, int T, int x) {
    s.frag_kind[nf] = kind; s.frag_k[nf] = k; s.frag_T[nf] = T; s.frag_x[nf] = x;
    return nf++;
  };
  auto S = [&](int k, int T, int kd) {
    const int f = frag(0, k, T, kd);
    for (int q = 0; q < NQ; ++q) s.op[n++] = MfmaOp{0, k, T, kd, q, f};
  };
  auto P = [&](int k, int dt) {
    const int f = frag(1, k, 0, dt);
    for (int q = 0; q < NQ; ++q) s.op[n++] = MfmaOp{1, k, 0, dt, q, f};
  };
  auto L = [&](int k) {
    for (int q = 0; q < NQ; ++q) s.op[n++] = MfmaOp{2, k, 0, 0, q, -1};
  };
  for (int k = 0; k < 2; ++k)
    for (int T = 0; T < 2; ++T)
      for (int kd = 0; kd < 4; ++kd) S(k, T, kd);
  for (int kd = 0; kd < 4; ++kd) S(2, 0, kd);
  for (int kd = 0; kd < 4; ++kd) { S(2, 1, kd); P(0, 2 * kd); P(0, 2 * kd + 1); }
  L(0);
  for (int kd = 0; kd < 4; ++kd) { S(3, 0, kd); P(1, 2 * kd); P(1, 2 * kd + 1); }
  L(1);
  // the last row tile of S early: its exponentials come last
  if (NQ == 4) {
    for (int kd = 0; kd < 4; ++kd) { S(3, 1, kd); P(2, kd); }
    for (int dt = 4; dt < 8; ++dt) P(2, dt);
  } else {
    for (int kd = 0; kd < 4; ++kd) S(3, 1, kd);
    for (int dt = 0; dt < 8; ++dt) P(2, dt);
  }
  L(2);
  // the first d tiles of the last P.V take the last column group late: its probabilities are the last to be ready
  constexpr int HEAD = NQ == 4 ? 2 : 5;
  int head[HEAD] = {};
  for (int dt = 0; dt < HEAD; ++dt) {
    head[dt] = frag(1, 3, 0, dt);
    for (int q = 0; q < NQ - 1; ++q) s.op[n++] = MfmaOp{1, 3, 0, dt, q, head[dt]};
  }
  for (int dt = 0; dt < HEAD; ++dt) s.op[n++] = MfmaOp{1, 3, 0, dt, NQ - 1, head[dt]};
  for (int dt = HEAD; dt < 6; ++dt) P(3, dt);
  L(3);
  P(3, 6);
  P(3, 7);
  for (int f = 0; f < N_FRAG; ++f) s.first_use[f] = -1;
  for (int i = 0; i < s.N_MFMA; ++i) {
    const int f = s.op[i].frag;
    if (f < 0) continue;
    if (s.first_use[f] < 0) s.first_use[f] = i;
    s.last_use[f] = i;
  }
  int prev = -1;
  for (int f = 0; f < N_FRAG; ++f) {   // FRAG_AHEAD before the first use, not before the register is free, one read per gap
    int r = s.first_use[f] - FRAG_AHEAD;
    if (f >= FRAG_BUFS && r < s.last_use[f - FRAG_BUFS]) r = s.last_use[f - FRAG_BUFS];
    if (r < 0) { s.read_after[f] = -1; continue; }
    if (r <= prev) r = prev + 1;
    s.read_after[f] = prev = r;
  }
  return s;
}
template <int NQ>
constexpr TileSchedule<NQ> SCHED = make_schedule<NQ>();
// 0, or the number of the rule that the schedule breaks
template <int NQ>
constexpr int check_schedule() {
  constexpr TileSchedule<NQ> s = SCHED<NQ>;
  int last_s[4][2][NQ] = {}, first_s[4][2][NQ] = {}, last_p[4][NQ] = {}, first_p[4][NQ] = {}, n_s = 0, n_p = 0, n_l = 0;
  for (int k = 0; k < 4; ++k)
    for (int q = 0; q < NQ; ++q) {
      first_p[k][q] = s.N_MFMA;
      first_s[k][0][q] = first_s[k][1][q] = s.N_MFMA;
    }
  for (int i = 0; i < s.N_MFMA; ++i) {
    const MfmaOp m = s.op[i];
    int& first = m.kind == 0 ? first_s[m.k][m.T][m.q] : first_p[m.k][m.q];
    int& last = m.kind == 0 ? last_s[m.k][m.T][m.q] : last_p[m.k][m.q];
    if (i < first) first = i;
    last = i;
    ++(m.kind == 0 ? n_s : m.kind == 1 ? n_p : n_l);
  }
  if (n_s != 32 * NQ || n_p != 32 * NQ || n_l != 4 * NQ) return 8;
  for (int k = 0; k < 4; ++k)
    for (int T = 0; T < 2; ++T)
      for (int q = 0; q < NQ; ++q) {
        const int c = NQ * (2 * k + T) + q;
        if (s.unit_gap(c, 0) < last_s[k][T][q] + 3) return 1;                          // logits complete before they are read (32 cycles)
        if (first_p[k][q] < s.unit_gap(c, 6) + 3) return 2;                            // probabilities written before they are read
        if (k >= 2 && first_s[k][T][q] <= s.unit_gap(c - 4 * NQ, 2)) return 3;         // logits read before they are overwritten
        if (k >= 2 && s.unit_gap(c, 6) < last_p[k - 2][q]) return 4;                   // probabilities too
      }
  for (int f = 0; f < N_FRAG; ++f) {
    if (s.read_after[f] >= 0 && s.first_use[f] < s.read_after[f] + 6) return 5;
    if (f >= FRAG_BUFS && s.read_after[f] < s.last_use[f - FRAG_BUFS]) return 6;
  }
  if (s.unit_gap(8 * NQ - 1, 6) >= s.N_MFMA || COPY_FIRST_GAP + 15 * copy_gap_step(NQ, true) >= s.N_MFMA) return 7;
  return 0;
}
static_assert(check_schedule<4>() == 0 && check_schedule<2>() == 0, "tile schedule");
template <int NQ>
constexpr int frag_read_after(int i) {
  for (int f = 0; f < N_FRAG; ++f)
    if (SCHED<NQ>.read_after[f] == i) return f;
  return -1;
}
template <int NQ>
constexpr int frag_first_used_at(int i) {
  for (int f = 0; f < N_FRAG; ++f)
    if (SCHED<NQ>.first_use[f] == i) return f;
  return -1;
}
// LDS read instructions that go out after fragment f's and not later than behind matrix instruction i
template <int NQ>
constexpr int lds_reads_younger(int f, int i, bool v_rows) {
  int c = 0;
  for (int g = f + 1; g < N_FRAG; ++g)
    if (SCHED<NQ>.read_after[g] <= i) c += (v_rows && SCHED<NQ>.frag_kind[g] == 1) ? 2 : 1;
  return c < 15 ? c : 15;
}
// ka[kd] / va[ks]: this lane's byte addresses of the K fragments of d-step kd (row tile 0, sub-tile 0) and of the V^T
// fragments of sub-tile ks (d tile 0) in the tile's buffers: held in registers and switched between the two buffers
// once per tile, so that a fragment read needs no address arithmetic.
// Q0, NQ: the column groups that see the tile: all four, or the two of one of the pair's blocks.  (A block that does not visit
// a tile takes no part in it at all: with probabilities of zero instead, an infinity or a NaN of the tile's V would get
// into its rows.)  MASKED: the column groups
// (bits) whose diagonal block the tile is, read in original key order: logits of keys that lie after the query
// (key-in-tile > query-in-block) get no probability.  V_ROWS: the tile's V is a tile of the caller's tensor, and its fragments
// come from transposing reads; otherwise it is a transposed (V^T) tile and they are plain 16-byte reads.
// Exponentials are taken against a LAZY reference maximum (see pbs_attn.hip).  Row sums
// come from one more matrix instruction per sub-tile and column group, ones x P, whose every output row is the sum over
// the sub-tile's 32 keys of the probabilities as the P.V product sees them (rounded to bf16).
// `copy`: the next tile's copies, a piece every copy_gap_step matrix instructions.
template <int Q0, int NQ, int MASKED, bool V_ROWS, bool COPIES = true>
__device__ __forceinline__ void fast_tile(const uint32_t (&ka)[4], const uint32_t (&va)[4], float c_log2, float (&m_ref)[QG],
                                          float (&l_row)[QG], bool& poisoned, int wave, const TileCopy& copy) {
  typedef TileSchedule<NQ> Sched;
  float negm[QG];
#pragma unroll
  for (int q = Q0; q < Q0 + NQ; ++q) negm[q] = -m_ref[q];
  // The diagonal tile, by sub-tile k of 32 keys against the wave's 32 queries of the block: k < wave visible, k > wave
  // hidden, k == wave the triangle key 8 g + 4 T + r > query 16 (q % 2) + i.  The probabilities of masked column groups,
  // as bf16 pairs, are ANDed with all ones, zero or the triangle's bits (one register per pair, the same for both blocks),
  // whatever they are: a later key's logit may be NaN or infinite without a trace.  2 vector instructions per pair of logits
  // (comparing and selecting per logit takes 4, and held up the diagonal tile by 1300 cycles).
  uint32_t tri[2][2][2];          // [T][q % 2][pair]
  uint32_t some[MASKED ? 4 : 1], all[MASKED ? 4 : 1];   // all ones where k <= wave, where k < wave
  if (MASKED) {
    const int ln = lane_id_here();          // nothing below may be formed outside the tile
    const int qrel8 = (ln & 15) - 8 * (ln >> 4);
#pragma unroll
    for (int T = 0; T < 2; ++T)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
          const int key = 4 * T + 2 * pr - 16 * q;
          tri[T][q][pr] = (key <= qrel8 ? 0xffffu : 0u) | (key + 1 <= qrel8 ? 0xffff0000u : 0u);
          asm volatile("" : "+v"(tri[T][q][pr]));   // (formed here, not in the gaps)
        }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      some[k] = k <= wave ? ~0u : 0u;
      all[k] = k < wave ? ~0u : 0u;
      asm volatile("" : "+v"(some[k]), "+v"(all[k]));
    }
  }
  uint32_t vr = 0;
  if (V_ROWS) vr = vrow_lane_addr(LDS_V0 + (va[0] & 0x8000u), lane_id_here());   // va[] carries the buffer switch in bit 15
  u32x4 one_bits = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
  asm volatile("" : "+v"(one_bits));
  const bf16x8 ones = __builtin_bit_cast(bf16x8, one_bits);
  f32x4 sacc[2][2][NQ];    // [sub-tile parity][T][q], column group Q0 + q
  u32x4 pbuf[2][NQ];       // [sub-tile parity][q]: eight probabilities, bf16
  f32x4 lsum[NQ];
  bf16x8 fr[FRAG_BUFS];
  float x[4], e[4];        // the combo in work
  auto read_frag = [&](auto fc) __attribute__((always_inline)) {
    constexpr int f = decltype(fc)::value;
    if constexpr (f >= 0) {
      constexpr int k = SCHED<NQ>.frag_k[f], T = SCHED<NQ>.frag_T[f], fx = SCHED<NQ>.frag_x[f];
      if constexpr (SCHED<NQ>.frag_kind[f] == 0) fr[f % FRAG_BUFS] = ldsf(ka[fx] + T * 1024 + k * 8192);
      else if constexpr (V_ROWS) fr[f % FRAG_BUFS] = ldsf_transposed(vr + fx * 128 + k * 8192);
      else fr[f % FRAG_BUFS] = ldsf(va[k] + fx * 4096);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  static_for<FRAG_BUFS>([&](auto fc) __attribute__((always_inline)) {
    constexpr int f = decltype(fc)::value;
    read_frag(std::integral_constant<int, SCHED<NQ>.read_after[f] < 0 ? f : -1>{});
  });
  static_for<Sched::N_MFMA>([&](auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;
    constexpr MfmaOp m = SCHED<NQ>.op[i];
    if constexpr (m.kind == 0) {
      f32x4& d = sacc[m.k & 1][m.T][m.q];
      mfma_s<Q0 + m.q, m.x, m.x == 0>(d, fr[m.frag % FRAG_BUFS]);
    } else if constexpr (m.kind == 1) {
      mfma_o<m.x, Q0 + m.q>(fr[m.frag % FRAG_BUFS], __builtin_bit_cast(bf16x8, pbuf[m.k & 1][m.q]));
    } else {
      f32x4& d = lsum[m.q];
      const bf16x8 fa = ones, fb = __builtin_bit_cast(bf16x8, pbuf[m.k & 1][m.q]);
      if constexpr (m.k == 0) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=v"(d) : "v"(fa), "v"(fb));
      else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(fa), "v"(fb));
    }
    __builtin_amdgcn_sched_barrier(0);
    // the next matrix instruction's fragment has landed; then this gap's read, copy piece and vector unit
    constexpr int f_next = frag_first_used_at<NQ>(i + 1);
    if constexpr (f_next >= 0) {
      __builtin_amdgcn_s_waitcnt(0xC07F | lds_reads_younger<NQ>(f_next, i - 1, V_ROWS) << 8);   // lgkmcnt only
      __builtin_amdgcn_sched_barrier(0);
    }
    read_frag(std::integral_constant<int, frag_read_after<NQ>(i)>{});
    constexpr int past = i - COPY_FIRST_GAP, step = copy_gap_step(NQ, MASKED == 12);
    if constexpr (COPIES && past >= 0 && past % step == 0 && past / step < 16) {
      copy_piece<past / step>(copy);
      __builtin_amdgcn_sched_barrier(0);
    }
    constexpr int u = i - Sched::FIRST_UNIT_GAP;
    if constexpr (u >= 0 && u < Sched::N_UNITS) {
      constexpr int combo = u / UNITS_PER_COMBO, unit = u % UNITS_PER_COMBO, k = combo / (2 * NQ), T = combo / NQ & 1, q = combo % NQ;
      auto scaled = [&](auto rc) __attribute__((always_inline)) {
        constexpr int r = decltype(rc)::value;
        x[r] = __builtin_fmaf(sacc[k & 1][T][q][r], c_log2, negm[Q0 + q]);
      };
      if constexpr (unit == 0) { scaled(std::integral_constant<int, 0>{}); scaled(std::integral_constant<int, 1>{}); }
      if constexpr (unit == 1) e[0] = __builtin_amdgcn_exp2f(x[0]);
      if constexpr (unit == 2) { scaled(std::integral_constant<int, 2>{}); scaled(std::integral_constant<int, 3>{}); }
      if constexpr (unit >= 3 && unit <= 5) e[unit - 2] = __builtin_amdgcn_exp2f(x[unit - 2]);
      if constexpr (unit == 6) {
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
          uint32_t two = __builtin_bit_cast(uint32_t, (bf16x2){(__bf16)e[2 * pr], (__bf16)e[2 * pr + 1]});
          if constexpr (MASKED >> (Q0 + q) & 1) two &= (tri[T][q & 1][pr] & some[k]) | all[k];
          pbuf[k & 1][q][2 * T + pr] = two;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  });
  // row sums of this tile, the same in the four lanes of a query
  bool any_big = false;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    l_row[Q0 + q] += lsum[q][0];
    any_big |= lsum[q][0] > 16384.0f;
  }
  // lazy reference maximum without tracking maxima: a row sum of this tile above 2^14 says some
  // exponential was large; any reference >= the old one is valid, so move it up by log2(sum)
  if (PBS_UNLIKELY(__any(any_big))) {
    MFMA_FENCE();
    static_for<NQ>([&](auto qc) __attribute__((always_inline)) {
      constexpr int q = Q0 + decltype(qc)::value;
      const float big = lsum[q - Q0][0];
      if (__any(!(big < 1e30f))) poisoned = true;   // overflow (inf / nan): redo the row without speculation
      const float m_new = (big > 16384.0f) ? m_ref[q] + __builtin_amdgcn_logf(big) : m_ref[q];
      const float alpha = (big > 16384.0f) ? __builtin_amdgcn_exp2f(m_ref[q] - m_new) : 1.0f;   // (m_ref may be -inf: a block that has seen no tile)
      m_ref[q] = m_new;
      l_row[q] *= alpha;
      o_scale<q>(alpha);
    });
    MFMA_FENCE();
  }
}

}  // namespace
