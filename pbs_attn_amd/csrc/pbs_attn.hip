// Block-sparse flash-attention forward of PBS-Attn (bf16, head_dim 128).
//
// What a query block attends to
//   * the permuted K / V tiles of the selected key blocks of EARLIER segments (the visit list), no mask;
//   * its own segment, read from the ORIGINAL K and V (the caller's tensors, in place): blocks
//     first-of-segment .. query block, with the plain causal triangle on the last one (the diagonal block).
//     A segment's permuted blocks hold the same keys as its original blocks and attention does not depend
//     on key order, so this is the reference's "every block of the own segment, element mask original key
//     position > query position" with half the tiles and one masked tile instead of all.
// Work decomposition
//   A work item is two adjacent 128-query blocks of one head, or in a short pass one (item_span), served by one workgroup
//   (4 waves, one per SIMD): wave w takes queries 32 w .. 32 w + 31 of either block, so that the waves finish a tile together
//   also where only one block visits it, as the last tile of a pair, the second block's diagonal one; such a tile takes half a
//   tile's time.  A pair's two visit lists come merged into one list in HBM (ascending key-block indices, own-segment blocks appended),
//   written by the block selection, by the list kernel below from CSR rows, or, for a sequence inside one segment, formed in
//   LDS by the workgroup itself; every merged tile is copied ONCE into LDS for both query blocks of a pair, which
//   halves the L2 -> LDS traffic and doubles the time a tile stays in flight.  K and V tiles are
//   double-buffered (2 x 64 KB) and fetched one tile ahead with asynchronous global -> LDS copies (no
//   registers), one workgroup barrier per tile.
//   The attention kernel is PERSISTENT: one workgroup per CU takes item after item from a counter (one per
//   XCD, over that XCD's share of the items; when it runs dry, the other XCDs' counters), the first one without asking.  The tile pipeline
//   runs across items: the next item is claimed three tiles before the end of the current one, its list is
//   requested one tile later, its queries and its first K / V tiles at the last tile, so that an
//   item's fixed costs (list, first tile, write-out of the previous item) overlap attention work.  With short
//   visit lists (a few tiles per item) that is the difference between waiting for HBM three times per item
//   and once.
// Data layout
//   K tile: 128 keys x 128 d row-major; permuted V tile: stored TRANSPOSED in HBM by the gather kernel,
//   128 d x 128 keys; V tile of an own segment: 128 keys x 128 d as in the caller's tensor, its MFMA fragments
//   read with the transposing LDS read.  K and V^T tiles sit in LDS as 128 rows x 16 chunks of 16 bytes with the
//   chunk index XORed with a hash of the row (pbs_attn_tile.h), so that fragment reads are bank-conflict free.
// Math (transposed formulation, v_mfma_f32_16x16x32_bf16)
//     S^T = K Q^T   (rows = keys, columns = queries)      O^T += V^T P^T   (rows = d, columns = queries)
//   Every lane owns query columns (one per column group of 16 queries), so the softmax reference values are
//   per-lane, and the S^T accumulator registers are, after conversion to bf16, exactly the B operand of the
//   second product (the key rows of each 16-row MFMA tile are fed in the order that makes this so).
//   Softmax runs in the exp2 domain in fp32; P is rounded to bf16 before P.V, and a pipelined tile takes its row
//   sums from one more matrix product, ones x P, i.e. of the rounded values; the output is normalised once at
//   the end.
// Tile kinds
//   * fast tiles: a software pipeline over the four 32-key sub-tiles in a static schedule (pbs_attn_tile.h): one
//     matrix instruction, one unit of exponential work, and so on; the next tile's copies go out in between.
//     Exponentials are taken against a LAZY reference maximum: it is not updated per tile; a row
//     sum of one tile above 2^14 triggers a uniform rescale (exact, all terms share the reference); an
//     overflow marks the row and the whole workgroup redoes it without speculation.  The first tile of a
//     row takes its reference from the exact maximum over its first 32 keys.  The diagonal tile runs the
//     same pipeline and zeroes the probabilities of keys after the query (key-in-tile > query-in-block).
//   * careful tiles (the redo pass): one 32-key sub-tile at a time, exact running maximum, classic online softmax; so, in vector
//     registers, a diagonal tile that is its block's first tile.
//   An item's tiles come in the order permuted tiles, own-segment tiles before the diagonal, diagonal tile, and
//   each kind has a loop of its own (see the loops).
#include "pbs_attn_tile.h"
#include "pbs_attn_block.h"
#include "pbs_wave.h"
#include "../../include/pbs_hip.h"   // the definitions below are checked against the public declarations
#include <atomic>
#include <type_traits>

namespace {

struct AttnArgs {
  const uint16_t* q;
  const uint16_t* pk;    // (B*Hq, nb*128, 128)  permuted K
  const uint16_t* pvt;   // (B*Hq, nb, 128, 128) permuted V blocks, transposed
  const uint16_t* k;     // original K at the KV heads, caller's strides
  const uint16_t* v;     // original V at the KV heads, caller's strides
  const uint16_t* plist; // (B*Hq * n_items, cap) merged visit lists, in item order
  int* queue;            // 8 work counters, one per XCD
  int cap;               // entries per list row (multiple of 8); 0: no lists in memory (see own_list)
  int one_each;          // every item is some workgroup's first: nobody asks for a further one
  uint16_t* o;
  int BH, Hq, Hkv, S, nb, bps;
  int span;           // query blocks of an item (two, or one: see item_span)
  uint32_t k_ss, v_ss;   // key / value row strides in elements (< 2^22)
  int xcd_start[9];   // work items (head-major, long rows first) of XCD x: [xcd_start[x], xcd_start[x + 1])
  struct Deal {
    int how;     // how tickets become items (see ticket_item)
    int n;       // items of a head
    int heads;   // heads dealt together
    uint32_t group_magic, heads_magic;   // quotients by heads * n and by heads: high word of a product
  } deal;
  int64_t q_sb, q_sh, q_ss, k_sb, k_sh, v_sb, v_sh, o_sb, o_sh, o_ss;
  float scale_log2;
};

typedef const __attribute__((address_space(4))) struct AttnArgs* ArgsPtr;

// ---- merged visit list of an item (a pair of query blocks, or one), built once per pass by its own kernel.  Row `item` of `plist` (items
// are numbered head by head, the long ones of a head first) starts with a header that saves the attention kernel its
// divisions -- [0] number of tiles, [1] batch, [2] query head, [3] KV head, [4] first query block, [5] how many -- and holds from
// LIST_HEADER on entries kb | ENT_ORIG? | use_first << 14 |
// use_second << 15: the union of the two visit lists (ascending), then the own segments in ORIGINAL key order
// (blocks first-of-segment .. query block, shared where the two blocks share a segment).  Without `cols` every block of
// every earlier segment is visited.  Block 0 also sets the work counters of the attention kernel that follows on the
// stream: its workgroups start on the first `first_tickets` tickets of their ranges without asking.
constexpr int MERGE_THREADS = 256;
__global__ __launch_bounds__(MERGE_THREADS) void merge_pair_lists_kernel(const int32_t* __restrict__ cols, const int32_t* __restrict__ cnt,
                                                               uint16_t* __restrict__ plist, int* __restrict__ queue, int nb,
                                                               int span, int bps, int cap, int Hq, int group, int first_tickets,
                                                               const uint8_t* __restrict__ own_needed) {
  __shared__ uint8_t flags0[4096], flags1[4096];
  __shared__ int wsum[MERGE_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n_items = (nb + span - 1) / span;
  const int bh = blockIdx.x / n_items, item = blockIdx.x % n_items;
  if (blockIdx.x == 0 && tid < 8) queue[tid] = first_tickets;
  const int qb0 = span * item;
  const bool second = span == 2 && qb0 + 1 < nb;
  const int qb1 = second ? qb0 + 1 : qb0;
  const int sf0 = (qb0 / bps) * bps, sf1 = (qb1 / bps) * bps;
  const int32_t* l0 = cols + ((int64_t)bh * nb + qb0) * nb;
  const int32_t* l1 = l0 + (second ? nb : 0);
  const int n0 = cols ? cnt[(int64_t)bh * nb + qb0] : 0;
  const int n1 = cols && second ? cnt[(int64_t)bh * nb + qb1] : 0;
  constexpr int MAX_PER = 4096 / MERGE_THREADS;
  int c0[MAX_PER], c1[MAX_PER];
#pragma unroll
  for (int u = 0; u < MAX_PER; ++u) {
    const int i = tid + MERGE_THREADS * u;
    c0[u] = i < n0 ? l0[i] : 0;
    c1[u] = i < n1 ? l1[i] : 0;
  }
  for (int i = tid; i < nb; i += MERGE_THREADS) {
    flags0[i] = !cols && i < sf0 ? 1 : 0;
    flags1[i] = !cols && second && i < sf1 ? 2 : 0;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < MAX_PER; ++u) {
    const int i = tid + MERGE_THREADS * u;
    if (i < n0) flags0[c0[u]] = 1;
    if (i < n1) flags1[c1[u]] = 2;
  }
  __syncthreads();
  // compaction: thread t owns `per` consecutive key blocks; wave-level prefix, then wave totals
  const int per = (nb + MERGE_THREADS - 1) / MERGE_THREADS;
  const int k0 = tid * per, k1 = min(k0 + per, nb);
  int c = 0;
  for (int kb = k0; kb < k1; ++kb) c += (flags0[kb] | flags1[kb]) ? 1 : 0;
  int incl = c;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int up = __shfl_up(incl, off, 64);
    if (lane >= off) incl += up;
  }
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  int w = incl - c, total = 0;
#pragma unroll
  for (int x = 0; x < MERGE_THREADS / 64; ++x) {
    const int ws = wsum[x];
    if (x < wave) w += ws;
    total += ws;
  }
  uint16_t* out = plist + ((int64_t)bh * n_items + (n_items - 1 - item)) * cap;
  if (tid == 0) {
    const int h = bh % Hq;
    out[1] = (uint16_t)(bh / Hq);
    out[2] = (uint16_t)h;
    out[3] = (uint16_t)(h / group);
    out[4] = (uint16_t)qb0;
    out[5] = (uint16_t)(second ? 2 : 1);
  }
  uint16_t* const header = out;
  out += LIST_HEADER;
  for (int kb = k0; kb < k1; ++kb) {
    const int f = flags0[kb] | flags1[kb];
    if (f) out[w++] = (uint16_t)(kb | (f << 14));
  }
  const int n_own = qb1 - sf0 + 1;
  if (own_needed) {
    // one-block segments with an optional diagonal: a query block's own block is listed only where its flag is set
    if (tid == 0) {
      int n = total;
      if (own_needed[(int64_t)bh * nb + qb0]) out[n++] = (uint16_t)(qb0 | ENT_ORIG | (1u << 14));
      if (second && own_needed[(int64_t)bh * nb + qb1]) out[n++] = (uint16_t)(qb1 | ENT_ORIG | (2u << 14));
      // every list ends with an own-segment entry: a pair with neither own block listed gets the first one's, used by
      // neither query block.  The attention kernel's item protocol -- first tile in flight, claim and hand-over of the
      // next item at the last tiles -- then needs no empty case and none where a permuted tile ends the item; a query
      // block that used no tile writes zeros
      if (n == total) out[n++] = (uint16_t)(qb0 | ENT_ORIG);
      header[0] = (uint16_t)n;
    }
    return;
  }
  for (int t = tid; t < n_own; t += MERGE_THREADS) {
    const int kb = sf0 + t;
    const int f = (kb <= qb0 ? 1 : 0) | ((second && kb >= sf1) ? 2 : 0);
    out[total + t] = (uint16_t)(kb | ENT_ORIG | (f << 14));
  }
  if (tid == 0) header[0] = (uint16_t)(total + n_own);
}

// Ticket `ticket` (counted from the range's first) of XCD range x, [begin, end) -> work item, or NO_ITEM past the range's end.  Items
// are numbered head by head, long ones first, and in a large launch handed out in that order (an XCD walks one head at a time: its
// workgroups share that head's K / V stream in L2).  A launch with only a few items per workgroup cannot balance that way: a
// workgroup that starts with a short item of one head is handed a long item of the next and finishes last.  There the
// same item of several heads goes out before the next shorter one.  DEAL_GROUPS (every range is of whole heads): DEAL_HEADS heads
// of the range at a time, since an XCD's L2 holds the tiles of a few (4 x 28 / 4 heads x 2513, over the range's fourteen: 285 -> 291 us);
// at two items a workgroup and fewer, all of the range's (4 x 32 / 8 heads x 1021 in one segment 49 us, four at a time 55).
// DEAL_ALL: all heads, dealt to the XCDs in turn.  Whole pass, head by head -> dealt: 28 / 4 heads x 4096
// 199 -> 164 us, x 5120 250 -> 222, x 10240 675 -> 641; 32 / 8 x 4352 219 -> 200, x 5120 260 -> 248, x 10240 731 -> 711.
// DEAL_BY_LISTS: DEAL_GROUPS where the visit lists are short, else DEAL_NONE (see lists_are_short).
// (Wave-uniform values: scalar arithmetic only.)
constexpr int NO_ITEM = 1 << 28, DEAL_NONE = 0, DEAL_GROUPS = 1, DEAL_ALL = 2, DEAL_BY_LISTS = 3, DEAL_HEADS = 4;
__device__ __forceinline__ int quotient(int r, int divisor, uint32_t magic) { return divisor == 1 ? r : (int)(((uint64_t)(uint32_t)r * magic) >> 32); }
__device__ __forceinline__ int ticket_item(const AttnArgs::Deal& d, int how, int x, int begin, int end, int ticket) {
  if (begin + ticket >= end) return NO_ITEM;
  if (how == DEAL_NONE) return begin + ticket;
  const int n = d.n, m = d.heads;
  if (how == DEAL_ALL) {
    const int r = 8 * ticket + x, len = quotient(r, m, d.heads_magic);
    return (r - len * m) * n + len;
  }
  const int group = quotient(ticket, m * n, d.group_magic) * (m * n), r = ticket - group;
  const int left = end - begin - group;   // items of this group of heads and those after it
  int heads = m, len;
  if (left >= m * n) {
    len = quotient(r, m, d.heads_magic);
  } else {   // the last DEAL_HEADS - 1 heads of a range and fewer
    heads = left >= 3 * n ? 3 : left >= 2 * n ? 2 : 1;
    len = heads == 3 ? quotient(r, 3, 0x55555556u) : r >> (heads - 1);
  }
  return begin + group + (r - len * heads) * n + len;
}

// Whether an item visits few tiles, from 64 lists across the launch: every workgroup reads the same ones.  Such a launch gains by
// the dealt order at any length: 2 x 32 / 8 heads x 13333 concentrated 947 -> 877 us a pass, 32 / 8 x 30000 1449 -> 1416, x 131072 2780 ->
// 2690.  Where lists are long it loses what an XCD's workgroups share of a head in L2: 32 / 8 x 64000 with 100 tiles an item
// 9.75 -> 10.11 ms, near-uniform 2 x 32 / 8 x 13333 (0.8 of an item's causal tiles and more) 2276 -> 2312 us.  Around the line, 32 / 8 x
// 64000 in segments of 512, head by head -> dealt: 35 tiles an item 3976 -> 3928 us, 40 4465 -> 4421, 47 5101 -> 5023, 56 5955 -> 5895, by about as
// much as runs differ (1 - 2 %): it lies at the lower end of where dealing stops to gain.  (A round trip to memory at the kernel's start, 2 us.)
constexpr int SHORT_LIST = 40;
__device__ __forceinline__ bool lists_are_short(ArgsPtr a) {
  const int n = a->deal.n, lane = lane_id_here();
  // one of every 64th part of the items, at another place in each: lists grow shorter towards a head's end (65 * 63 < 4096: never past the last)
  const int64_t item = ((int64_t)a->BH * n * (65 * lane)) >> 12;
  uint32_t tiles = a->plist[item * a->cap];
  auto add = [&](auto t) __attribute__((always_inline)) { return t.a + t.b; };
  tiles = add(with_lane_xor<1>(tiles));
  tiles = add(with_lane_xor<2>(tiles));
  tiles = add(with_lane_xor<4>(tiles));
  tiles = add(with_lane_xor<8>(tiles));
  tiles = add(with_lane_xor<16>(tiles));
  tiles = add(with_lane_xor<32>(tiles));
  return __builtin_amdgcn_readfirstlane((int)tiles) <= min(46 * n, 64 * SHORT_LIST);   // (64 times 0.72)
}

// asynchronous copy of one list row (`chunks` 16-byte pieces) into LDS at byte offset `lds_byte`
__device__ __forceinline__ void stage_list_async(const uint16_t* src, int chunks, uint32_t lds_byte, int wave, int tid) {
  const uint64_t src0 = (uint64_t)(uintptr_t)src;
  const uint32_t src_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)src0);
  const uint32_t src_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(src0 >> 32));
  const uint64_t srcu = ((uint64_t)src_hi << 32) | (uint64_t)src_lo;
  for (int p = 0; p * THREADS < chunks; ++p) {
    const int chunk = p * THREADS + tid;
    const uint32_t voff = (uint32_t)chunk * 16u;
    if (chunk < chunks) {
      register uint32_t m0v asm("m0") = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_byte + p * (THREADS * 16) + wave * 1024));
      asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0v), "v"(voff), "s"(srcu) : "memory");   // (wait states: see copy_tile_now)
    }
  }
}

__global__ __launch_bounds__(THREADS, 1) void sparse_attn_kernel(AttnArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];   // starts at LDS offset 0
  RESERVE_ACC_REGS();
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);

  // Work items = (head, one or two query blocks), numbered head by head with the long rows of a head first and cut
  // into eight contiguous ranges, one per XCD (blockIdx % 8).  Handed out in that order (ranges of about equal work) an XCD works
  // through one head at a time, so its resident workgroups walk the same permuted K/V stream at about the same pace and
  // share its tiles in that XCD's L2; passes of few items a head or of short lists deal several heads' items in turn instead
  // (ticket_item).  The launch holds one workgroup per CU; each takes the next item of its
  // XCD's range from a counter until the range is used up, so that the copies of an item's first tiles, the
  // fetch of its list and of its queries overlap the previous item's last tile and epilogue.
  // The arguments are read through the kernel-argument pointer where they are needed, and that pointer is made
  // opaque once per item: scalar loads from it stay next to their use instead of pinning some fifty scalar
  // registers for the whole kernel.
#define PBS_ARGS() ({ ArgsPtr p_ = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr(); asm volatile("" : "+s"(p_)); p_; })
  ArgsPtr a0 = PBS_ARGS();
  auto deal_of = [](ArgsPtr p) __attribute__((always_inline)) {
    return AttnArgs::Deal{p->deal.how, p->deal.n, p->deal.heads, p->deal.group_magic, p->deal.heads_magic};
  };
  AttnArgs::Deal d0 = deal_of(a0);
  // (loaded together, ahead of the branches that use them: one round trip at the kernel's start)
  asm volatile("" : "+s"(d0.how), "+s"(d0.n), "+s"(d0.heads), "+s"(d0.group_magic), "+s"(d0.heads_magic));
  int deal = d0.how;
  if (deal == DEAL_BY_LISTS) deal = lists_are_short(a0) ? DEAL_GROUPS : DEAL_NONE;
  const int xcd = blockIdx.x & 7;
  int q_begin = a0->xcd_start[xcd], q_end = a0->xcd_start[xcd + 1];   // the range being served: this XCD's, later others'
  int vic = xcd, vic_tried = a0->one_each ? 7 : 0;
  int* misc = reinterpret_cast<int*>(smem + LDS_MISC);   // [1] redo flag, [4] next item, [5] ranges with items left
  // Another range that still has items, once this one is used up: true with the item in `found` and the range in
  // vic / q_begin / q_end.  All eight counters are read at once, and a range whose counter has passed its end is skipped
  // without asking for a ticket (counters only grow): at the end of a launch, when every range is used up, that is one round
  // trip to memory instead of seven.  (Read ahead, during the last item, they are out of date when they are looked at, and the
  // tickets asked for in vain cost more than the round trip: 32 / 8 heads x 4096 166.6 -> 169.0 us.)
  int found = 0;
  auto claim_elsewhere = [&]() __attribute__((always_inline)) {
    if (vic_tried >= 7) return false;
    ArgsPtr as = PBS_ARGS();
    __syncthreads();   // everyone has read the previous ticket
    if (wave == 0) {
      const int ln = lane_id_here();
      bool left = false;
      if (ln < 8) left = as->xcd_start[ln] + __hip_atomic_load(as->queue + ln, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < as->xcd_start[ln + 1];
      const uint64_t ranges = __ballot(left);
      if (ln == 0) misc[5] = (int)ranges;
    }
    __syncthreads();
    const int ranges = __builtin_amdgcn_readfirstlane(misc[5]);
    while (vic_tried < 7) {
      ++vic_tried;
      vic = (xcd + vic_tried) & 7;
      if (!(ranges >> vic & 1)) continue;
      q_begin = as->xcd_start[vic];
      q_end = as->xcd_start[vic + 1];
      __syncthreads();   // everyone has read the previous ticket
      if (wave == 0 && lane_id_here() == 0) misc[4] = atomicAdd(as->queue + vic, 1);
      __syncthreads();
      found = ticket_item(deal_of(as), deal, vic, q_begin, q_end, __builtin_amdgcn_readfirstlane(misc[4]));
      if (found < NO_ITEM) return true;
    }
    return false;
  };
  // The first item: workgroup n of an XCD takes ticket n, without asking (the counters start behind these tickets); where the
  // range is shorter than that, an item of another one.
  if (threadIdx.x == 0) misc[1] = 0;
  int cur = ticket_item(d0, deal, xcd, q_begin, q_end, (int)blockIdx.x >> 3);
  if (PBS_UNLIKELY(cur == NO_ITEM)) {
    if (!claim_elsewhere()) return;
    cur = found;
  }
  int nxt = NO_ITEM;   // the next item is claimed late in the current one: an item claimed early waits for this
                     // workgroup while others may be idle
  bool has_nxt = false;

  // an item's coordinates, from the header of its list in LDS, and the base pointers of its head's tiles: permuted K,
  // permuted V^T, original K and V rows
  struct Item {
    int n_tiles, b, h, qb0;
    const uint16_t *pk, *pvt, *korig, *vorig;
    uint32_t k_ss, v_ss;
    int S, q_end;   // q_end: end of the item's queries
  };
  auto read_item = [&](ArgsPtr ap, const uint16_t* list) __attribute__((always_inline)) {
    Item t;
    const u32x4 hd = *reinterpret_cast<const u32x4*>(list);
    const uint32_t w0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)hd[0]), w1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)hd[1]);
    t.n_tiles = (int)(w0 & 0xffffu);
    t.b = (int)(w0 >> 16);
    t.h = (int)(w1 & 0xffffu);
    const uint32_t w2 = (uint32_t)__builtin_amdgcn_readfirstlane((int)hd[2]);
    t.qb0 = (int)(w2 & 0xffffu);
    const int64_t tiles = (int64_t)(t.b * ap->Hq + t.h) * ap->nb * (BS * D), kvh = (int)(w1 >> 16);
    t.pk = ap->pk + tiles;
    t.pvt = ap->pvt + tiles;
    t.korig = ap->k + t.b * ap->k_sb + kvh * ap->k_sh;
    t.vorig = ap->v + t.b * ap->v_sb + kvh * ap->v_sh;
    t.k_ss = ap->k_ss;
    t.v_ss = ap->v_ss;
    t.S = ap->S;
    t.q_end = min(t.S, (t.qb0 + (int)(w2 >> 16)) * BS);
    return t;
  };
  auto first_entry = [&](const uint16_t* list) __attribute__((always_inline)) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)list[LIST_HEADER]);
  };
  // Aims the tile copy at the tile of list entry `e`, into the buffers at LDS byte offset `buf`: the addresses here, and
  // where the kind of tile changes the per-lane offsets (16 registers).  The copy in hand at a tile's head is always the
  // one that fetched that tile, so the tile loops, which run over tiles of one kind, leave the offsets alone: written
  // under a branch of such a loop they would be copied twice per tile.
  TileCopy copy;
  auto aim_perm = [&](const Item& t, uint32_t e, uint32_t buf) __attribute__((always_inline)) {
    const int64_t tile = (int64_t)(e & ENT_KB) * (BS * D);
    copy.lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(buf + (uint32_t)wave * 8192u));
    copy.k = uniform64((uint64_t)(uintptr_t)(t.pk + tile) - COPY_BIAS);
    copy.v = uniform64((uint64_t)(uintptr_t)(t.pvt + tile) - COPY_BIAS);
  };
  auto aim_rows = [&](const Item& t, uint32_t e, uint32_t buf) __attribute__((always_inline)) {
    const int64_t row = (int64_t)(e & ENT_KB) * BS;
    copy.lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(buf + (uint32_t)wave * 8192u));
    copy.k = uniform64((uint64_t)(uintptr_t)(t.korig + row * t.k_ss) - COPY_BIAS);
    copy.v = uniform64((uint64_t)(uintptr_t)(t.vorig + row * t.v_ss) - COPY_BIAS);
  };
  auto rows_of = [&](const Item& t, uint32_t e) __attribute__((always_inline)) { return t.S - (int)(e & ENT_KB) * BS; };   // >= 128 but for the last block
  auto aim_anew = [&](const Item& t, uint32_t e, uint32_t buf) __attribute__((always_inline)) {
    // the lane ids are formed afresh: what is derived from the item's one gets hoisted out of the tile loops
    if (e & ENT_ORIG) {
      aim_rows(t, e, buf);
      copy_offsets_rows(copy, t.k_ss, t.v_ss, rows_of(t, e), wave, lane_id_here());
    } else {
      aim_perm(t, e, buf);
      copy_offsets_perm(copy, wave, lane_id_here());
    }
  };
  auto list_row = [&](ArgsPtr ap, int item) __attribute__((always_inline)) { return ap->plist + (int64_t)item * ap->cap; };
  // an item's Q^T fragments (B operand): column i16 of group qg is query 32 wave + 16 (qg % 2) + i16 of block qg / 2,
  // d = 32 kd + 8 g4 + 0..7.  Rows past the end of the item's queries compute on the last row's values and are never stored.
  auto load_q = [&](ArgsPtr aq, const Item& t, auto set) __attribute__((always_inline)) {
    const int ln = lane_id_here();
    const int64_t q_ss = aq->q_ss;
    const uint16_t* qhead = aq->q + t.b * aq->q_sb + t.h * aq->q_sh + 8 * (ln >> 4);
    const int last = t.q_end - 1, pos0 = t.qb0 * BS + 32 * wave + (ln & 15);
    static_for<QG>([&](auto qc) __attribute__((always_inline)) {
      constexpr int qg = decltype(qc)::value, st = decltype(set)::value;
      const uint16_t* qrow = qhead + (int64_t)min(pos0 + (qg >> 1) * BS + (qg & 1) * 16, last) * q_ss;
      q_load<qg, 0, st>(qrow);
      q_load<qg, 1, st>(qrow + 32);
      q_load<qg, 2, st>(qrow + 64);
      q_load<qg, 3, st>(qrow + 96);
    });
  };

  // Without lists in memory: the list of an item of a sequence inside one segment, straight into LDS.  Taken where every item
  // has a workgroup of its own, so that nothing is left of the list kernel (counters, further items).
  auto own_list = [&](ArgsPtr ap, int item) __attribute__((always_inline)) {
    uint16_t* list = reinterpret_cast<uint16_t*>(smem + LDS_LIST);
    const int n_items = ap->deal.n, bh = item / n_items, qb0 = ap->span * (n_items - 1 - (item - bh * n_items));
    const bool second = ap->span == 2 && qb0 + 1 < ap->nb;
    const int n_own = second ? qb0 + 2 : qb0 + 1;
    for (int kb = (int)threadIdx.x; kb < n_own; kb += THREADS)
      list[LIST_HEADER + kb] = (uint16_t)((uint32_t)kb | ENT_ORIG | (kb <= qb0 ? 1u << 14 : 0u) | (second ? 2u << 14 : 0u));
    if (threadIdx.x == 0) {
      const int b = bh / ap->Hq, h = bh - b * ap->Hq;
      list[0] = (uint16_t)n_own;
      list[1] = (uint16_t)b;
      list[2] = (uint16_t)h;
      list[3] = (uint16_t)(h / (ap->Hq / ap->Hkv));
      list[4] = (uint16_t)qb0;
      list[5] = (uint16_t)(second ? 2 : 1);
    }
  };

  // the first item's list, then its first tile
  if (a0->cap) stage_list_async(list_row(a0, cur), a0->cap >> 3, LDS_LIST, wave, (int)threadIdx.x);
  else own_list(a0, cur);
  __builtin_amdgcn_s_waitcnt(0x0f70);
  __syncthreads();
  uint32_t li = 0;        // which list buffer holds the current item's list
  uint32_t par = 0;       // which tile buffers hold the current item's first tile (0 or 0x8000)
  {
    const uint16_t* list0 = reinterpret_cast<const uint16_t*>(smem + LDS_LIST);
    aim_anew(read_item(a0, list0), first_entry(list0), 0u);
  }
  copy_tile_now(copy);

  bool careful_only = false;   // the current pass repeats an item without speculation
  bool q_ready = false;        // the item's queries have been loaded ahead
  for (;;) {
    const uint16_t* mlist = reinterpret_cast<const uint16_t*>(smem + LDS_LIST + li * LIST_BYTES);
    const uint16_t* nlist = reinterpret_cast<const uint16_t*>(smem + LDS_LIST + (li ^ 1u) * LIST_BYTES);
    ArgsPtr ap = PBS_ARGS();
    // everything per lane is derived afresh from the lane id in every item: nothing but scalars lives across items
    const int lane = lane_id_here();
    const int i16 = lane & 15, g4 = lane >> 4;
    // per-lane LDS byte offsets of the fragments inside buffer 0; XOR 0x8000 switches buffer.
    //   K fragment (sub-tile ks, row tile T, d-step kd) : (koff0 ^ kd << 6) + T * 1024 + ks * 8192
    //   V^T fragment (sub-tile ks, d tile dt)           : (voff0 ^ ks << 6) + dt * 4096
    // The 16-byte chunk index is XORed with a hash of the row, so the fragments of a row lie at (offset of the
    // first) ^ (n << 6).
    const int krow = 8 * (i16 >> 2) + (i16 & 3);   // k_row_hash(krow) == i16
    const uint32_t koff0 = (uint32_t)(krow * 256 + ((g4 ^ i16) * 16));
    const uint32_t voff0 = LDS_V0 + (uint32_t)(i16 * 256 + ((g4 ^ i16) * 16));
    // the addresses in the buffers of the item's first tile; switched to the other buffers after every tile
    uint32_t ka[4], va[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      ka[n] = koff0 ^ (uint32_t)(n << 6) ^ par;
      va[n] = voff0 ^ (uint32_t)(n << 6) ^ par;
    }
    int claim = 0;   // ticket of the next item: in flight during one tile

    const Item hb = read_item(ap, mlist);
    const int qb0 = hb.qb0, n_tiles = hb.n_tiles;
    const float c_log2 = ap->scale_log2;

    // the next item: claimed three tiles before the end of this one (the counter's latency passes under a
    // tile), published and its list requested one tile later, its queries and its first tile requested at the last
    // tile.  Items of fewer than three tiles finish these steps after their loop.
    const int claim_it = careful_only || ap->one_each ? -8 : max(n_tiles - 3, 0);
    auto publish_and_fetch = [&]() __attribute__((always_inline)) {   // between the wait for this thread's loads and the barrier ...
      if (wave == 0 && lane_id_here() == 0) misc[4] = claim;
    };
    auto adopt_next = [&]() __attribute__((always_inline)) {          // ... and after the barrier
      nxt = ticket_item(deal_of(PBS_ARGS()), deal, vic, q_begin, q_end, __builtin_amdgcn_readfirstlane(misc[4]));
      has_nxt = nxt < NO_ITEM;
      if (has_nxt)
        stage_list_async(list_row(PBS_ARGS(), nxt), PBS_ARGS()->cap >> 3, LDS_LIST + (li ^ 1u) * LIST_BYTES, wave, wave * 64 + lane_id_here());
    };
    // the next item's queries and first tile, once its list has landed
    auto aim_at_next = [&](uint32_t buf) __attribute__((always_inline)) {
      ArgsPtr an = PBS_ARGS();
      const Item t = read_item(an, nlist);
      load_q(an, t, std::integral_constant<int, Q_NEXT>{});
      aim_anew(t, first_entry(nlist), buf);
    };

    {
      float m_ref[QG], l_row[QG];   // reference maxima and row sums of queries 16 qg + i16, identical in the four lanes i16 + 16 g
#pragma unroll
      for (int qg = 0; qg < QG; ++qg) {
        m_ref[qg] = -INFINITY;
        l_row[qg] = 0.f;
      }
      bool poisoned = false;
      uint32_t unseen = 3u << 14;   // use bits of the query blocks that have seen no tile yet (their reference is still -inf)

      uint32_t bufx = par;
      auto next_buffers = [&]() __attribute__((always_inline)) {
        bufx ^= 0x8000u;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          ka[n] ^= 0x8000u;
          va[n] ^= 0x8000u;
        }
      };
      // a tile's copies are awaited at the end of the tile before it, those of an item's first tile here, and with them the
      // item's queries.  Loads from inline assembly are unknown to the compiler and not interlocked by the hardware, so nothing
      // may touch their registers before this wait (tests/test_attention_registers.py follows every path through the compiled
      // code); the accumulators are cleared in its shadow.
      auto wait_copies = [&]() __attribute__((always_inline)) { __builtin_amdgcn_s_waitcnt(0x0f70); };   // vmcnt(0)
      if (PBS_UNLIKELY(careful_only)) {
        // the redo pass starts the item over: its first tile goes back into the buffers it had (the next
        // item's first tile, if it was on its way there, is fetched again at the end of this pass)
        wait_copies();
        __syncthreads();
        aim_anew(hb, first_entry(mlist), par);
        copy_tile_now(copy);
        o_clear();
        wait_copies();
      } else if (q_ready) {
        // requested at the previous item's last tile.  (Leaving the previous item's stores on their way, which are younger, is
        // no faster: 1000 tokens 73.8 us either way, 128k concentrated 3.00 ms)
        o_clear();
        wait_copies();
        q_advance();
      } else {
        load_q(ap, hb, std::integral_constant<int, 0>{});
        o_clear();
        wait_copies();
      }
      uint32_t e_cur = first_entry(mlist);         // the entry of the current tile
      uint32_t e_nxt = 0;                          // of the next one, set by tile_head
      uint16_t e_ahead = mlist[LIST_HEADER + 1];   // per lane, not yet made uniform
      // what every tile starts with: hand over the buffers of the tile before
      auto tile_head = [&](int it) __attribute__((always_inline)) {
        if (PBS_UNLIKELY(it == claim_it + 1)) publish_and_fetch();
        __syncthreads();                      // every wave's share of tile `it` has landed; every wave is done with tile it - 1
        if (PBS_UNLIKELY((unsigned)(it - claim_it) < 2u)) {
          if (it != claim_it) adopt_next();
          else if (wave == 0 && lane_id_here() == 0) claim = atomicAdd(PBS_ARGS()->queue + vic, 1);
        }
        // the list entries are read from LDS one tile ahead of their use (the read's latency would otherwise sit in
        // front of the copy requests of every tile): `e_ahead` holds entry it + 1, requested at the tile before
        e_nxt = (uint32_t)__builtin_amdgcn_readfirstlane((int)e_ahead);
        e_ahead = mlist[LIST_HEADER + 2 + it];
      };
      // at the item's last tile: the next item's first tile
      auto aim_past_item = [&]() __attribute__((always_inline)) {
        if (has_nxt && (careful_only || n_tiles >= 3)) aim_at_next(bufx ^ 0x8000u);   // shorter items: after the loop, once the list has landed
        else copy.lds ^= 0x8000u;   // nothing to fetch: the same tile again, into buffers nobody reads (a pipelined tile always copies)
      };
      // logits of the 32 keys at byte offset `at` of the K buffer against the queries of column groups Q0 .. Q0 + NQ - 1 (the
      // fence behind them is the caller's); `between` goes out after every d-step
      auto logits_of = [&](auto q0c, auto& s, int at, auto between) __attribute__((always_inline)) {
        constexpr int Q0 = decltype(q0c)::value, NQ = sizeof(s[0]) / sizeof(s[0][0]);
        static_for<2>([&](auto tc) __attribute__((always_inline)) {
          constexpr int T = decltype(tc)::value;
          bf16x8 fk[4];
#pragma unroll
          for (int kd = 0; kd < 4; ++kd) fk[kd] = ldsf(ka[kd] + at + T * 1024);
          static_for<4>([&](auto kc) __attribute__((always_inline)) {
            constexpr int kd = decltype(kc)::value;
            static_for<NQ>([&](auto qc) __attribute__((always_inline)) {
              constexpr int q = decltype(qc)::value;
              mfma_s<Q0 + q, kd, kd == 0>(s[T][q], fk[kd]);
            });
            between(std::integral_constant<int, 4 * T + kd>{});
          });
        });
      };
      // first tile of a row, every key visible: the exact maximum over its first 32 keys is a good enough reference
      // to start the pipelined path (later keys move it up lazily).  (Over 16 keys the results' error against 64-bit arithmetic was 0.5 to 1 %
      // larger: a reference that is the maximum has the probability 1, which bf16 holds exactly.)
      auto first_reference = [&](auto q0c, uint32_t ent) __attribute__((always_inline)) {   // for column groups q0c .. QG - 1
        constexpr int Q0 = decltype(q0c)::value;
        f32x4 s0[2][QG - Q0];
        logits_of(q0c, s0, 0, [](auto) {});
        MFMA_FENCE();
#pragma unroll
        for (int qg = Q0; qg < QG; ++qg) {
          const f32x4 a = s0[0][qg - Q0], b = s0[1][qg - Q0];
          const float mx = max3(max3(a[0], a[1], a[2]), max3(a[3], b[0], b[1]), max3(b[2], b[3], b[3]));
          const float m_new = max_over_lane_groups(mx) * c_log2;
          if (ent & unseen & (1u << (14 + (qg >> 1)))) m_ref[qg] = m_new;
        }
        unseen &= ~ent;
      };
      // online softmax over the 32 keys with logits s ([row tile][column group]): the running maxima m move up, the sums l follow;
      // alpha is what earlier sums are to be scaled by, pf the probabilities
      auto online_step = [&](const f32x4 (&s)[2][2], float (&m)[2], float (&l)[2], float (&alpha)[2], bf16x8 (&pf)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float mx = max3(s[0][q][0], s[0][q][1], s[0][q][2]);
          mx = max3(mx, s[0][q][3], s[1][q][0]);
          mx = max3(mx, s[1][q][1], s[1][q][2]);
          mx = max_over_lane_groups(max3(mx, mx, s[1][q][3]));
          const float m_new = fmaxf(m[q], mx * c_log2);
          const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
          alpha[q] = __builtin_amdgcn_exp2f(m[q] - m_use);
          m[q] = m_new;
          float rs = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float pe = __builtin_amdgcn_exp2f(s[e >> 2][q][e & 3] * c_log2 - m_use);
            rs += pe;
            pf[q][e] = (__bf16)pe;
          }
          l[q] = l[q] * alpha[q] + sum_over_lane_groups(rs);
        }
      };
      // the logits of sub-tile ks of a block's diagonal tile: keys after the query out
      auto hide_later_keys = [&](f32x4 (&s)[2][2], int ks) __attribute__((always_inline)) {
        const int ln = lane_id_here();   // keep the compares inside the tile (see fast_tile)
        const int qrel8 = 32 * (wave - ks) + (ln & 15) - 8 * (ln >> 4);
#pragma unroll
        for (int T = 0; T < 2; ++T)
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (4 * T + r - 16 * q > qrel8) s[T][q][r] = -INFINITY;
      };
      // careful tile (the redo pass), for one of the pair's blocks: classic online softmax, one 32-key sub-tile at a time
      auto careful_tile = [&](auto bc, uint32_t ent) __attribute__((always_inline)) {
        constexpr int block = decltype(bc)::value, Q0 = 2 * block;
        const bool masked = (ent & ENT_ORIG) && (int)(ent & ENT_KB) == qb0 + block;
        MFMA_FENCE();
#pragma nounroll
        for (int ks = 0; ks < 4; ++ks) {   // a real loop: the rare path stays small, in code and in registers
          f32x4 s[2][2];   // [T][column group - Q0]
          logits_of(std::integral_constant<int, Q0>{}, s, ks * 8192, [](auto) {});
          MFMA_FENCE();
          if (masked) hide_later_keys(s, ks);
          float m[2] = {m_ref[Q0], m_ref[Q0 + 1]}, l[2] = {l_row[Q0], l_row[Q0 + 1]}, alpha[2];
          bf16x8 pf[2];
          online_step(s, m, l, alpha, pf);
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            m_ref[Q0 + q] = m[q];
            l_row[Q0 + q] = l[q];
          }
          if (__any(alpha[0] != 1.0f || alpha[1] != 1.0f)) {
            o_scale<Q0>(alpha[0]);
            o_scale<Q0 + 1>(alpha[1]);
          }
          MFMA_FENCE();
          static_for<8>([&](auto dc) __attribute__((always_inline)) {
            constexpr int dt = decltype(dc)::value;
            const bf16x8 fv = (ent & ENT_ORIG)
                                  ? ldsf_transposed(vrow_lane_addr(LDS_V0 + (va[0] & 0x8000u), lane_id_here()) + dt * 128 + ks * 8192)
                                  : ldsf((va[0] ^ (uint32_t)(ks << 6)) + dt * 4096);
            mfma_o<dt, Q0>(fv, pf[0]);
            mfma_o<dt, Q0 + 1>(fv, pf[1]);
          });
          MFMA_FENCE();
        }
      };
      // A diagonal tile that is its block's first tile (the first 128 keys of a sequence, or a block that selected nothing): online
      // softmax as well, since with a reference from some of so few keys the error against 64-bit arithmetic was 3 %
      // larger.  The logits come first, the next tile's copies between them, and the sums stay in vector registers, O being
      // zero so far; sub-tiles up to the wave's own (the rest is hidden), none where its queries lie past the sequence.  (Attention
      // launch, pipelined form -> this: 77 tokens 10.3 -> 10.4 us, 128 tokens 10.4 -> 11.0, 256 tokens on 16 heads 12.9 -> 15.0; with
      // the careful tile above 77 tokens took 13.0 and 256 about 18.)
      auto first_diagonal_tile = [&](auto bc) __attribute__((always_inline)) {
        constexpr int block = decltype(bc)::value, Q0 = 2 * block;
        if ((qb0 + block) * BS + 32 * wave >= hb.q_end) {
          copy_tile_now(copy);
          return;
        }
        f32x4 s[4][2][2], o[8][2];
        asm volatile("s_nop 4");   // (as in copy_tile_now)
        static_for<4>([&](auto kc) __attribute__((always_inline)) {
          constexpr int ks = decltype(kc)::value;
          logits_of(std::integral_constant<int, Q0>{}, s[ks], ks * 8192, [&](auto ic) __attribute__((always_inline)) {
            constexpr int i = 8 * ks + decltype(ic)::value;
            if constexpr (i % 2 == 0) copy_piece<i / 2>(copy);
          });
        });
        const uint32_t vr = vrow_lane_addr(LDS_V0 + (va[0] & 0x8000u), lane_id_here());
        float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
        MFMA_FENCE();
        static_for<4>([&](auto kc) __attribute__((always_inline)) {
          constexpr int ks = decltype(kc)::value;
          if (ks == 0 || ks <= wave) {
            if (ks == wave) hide_later_keys(s[ks], ks);
            float alpha[2];
            bf16x8 pf[2];
            online_step(s[ks], m, l, alpha, pf);
            if constexpr (ks > 0) {
#pragma unroll
              for (int dt = 0; dt < 8; ++dt)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                  for (int r = 0; r < 4; ++r) o[dt][q][r] *= alpha[q];
            }
            bf16x8 fv[8];
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) fv[dt] = ldsf_transposed(vr + dt * 128 + ks * 8192);
            MFMA_FENCE();
            static_for<8>([&](auto dc) __attribute__((always_inline)) {
              constexpr int dt = decltype(dc)::value;
              mfma_v<ks == 0>(o[dt][0], fv[dt], pf[0]);
              mfma_v<ks == 0>(o[dt][1], fv[dt], pf[1]);
            });
            MFMA_FENCE();
          }
        });
        static_for<8>([&](auto dc) __attribute__((always_inline)) {
          constexpr int dt = decltype(dc)::value;
          o_set<dt, Q0>(o[dt][0]);
          o_set<dt, Q0 + 1>(o[dt][1]);
        });
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          m_ref[Q0 + q] = m[q];
          l_row[Q0 + q] = l[q];
        }
      };
      constexpr std::integral_constant<int, 0> block0{};
      constexpr std::integral_constant<int, 1> block1{};
      // The merged list holds the permuted tiles of earlier segments first, then the tiles of the own segments in
      // ascending order: for a query block those before its own block, its own (diagonal) block, and -- for the first
      // block of a pair -- the second block's, which it skips.  Each kind has a loop of its own, and so has the redo
      // pass: what differs between kinds -- the sixteen per-lane offsets of the tile copy, the fragment reads of V, the masks
      // -- is then fixed inside a loop, and its common path is straight code.  (O's 128 accumulation registers are named, see
      // pbs_attn_tile.h, and stay in place whatever the loops look like.)
      int it = 0;
      constexpr uint32_t USE0 = 1u << 14, USE1 = 1u << 15;
      if (PBS_UNLIKELY(careful_only)) {
        for (; it < n_tiles; ++it, next_buffers(), e_cur = e_nxt) {
          tile_head(it);
          if (it + 1 < n_tiles) aim_anew(hb, e_nxt, bufx ^ 0x8000u);
          else aim_past_item();
          copy_tile_now(copy);
          if (e_cur & USE0) careful_tile(block0, e_cur);
          if (e_cur & USE1) careful_tile(block1, e_cur);
          wait_copies();
        }
      } else {
        auto next_tile = [&]() __attribute__((always_inline)) {
          ++it;
          next_buffers();
          e_cur = e_nxt;
        };
        // A tile that one block only visits runs for that block's column groups: what the other one did not select stays out of
        // its rows, whatever its values.  The second blocks' diagonal tiles included, 9 to 14 % of all tiles are of that kind at 4k .. 64k,
        // 1.4 % at 128k (zero probabilities for the other two groups instead -> this: MeanPooling 16k 1648 -> 1583 us, 32k
        // 6.11 -> 5.93 ms, 64k layer 23.97 -> 23.05 ms; 128k 86.0 ms either way).
        auto visit = [&](auto masked, auto v_rows) __attribute__((always_inline)) {
          constexpr int MASKED = decltype(masked)::value;
          constexpr bool V_ROWS = decltype(v_rows)::value;
          if (PBS_UNLIKELY(e_cur & unseen)) first_reference(std::integral_constant<int, 0>{}, e_cur);
          if (PBS_LIKELY((e_cur & (USE0 | USE1)) == (USE0 | USE1)))
            fast_tile<0, 4, MASKED, V_ROWS>(ka, va, c_log2, m_ref, l_row, poisoned, wave, copy);
          else if ((MASKED && V_ROWS) || (e_cur & USE0))   // (a diagonal tile is one of its own block)
            fast_tile<0, 2, MASKED, V_ROWS>(ka, va, c_log2, m_ref, l_row, poisoned, wave, copy);
          else
            fast_tile<2, 2, MASKED, V_ROWS>(ka, va, c_log2, m_ref, l_row, poisoned, wave, copy);
        };
        constexpr std::integral_constant<int, 0> all_visible{};
        constexpr std::integral_constant<int, 3> diagonal0{};
        // permuted tiles (an item's last tile never is one), the last one apart
        if (!(e_cur & ENT_ORIG)) {
          for (;;) {
            tile_head(it);
            if (PBS_UNLIKELY(e_nxt & ENT_ORIG)) break;
            aim_perm(hb, e_nxt, bufx ^ 0x8000u);
            visit(all_visible, std::false_type{});
            wait_copies();
            next_tile();
          }
          aim_anew(hb, e_nxt, bufx ^ 0x8000u);
          visit(all_visible, std::false_type{});
          wait_copies();
          next_tile();
        }
        // own-segment tiles before the first diagonal: every key visible, a diagonal tile follows; the last one apart
        if ((int)(e_cur & ENT_KB) < qb0) {
          for (;;) {
            tile_head(it);
            if ((int)(e_nxt & ENT_KB) >= qb0) break;
            aim_rows(hb, e_nxt, bufx ^ 0x8000u);
            visit(all_visible, std::true_type{});
            wait_copies();
            next_tile();
          }
          aim_anew(hb, e_nxt, bufx ^ 0x8000u);
          visit(all_visible, std::true_type{});
          wait_copies();
          next_tile();
        }
        if ((int)(e_cur & ENT_KB) == qb0) {   // the first block's diagonal tile, or the place-holder of a pair that uses none
          tile_head(it);
          const bool more = it + 1 < n_tiles;
          if (more) aim_anew(hb, e_nxt, bufx ^ 0x8000u);
          else aim_past_item();
          if (PBS_UNLIKELY(e_cur & unseen & USE0)) {
            first_diagonal_tile(block0);
            if (e_cur & USE1) {
              if (unseen & USE1) first_reference(std::integral_constant<int, 2>{}, USE1);
              fast_tile<2, 2, 0, true, false>(ka, va, c_log2, m_ref, l_row, poisoned, wave, copy);
            }
          } else if (e_cur & (USE0 | USE1)) {
            visit(diagonal0, std::true_type{});
          } else {
            copy_tile_now(copy);
          }
          if (more) wait_copies();
          next_tile();
        }
        if (it < n_tiles) {   // the second block's diagonal tile, which nobody else sees
          tile_head(it);
          aim_past_item();
          if (PBS_UNLIKELY(e_cur & unseen)) {
            first_diagonal_tile(block1);
          } else {
            fast_tile<2, 2, 12, true>(ka, va, c_log2, m_ref, l_row, poisoned, wave, copy);
          }
          next_tile();
        }
      }
      if (claim_it >= 0 && n_tiles < 3) {
        if (n_tiles < 2) {
          __builtin_amdgcn_s_waitcnt(0x0f70);
          publish_and_fetch();
          __syncthreads();
          adopt_next();
        }
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
        if (has_nxt) {
          aim_at_next(bufx);
          copy_tile_now(copy);
        }
      }
      if (poisoned) misc[1] = 1;
      __syncthreads();   // every wave is done with the last tile
      if (!careful_only && misc[1] != 0) {   // the whole workgroup redoes both rows without speculation
        careful_only = true;
        continue;
      }

      // ---- epilogue: normalise and store from the registers.  Lane group g holds d 4 g .. 4 g + 3 of each d tile of its query; once the
      // odd and even groups have exchanged between two d tiles it is eight consecutive ones of the first (groups 0 and 2) or the
      // second (1 and 3): 16-byte stores, 64 consecutive bytes a row, the line's other half by the next store.  (Through LDS, in whole
      // rows of 256 bytes a store, 77 tokens of 32 / 8 heads took 9.89 us a call, now 9.36, before they had a kernel of their own; 1000 to 128k tokens
      // take the same.)  What bounds it is the arithmetic of a wave by itself on its SIMD: 400 vector instructions and 56 wait states for its sixteen
      // stores, 3770 to 3840 cycles, of which 3070 to 3150 remain with the stores masked off; 300 to 400 more pass before the first store.
      // a query block that used no tile (no selected block and no own block: possible only with an optional diagonal)
      // has a zero sum and writes zeros, as the reference does for a row without selected blocks
      MFMA_FENCE();
      // lane-dependent addresses of the epilogue come from a fresh opaque lane id: derived from the item's one
      // they would be computed at the top of the item and held across the tile loop
      const int lane_e = lane_id_here();
      ArgsPtr ae = PBS_ARGS();
      const int64_t o_ss = ae->o_ss;
      const int pos0 = qb0 * BS + 32 * wave + (lane_e & 15);      // this lane's first row
      uint16_t* const obase = ae->o + hb.b * ae->o_sb + hb.h * ae->o_sh + pos0 * o_ss + 16 * ((lane_e >> 4) & 1) + 8 * (lane_e >> 5);
      const bool full = (qb0 + 2) * BS <= hb.q_end;
      auto out_rows = [&](auto all, auto block) __attribute__((always_inline)) {
        static_for<2>([&](auto qc) __attribute__((always_inline)) {
          constexpr int qg = 2 * decltype(block)::value + decltype(qc)::value, rel = decltype(block)::value * BS + decltype(qc)::value * 16;
          const float inv = l_row[qg] == 0.f ? 0.f : 1.0f / l_row[qg];
          const bool live = decltype(all)::value || pos0 + rel < hb.q_end;
          uint16_t* const dst = obase + rel * o_ss;
          static_for<4>([&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            uint32_t two[2][2];
            static_for<2>([&](auto tc) __attribute__((always_inline)) {
              constexpr int t = decltype(tc)::value;
              const f32x4 o4 = o_get<2 * j + t, qg>();
#pragma unroll
              for (int e = 0; e < 2; ++e)
                two[t][e] = __builtin_bit_cast(uint32_t, (bf16x2){(__bf16)(o4[2 * e] * inv), (__bf16)(o4[2 * e + 1] * inv)});
            });
            const auto lo = __builtin_amdgcn_permlane16_swap(two[0][0], two[1][0], false, false);
            const auto hi = __builtin_amdgcn_permlane16_swap(two[0][1], two[1][1], false, false);
            if (live) *reinterpret_cast<u32x4*>(dst + 32 * j) = (u32x4){lo[0], hi[0], lo[1], hi[1]};
          });
        });
      };
      if (PBS_LIKELY(full)) {
        out_rows(std::true_type{}, block0);
        out_rows(std::true_type{}, block1);
      } else {   // the last block of a sequence, or an item of one block
        if (qb0 * BS + 32 * wave < hb.q_end) out_rows(std::false_type{}, block0);
        if ((qb0 + 1) * BS + 32 * wave < hb.q_end) out_rows(std::false_type{}, block1);
      }
    }
    bool stolen = false;
    if (!has_nxt) {
      // the range is used up: serve the other XCDs' ranges, one after the other.  No look-ahead on this path:
      // claim, fetch the list, request the first tile, each after the other
      ArgsPtr as = PBS_ARGS();
      has_nxt = claim_elsewhere();
      if (has_nxt) nxt = found;
      if (has_nxt) {
        stolen = true;
        stage_list_async(list_row(as, nxt), as->cap >> 3, LDS_LIST + (li ^ 1u) * LIST_BYTES, wave, wave * 64 + lane_id_here());
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
        aim_anew(read_item(as, nlist), first_entry(nlist), par ^ ((n_tiles & 1) ? 0x8000u : 0u));
        copy_tile_now(copy);
      }
    }
    if (!has_nxt) {
      __builtin_amdgcn_s_waitcnt(0x0f70);   // the last tile's copies, which nobody waits for, do not outlive the workgroup's LDS
      break;
    }
    q_ready = !stolen;
    careful_only = false;
    par ^= (n_tiles & 1) ? 0x8000u : 0u;
    li ^= 1u;
    cur = nxt;
    nxt = NO_ITEM;
    has_nxt = false;
    // (nobody is still to read it: it was zero when this item's last barrier had been passed, or the item was a repetition, which
    // does not read it; the next item's barriers lie before it can be set again)
    if (wave == 0 && lane_id_here() == 0) misc[1] = 0;
  }
}

std::atomic<uint64_t> g_lds_reserved{0};   // bit d: the kernel's LDS size has been raised on device d
std::atomic<int> g_cu_count[64];           // CUs of device d (0: not looked up yet)

}  // namespace

// uint16 per merged list row (a multiple of 8: rows stay 16-byte aligned): the header, at most nb blocks of
// earlier segments, at most bps + 1 own-segment blocks
static int list_cap(int nb, int bps) { return (LIST_HEADER + nb + std::min(bps, nb) + 1 + 7) / 8 * 8; }

// Query blocks per work item: two, which share every tile and each of its fragments, or, in a short pass, one.  A pass of few blocks
// leaves CUs idle or waits for its longest pair, and a tile for one block takes 2950 cycles against 5100 for two.  Whole pass,
// pairs -> single blocks, us: 32 / 8 heads x 1024 70.5 -> 67.8, x 1536 85.9 -> 81.8; 28 / 4 x 1000 74.3 -> 69.7; 4 / 1 x 8192 191 -> 146;
// in one segment 32 / 8 x 512 18.4 -> 14.9, x 1024 28.7 -> 21.5, 8 / 2 x 4096 84.7 -> 58.4.  Up to 512 blocks (two items a
// workgroup) few, long heads still gain: 8 / 2 x 8192 198 -> 169, 4 / 1 x 16384 343 -> 278; many short ones do not on every input (32 / 8 x
// 2048 99.6 -> 97.5, concentrated 86.4 -> 88.9).  With 560 blocks and more pairs are better everywhere (32 / 8 x 2560 116 -> 128).
constexpr int SINGLE_BLOCK_ITEMS = 384;
constexpr int SINGLE_FEW_HEADS = 512;
// Limits of the dealt ticket orders (plan_ranges), near-uniform passes, head by head -> dealt.
// Items a head up to which whole heads are dealt whatever their lists: 2 x 28 / 4 heads, 32 items 859 -> 827 us, 40 1221 -> 1204, 44 1459 ->
// 1437, 48 1703 -> 1687, 56 2234 -> 2231, 64 2822 -> 2845; 32 / 8, 40 items 745 -> 729, 44 869 -> 846, 48 994 -> 978, 52 1142 -> 1138, 64 1639 -> 1642; 16 / 16 equal
// from 32 to 64.  Above 44 the lists decide (DEAL_BY_LISTS).
constexpr int DEAL_ROW = 44;
// Items of a launch of other head counts: 28 / 4 heads, 1176 items 750 -> 700 us, 1400 989 -> 949, 1596 1258 -> 1213, 1988 1829 -> 1794, 2576 2833 -> 2916;
// 12 / 4, 1392 2144 -> 1988, 1992 4048 -> 3927, 2592 6319 -> 6474.  (The gain ends between 2000 and 2600.)
constexpr int DEAL_ITEMS = 1400;
// A sequence inside one segment with more single blocks than workgroups would need the list kernel besides (see pbs_sparse_attn_launch): only from
// ONE_SEGMENT_ROW blocks a row on (128 heads x 295 tokens 29 against 40 us, 32 heads x 1536 38.9 against 37.0).
constexpr int ONE_SEGMENT_ROW = 12, ITEMS_WITHOUT_LISTS = 256;
static int item_span(int rows, int nb, int bps) {
  const int64_t blocks = (int64_t)rows * nb;
  if (blocks > (rows <= 16 ? SINGLE_FEW_HEADS : SINGLE_BLOCK_ITEMS)) return 2;
  return bps < nb || blocks <= ITEMS_WITHOUT_LISTS || nb >= ONE_SEGMENT_ROW ? 1 : 2;
}
static int items_of(int nb, int span) { return (nb + span - 1) / span; }

// workspace: 256 bytes of work counters, then one merged visit list per item.  Room for the lists of every call of fewer heads, a shorter
// sequence or a shorter segment as well, whose items may be single blocks: callers make one workspace for their largest call, and
// pbs_sparse_attn_fwd is not told its size.

extern "C" size_t pbs_sparse_attn_workspace_bytes(int B, int Hq, int S, int segment_size) {
  const int64_t rows = (int64_t)B * Hq, nb = (S + BS - 1) / BS, cap = list_cap((int)nb, segment_size / BS);
  static_assert(SINGLE_BLOCK_ITEMS <= SINGLE_FEW_HEADS, "the most single-block items of a launch");
  const int64_t lists = std::max<int64_t>(rows * items_of((int)nb, 2), std::min<int64_t>(rows * nb, SINGLE_FEW_HEADS));
  return 256 + (size_t)lists * cap * 2;
}

extern "C" int pbs_sparse_attn_fwd(const void* q, const void* perm_k, const void* perm_vt, const void* k, const void* v,
                                   const int32_t* csr_cols, const int32_t* csr_cnt, void* out, int B, int Hq, int Hkv, int S,
                                   int head_dim, int block_size, int segment_size, int64_t q_sb, int64_t q_sh, int64_t q_ss,
                                   int64_t k_sb, int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss,
                                   int64_t o_sb, int64_t o_sh, int64_t o_ss, float softmax_scale, void* workspace, void* stream) {
  PBS_REQUIRE(csr_cols && csr_cnt, "pbs_sparse_attn_fwd: null tensor pointer");
  return pbs_sparse_attn_launch(q, perm_k, perm_vt, k, v, csr_cols, csr_cnt, false, out, B, Hq, Hkv, S, head_dim, block_size, segment_size,
                            q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss, softmax_scale, nullptr,
                            workspace, stream);
}

extern "C" int pbs_sparse_attn_fwd_optional_diagonal(const void* q, const void* perm_k, const void* perm_vt, const void* k,
                                                     const void* v, const int32_t* csr_cols, const int32_t* csr_cnt,
                                                     const uint8_t* own_block_needed, void* out, int B, int Hq, int Hkv, int S,
                                                     int head_dim, int block_size, int64_t q_sb, int64_t q_sh, int64_t q_ss,
                                                     int64_t k_sb, int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh,
                                                     int64_t v_ss, int64_t o_sb, int64_t o_sh, int64_t o_ss, float softmax_scale,
                                                     void* workspace, void* stream) {
  PBS_REQUIRE(own_block_needed, "pbs_sparse_attn_fwd_optional_diagonal: null own_block_needed");
  PBS_REQUIRE(csr_cols && csr_cnt, "pbs_sparse_attn_fwd: null tensor pointer");
  return pbs_sparse_attn_launch(q, perm_k, perm_vt, k, v, csr_cols, csr_cnt, false, out, B, Hq, Hkv, S, head_dim, block_size, block_size,
                            q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss, softmax_scale,
                            own_block_needed, workspace, stream);
}

// the eight ranges of work items (AttnArgs::xcd_start) and the ticket order; returns the items of the longest range
static int plan_ranges(AttnArgs& a) {
  // eight ranges of equal estimated work: item p of a head costs about p + 1 (causal length)
  a.span = item_span(a.BH, a.nb, a.bps);
  const int64_t n = a.deal.n = items_of(a.nb, a.span);
  const double head_work = 0.5 * (double)n * (double)(n + 1);
  int max_items = 0;
  for (int x = 0; x <= 8; ++x) {
    const double target = head_work * a.BH * x / 8.0;
    int64_t head = (int64_t)(target / head_work);
    if (head > a.BH) head = a.BH;
    const double rem = target - head * head_work;
    // items of a head in launch order are n - 1, n - 2, ...: the first i of them cost
    // i * n - i (i - 1) / 2
    int64_t lo = 0, hi = n;
    while (lo < hi) {
      const int64_t mid = (lo + hi) / 2;
      if ((double)mid * n - 0.5 * (double)mid * (mid - 1) >= rem - 1e-6) hi = mid; else lo = mid + 1;
    }
    int64_t start = head * n + (head < a.BH ? lo : 0);
    if (x == 8) start = (int64_t)a.BH * n;
    a.xcd_start[x] = (int)start;
    if (x > 0) max_items = std::max(max_items, a.xcd_start[x] - a.xcd_start[x - 1]);
  }
  // Few items a head: longest first (see ticket_item; also at an item a workgroup, since the workgroups start one after the other).  With
  // more of them the head-by-head order balances well enough, and where attention is near-uniform it is faster by what an XCD's workgroups share of a head in L2: 32 / 8
  // heads x 16384 1616 against 1644 us, x 32768 5.78 against 6.00 ms; 16 / 16 x 22016 1427 against 1435.
  const int64_t total = (int64_t)a.BH * n;
  const bool whole_heads = a.BH % 8 == 0;
  a.deal.how = whole_heads ? (a.BH == 8 ? DEAL_NONE : n <= DEAL_ROW ? DEAL_GROUPS : DEAL_BY_LISTS) : total <= DEAL_ITEMS ? DEAL_ALL : DEAL_NONE;
  a.deal.heads = !whole_heads ? a.BH : total <= 2 * 256 ? a.BH / 8 : DEAL_HEADS;
  const int64_t group = a.deal.heads * n;
  // (divisors of 1 are not used) quotients are exact below 2^32 / divisor
  a.deal.group_magic = (uint32_t)((1ull << 32) / group + 1);
  a.deal.heads_magic = (uint32_t)((1ull << 32) / a.deal.heads + 1);
  if (total / 8 >= (1ll << 32) / group) a.deal.how = DEAL_NONE;
  if (a.deal.how != DEAL_NONE) {
    max_items = 0;
    for (int x = 0; x <= 8; ++x) {
      a.xcd_start[x] = whole_heads ? (int)(x * total / 8) : (int)(x * (total / 8) + std::min<int64_t>(x, total % 8));   // (DEAL_ALL: items 8 t + x < total)
      if (x > 0) max_items = std::max(max_items, a.xcd_start[x] - a.xcd_start[x - 1]);
    }
  }
  return max_items;
}

// one workgroup per CU (the kernel's LDS leaves room for one), a multiple of 8 so that every XCD gets its share; fewer when
// there are fewer items.  The CU count is looked up once per device.
static int64_t workgroups(int max_items) {
  int dev = 0;
  const bool tracked = hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64;
  int n_cu = tracked ? g_cu_count[dev].load(std::memory_order_relaxed) : 0;
  if (n_cu <= 0) {
    if (hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n_cu <= 0) n_cu = 256;
    if (tracked) g_cu_count[dev].store(n_cu, std::memory_order_relaxed);
  }
  return std::min<int64_t>((int64_t)8 * max_items, (int64_t)(n_cu + 7) / 8 * 8);
}

bool pbs_sparse_attn_forms_lists(int B, int Hq, int S, int block_size) {
  AttnArgs a;
  a.BH = B * Hq;
  a.nb = (S + block_size - 1) / block_size;
  a.bps = a.nb;
  if ((int64_t)a.BH * a.nb > 4 * 256) return false;   // (two blocks an item, 256 workgroups or fewer)
  const int max_items = plan_ranges(a);
  return max_items <= workgroups(max_items) / 8;
}

PairLists pbs_pair_lists(int B, int Hq, int Hkv, int S, int block_size, int segment_size, void* workspace) {
  AttnArgs a;
  a.BH = B * Hq;
  a.nb = (S + block_size - 1) / block_size;
  a.bps = segment_size / block_size;
  PairLists l;
  l.plist = (uint16_t*)((char*)workspace + 256);
  l.queue = (int*)workspace;
  l.cap = list_cap(a.nb, segment_size / block_size);
  l.Hq = Hq;
  l.group = Hq / Hkv;
  l.first_tickets = (int)(workgroups(plan_ranges(a)) / 8);
  l.span = a.span;
  return l;
}

int pbs_sparse_attn_launch(const void* q, const void* perm_k, const void* perm_vt, const void* k, const void* v,
                              const int32_t* csr_cols, const int32_t* csr_cnt, bool lists_built, void* out, int B, int Hq, int Hkv, int S,
                              int head_dim, int block_size, int segment_size, int64_t q_sb, int64_t q_sh, int64_t q_ss,
                              int64_t k_sb, int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss, int64_t o_sb,
                              int64_t o_sh, int64_t o_ss, float softmax_scale, const uint8_t* own_block_needed, void* workspace,
                              void* stream) {
  PBS_REQUIRE(q && perm_k && perm_vt && k && v && out, "pbs_sparse_attn_fwd: null tensor pointer");
  PBS_REQUIRE(((uintptr_t)workspace % 256) == 0, "pbs_sparse_attn_fwd: workspace must be a 256-byte aligned device buffer of pbs_sparse_attn_workspace_bytes()");
  PBS_REQUIRE(head_dim == D && block_size == BS, "pbs_sparse_attn_fwd: head_dim and block_size must be 128 (got %d, %d)", head_dim, block_size);
  PBS_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && S > 0, "pbs_sparse_attn_fwd: bad shape");
  PBS_REQUIRE(segment_size > 0 && segment_size % block_size == 0, "pbs_sparse_attn_fwd: segment_size must be a multiple of block_size");
  PBS_REQUIRE(segment_size / block_size <= 511, "pbs_sparse_attn_fwd: more than 511 blocks per segment");
  PBS_REQUIRE(q_sb % 8 == 0 && q_sh % 8 == 0 && q_ss % 8 == 0 && o_sb % 8 == 0 && o_sh % 8 == 0 && o_ss % 8 == 0 &&
                  k_sb % 8 == 0 && k_sh % 8 == 0 && k_ss % 8 == 0 && v_sb % 8 == 0 && v_sh % 8 == 0 && v_ss % 8 == 0,
              "pbs_sparse_attn_fwd: strides must keep rows 16-byte aligned");
  PBS_REQUIRE(k_ss >= D && k_ss < (1 << 22), "pbs_sparse_attn_fwd: key row stride %lld outside [128, 2^22)", (long long)k_ss);
  PBS_REQUIRE(v_ss >= D && v_ss < (1 << 22), "pbs_sparse_attn_fwd: value row stride %lld outside [128, 2^22)", (long long)v_ss);
  PBS_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)out % 16) == 0 && ((uintptr_t)perm_k % 16) == 0 &&
                  ((uintptr_t)perm_vt % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)v % 16) == 0,
              "pbs_sparse_attn_fwd: pointers must be 16-byte aligned");
  AttnArgs a;
  a.q = (const uint16_t*)q; a.pk = (const uint16_t*)perm_k; a.pvt = (const uint16_t*)perm_vt;
  a.k = (const uint16_t*)k; a.v = (const uint16_t*)v;
  a.o = (uint16_t*)out;
  a.BH = B * Hq; a.Hq = Hq; a.Hkv = Hkv; a.S = S; a.nb = (S + BS - 1) / BS; a.bps = segment_size / block_size;
  a.q_sb = q_sb; a.q_sh = q_sh; a.q_ss = q_ss; a.k_sb = k_sb; a.k_sh = k_sh; a.k_ss = (uint32_t)k_ss; a.v_sb = v_sb; a.v_sh = v_sh; a.v_ss = (uint32_t)v_ss; a.o_sb = o_sb; a.o_sh = o_sh; a.o_ss = o_ss;
  a.scale_log2 = softmax_scale * 1.4426950408889634f;
  PBS_REQUIRE(a.nb <= 4096, "pbs_sparse_attn_fwd: more than 4096 blocks per sequence (%d)", a.nb);
  PBS_REQUIRE((int64_t)a.BH * ((a.nb + 1) / 2) < (1ll << 28) && B < 65536 && Hq < 65536, "pbs_sparse_attn_fwd: launch too large");
  // A sequence of one block needs no list and has a kernel of its own, which is faster for any number of heads (launches in a graph, this kernel ->
  // that one, us: 32 / 8 heads x 77 9.6 -> 4.7, x 128 10.5 -> 6.0, 28 / 4 x 33 8.7 -> 3.8, 16 x 32 / 8 x 128 28.7 -> 20.8, 256 x 32 / 8 x 128 333 -> 258).
  if (a.nb == 1 && !lists_built && !csr_cols && !own_block_needed)
    return pbs_one_block_attn_launch(OneBlockArgs{a.q, a.k, a.v, a.o, q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss, S, 0,
                                                  a.scale_log2}, B, Hq, Hkv, stream);
  const int max_items = plan_ranges(a);
  a.cap = list_cap(a.nb, a.bps);
  PBS_REQUIRE((uint32_t)a.cap * 2 <= LIST_BYTES, "pbs_sparse_attn_fwd: visit list too long");
  a.queue = (int*)workspace;
  a.plist = (const uint16_t*)((char*)workspace + 256);
  const int64_t n_wg = workgroups(max_items);
  // A sequence inside one segment with an item or less per workgroup: the attention kernel forms the lists itself (77 tokens, 32 / 8
  // heads: 19.9 -> 17.1 us when this came in, one launch instead of two) and needs no workspace.
  const bool own_lists = !lists_built && !csr_cols && !own_block_needed && a.bps >= a.nb && max_items <= n_wg / 8;
  PBS_REQUIRE(workspace || own_lists, "pbs_sparse_attn_fwd: workspace must be a 256-byte aligned device buffer of pbs_sparse_attn_workspace_bytes()");
  int dev = 0;
  hipError_t attr = hipGetDevice(&dev);
  const bool tracked = attr == hipSuccess && dev >= 0 && dev < 64;
  // the kernel's dynamic LDS size is raised once per device, not per call
  if (attr == hipSuccess && !(tracked && (g_lds_reserved.load(std::memory_order_acquire) >> dev & 1))) {
    if (const int rc = pbs_require_no_static_lds((const void*)sparse_attn_kernel, "pbs_sparse_attn_fwd")) return rc;
    attr = hipFuncSetAttribute((const void*)sparse_attn_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_TOTAL);
    if (attr == hipSuccess && tracked) g_lds_reserved.fetch_or(1ull << dev, std::memory_order_release);
  }
  if (attr != hipSuccess) {
    pbs_set_error("pbs_sparse_attn_fwd: cannot reserve %u bytes of LDS: %s", LDS_TOTAL, hipGetErrorString(attr));
    return (int)attr;
  }
  // Then nobody claims a further item, and above all nobody asks the other ranges for one before he ends, a round trip to memory behind the longest
  // item: whole pass, 28 / 4 heads x 1000 57.7 -> 55.6 us, 8 / 2 x 2000 63.2 -> 62.1, 32 / 8 x 600 43.7 -> 43.1, in one segment 32 / 8 x 256 10.3 -> 10.0.
  // (Launches without lists in memory have no counters either, and are of this kind.)
  a.one_each = max_items <= n_wg / 8;
  if (own_lists) {
    a.cap = 0;
    if (a.deal.how == DEAL_BY_LISTS) a.deal.how = DEAL_NONE;
  }
  else if (!lists_built)
    hipLaunchKernelGGL(merge_pair_lists_kernel, dim3((unsigned)(a.BH * a.deal.n)), dim3(MERGE_THREADS), 0, (hipStream_t)stream, csr_cols, csr_cnt,
                     (uint16_t*)((char*)workspace + 256), a.queue, a.nb, a.span, a.bps, a.cap, Hq, Hq / Hkv, (int)(n_wg / 8), own_block_needed);
  hipLaunchKernelGGL(sparse_attn_kernel, dim3((unsigned)n_wg), dim3(THREADS), LDS_TOTAL, (hipStream_t)stream, a);
  return pbs_check_launch("pbs_sparse_attn_fwd");
}
