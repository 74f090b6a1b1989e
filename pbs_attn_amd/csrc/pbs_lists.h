// Merged visit lists of the pairs of query blocks: their layout, shared by the kernels that write them (the block
// selection, or the merge of two CSR rows) and the attention kernel that reads them.
#pragma once
#include "pbs_common.h"

constexpr int LIST_HEADER = 8;              // uint16 entries in front of a row's tiles: [0] number of tiles, [1] batch, [2] query head,
                                            // [3] KV head, [4] first query block of the item, [5] how many (two, or one)
constexpr uint32_t ENT_KB = 0x1fffu;        // visit-list entry: key block ...
constexpr uint32_t ENT_ORIG = 0x2000u;      // ... | tile of the un-permuted K / V (own segment) | use bits 14, 15

// Where the lists go: row `bh * n + (n - 1 - item)` of `plist` for the n items of a head, `span` query blocks each (the last one
// may have fewer), `cap` entries a row, and the attention kernel's eight
// work counters, which start at `first_tickets`.
struct PairLists {
  uint16_t* plist;
  int* queue;
  int cap, Hq, group, first_tickets, span;   // group: query heads per KV head
};
// of the lists that pbs_sparse_attn_launch expects in `workspace` with lists_built set
PairLists pbs_pair_lists(int B, int Hq, int Hkv, int S, int block_size, int segment_size, void* workspace);

// Whether the launch below forms the lists of a sequence inside one segment by itself, and then needs no workspace
bool pbs_sparse_attn_forms_lists(int B, int Hq, int S, int block_size);

// pbs_sparse_attn_fwd (and its optional-diagonal form, with own_block_needed) after their null checks.  lists_built: the
// visit lists and counters are in the workspace already.  Otherwise they are merged from the CSR rows or, with csr_cols
// null (csr_cnt is not read), hold every block of every earlier segment.
int pbs_sparse_attn_launch(const void* q, const void* perm_k, const void* perm_vt, const void* k, const void* v,
                           const int32_t* csr_cols, const int32_t* csr_cnt, bool lists_built, void* out, int B, int Hq, int Hkv, int S,
                           int head_dim, int block_size, int segment_size, int64_t q_sb, int64_t q_sh, int64_t q_ss,
                           int64_t k_sb, int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss, int64_t o_sb,
                           int64_t o_sh, int64_t o_ss, float softmax_scale, const uint8_t* own_block_needed, void* workspace,
                           void* stream);

// The selection of pbs_select_blocks for rows of block probabilities that are non-zero in the candidates of `rule` only, up to
// PBS_PAIR_SELECT_MAX_BLOCKS blocks, straight into the merged lists.  EARLIER_SEGMENTS: the blocks of earlier segments are candidates,
// permuted tiles, and the own segment comes besides.  UP_TO_DIAGONAL: every block up to the diagonal one is, all of them tiles of the
// un-permuted K and V, the diagonal one always visited.  force_first: so is the block that holds original key 0, first_blk[row] or,
// with first_blk null, block 0.
constexpr int PBS_PAIR_SELECT_MAX_BLOCKS = 2048;
enum class Candidates { EARLIER_SEGMENTS = 1, UP_TO_DIAGONAL = 2 };   // candidate_rule of pbs_select_blocks
int pbs_select_pair_lists(const float* block_attn_scores, Candidates rule, const float* threshold_per_row, float threshold, bool force_first,
                          const int32_t* first_blk, int rows, int S, int block_size, int segment_size, uint8_t* block_needed, const PairLists& lists,
                          void* stream);
// pbs_block_logits_softmax and that selection in one launch, for rows of up to PBS_ESTIMATE_SELECT_MAX_BLOCKS blocks
constexpr int PBS_ESTIMATE_SELECT_MAX_BLOCKS = 64;
int pbs_estimate_select_pair_lists(const void* pooled_q, const void* pooled_k, Candidates rule, const float* threshold_per_row,
                                   float threshold, bool force_first, const int32_t* first_blk, int rows, int S, int head_dim, int block_size, int segment_size,
                                   uint8_t* block_needed, const PairLists& lists, void* stream);
// A pooling of query blocks (pbs_pool_q): all of it is a workgroup of 256 threads per block, so that it can ride in another launch
struct PoolQ {
  const uint16_t* q;
  uint16_t* pooled_q;
  int64_t q_sb, q_sh, q_ss;
  int pool_max, Hq, S, nb;   // nb 0: none
};
// pbs_segment_argsort; first_blk, if not null, receives per row the block of `block_size` that holds original key 0 (there has
// to be a complete segment).  `ride`: a query pooling in the same launch, of which the sort by waves alone can take one
int pbs_segment_argsort_launch(const float* scores, int32_t* key_indices, int32_t* first_blk, int block_size, int rows, int S,
                               int S_pad, int segment_size, void* stream, const PoolQ& ride = {});
bool pbs_segment_argsort_takes_ride(int segment_size);
// pbs_score_keys_workspace_bytes of this sequence or of any shorter one (which may be cut into more chunks), the largest
size_t pbs_score_keys_workspace_bound(int B, int Hq, int Hkv, int S, int segment_size);
// pbs_score_keys and pbs_segment_argsort_launch in one: the final scoring pass of short sequences of short segments sorts.  Where it can,
// the keys that a workgroup of it would take if it did not (it then takes a segment); else 0.
int pbs_score_sort_chunk(int B, int Hq, int Hkv, int S, int segment_size);
int pbs_score_sort_launch(const void* q, const void* k, int32_t* key_indices, int32_t* first_blk, int B, int Hq, int Hkv, int S, int S_pad,
                          int head_dim, int block_size, int segment_size, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t k_sb,
                          int64_t k_sh, int64_t k_ss, void* workspace, size_t workspace_bytes, void* stream);
// pbs_block_logits_softmax_causal without the entries that are no candidates
int pbs_block_logits_softmax_causal_candidates(const void* pooled_q, const void* pooled_k, float* block_attn_scores, int rows, int nb,
                                               int head_dim, void* stream);
// pbs_pool_blocks; key_indices null: every key in its own place
int pbs_pool_blocks_launch(const void* q, const void* k, const int32_t* key_indices, void* pooled_q, void* pooled_k,
                           uint8_t* block_needed, int B, int Hq, int Hkv, int S, int head_dim, int block_size,
                           int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t k_sb, int64_t k_sh, int64_t k_ss,
                           int query_pool_max, int key_pool_max, void* stream);
// Scores of the keys of the complete segments (rows, Sc), for a launch that sorts them; first_blk as in pbs_segment_argsort_launch
struct SegmentScores {
  const float* scores;   // null: none
  int32_t* first_blk;
  int Sc, seg;
};
constexpr int PBS_SORT_IN_GATHER_KEYS = 1024, PBS_RANKED_KEYS = 256;   // (up to the latter a workgroup ranks them)
// The sorting workgroups of that launch on the shader engine that gets the most of them, where a row's first `sorted_blocks` blocks are sorted
// (the launch goes round the eight XCDs, and inside one round its four engines)
int pbs_sorts_of_an_engine(int B, int Hq, int Hkv, int nb, int sorted_blocks);
// pbs_pool_blocks and an unfiltered pbs_gather_kv in one launch (the pooled key blocks have the bits of both), by key_indices or, for
// segments of up to PBS_SORT_IN_GATHER_KEYS keys, by the order of `scores`
int pbs_gather_pool_launch(const void* q, const void* k, const void* v, const int32_t* key_indices, void* pooled_q, void* pooled_k,
                           void* perm_k, void* perm_vt, int B, int Hq, int Hkv, int S, int head_dim, int block_size, int64_t q_sb,
                           int64_t q_sh, int64_t q_ss, int64_t k_sb, int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss,
                           int query_pool_max, int key_pool_max, void* stream, const SegmentScores& scores = {});
