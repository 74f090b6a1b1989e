// Causal attention of sequences of one block (up to 128 tokens): see pbs_attn_block.hip.
#pragma once
#include "pbs_common.h"

struct OneBlockArgs {
  const uint16_t *q, *k, *v;
  uint16_t* o;
  int64_t q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss;
  int S;
  uint32_t group_magic;   // quotient of a head's number by the heads of a KV group: high word of a product (0: one head a group)
  float scale_log2;
};
// the heads of all batches, B and Hq below 65536; the arguments have been checked
int pbs_one_block_attn_launch(OneBlockArgs a, int B, int Hq, int Hkv, void* stream);
