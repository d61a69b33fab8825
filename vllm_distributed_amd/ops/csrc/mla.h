// Arguments shared by the latent-attention kernels (mla.hip, mla_tile.hip).
#pragma once
#include "common.h"

struct MlaParams {
  const void* q;            // [T, H, DK]: absorbed q_nope followed by rotated q_pe
  const void* kc;
  const void* vt;
  void* out;                // [T, H, DV] latent-space output
  float* part_out;          // [T, H, nsplit, DV]
  float* part_lse;          // [T, H, nsplit] (log2 domain)
  const int* block_table;
  const int* seq_lens;
  const int* q_start_loc;
  int H, BS, max_blocks, nsplit;
  long q_stride, out_stride;
  float scale;              // softmax scale, times the cache scale for an fp8 cache
  float v_scale;            // 1, or the cache scale for an fp8 cache
  int window;               // > 0: a query at position i sees the keys j with 0 <= i - j < window
  const float* sink;        // [H] or null: exp(sink[h]) joins head h's softmax denominator, with no key and no value
  int cuts;                 // key pieces of each column block that fill the chip, if all are alike (mla_tile.hip)
  int num_seqs;             // (mla_tile.hip)
  int levels;               // workgroups are numbered by column block (1) or piece (2), then sequence (mla_tile.hip)
  int wave_cols;            // 1: every wave takes 16 columns of its own over all keys (prompts: neighbouring tokens
                            //    walk the same keys at the same time, so the rows come from the cache near the CU);
                            // 0: the 4 waves share 16 columns and split the keys (few query tokens)
};

// mla_tile.hip: caches of 576-value rows (16 bits or e4m3) in pages of a power of two tokens, 16 at least
struct MlaTilePlan {
  int groups;               // column groups of 32 per workgroup: 4, or 1 (the waves then share the 32 columns)
  int blocks;               // workgroups over the columns of one sequence
  int nsplit;               // pieces that a column block's keys can be cut into
  int cuts;                 // pieces of each that fill the chip, if all are alike
  long items;               // column blocks of the whole batch, at most
  int levels;               // 1: sequences of about one length, several column blocks each; 2: a few of one block each; 0: by their lengths
};
MlaTilePlan mla_tile_plan(int S, int T_tokens, int H, int BS, int max_blocks, int max_q);
int mla_tile_launch(const MlaParams& p, const MlaTilePlan& plan, int S, int dtype, bool f8, hipStream_t st);
