// Softmax attention of prompt chunks on the matrix cores (chunk_attention.hip): what a launch needs.
#pragma once
#include "mix_common.h"

namespace mxs {

struct ChunkArgs {
  bf16_t* out;  // [rows, H * dv]
  const bf16_t* q;  // rows of H * dk, q_stride apart, 8-byte aligned
  long q_stride;
  const int* qsl;       // [S + 1] first row of every sequence
  const int* seq_lens;  // [S] tokens in the cache, this step's among them
  int S, H, G, dk, dv;  // query heads, kv heads, head sizes (multiples of 16)
  float scale;
  int window, keep;    // position i sees j <= i when i - j < window or j < keep (window <= 0: every j <= i)
  const float* sink;   // [H] or null: one more score per head, without a value
  // keys and values in pages of 16 tokens: [G][16][dk] at koff, [G][16][dv] at voff of a block
  const bf16_t* cache;
  long block_stride;
  const int* block_tables;
  int bt_stride, koff, voff;
  // or in rows: key = kx[row * x_stride + head * 128 .. + 128) | kr[row * r_stride .. + dk - 128), value =
  // vx[row * x_stride + head * dv ..], row = base[s] + key position
  const bf16_t *kx, *vx, *kr;
  long x_stride, r_stride;
  const int* base;
};

// false: head sizes that no kernel holds.  max_q: an upper bound of a sequence's rows in this launch.
bool launch_chunk_attention(const ChunkArgs& a, int max_q, hipStream_t st);

}  // namespace mxs
