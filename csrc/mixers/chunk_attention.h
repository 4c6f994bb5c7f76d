// Softmax attention of prompt chunks on the matrix cores (chunk_attention.hip): what a launch needs.
#pragma once
#include <hip/hip_runtime.h>

namespace mxs {

typedef unsigned short bf16_t;  // raw bits

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
  // or in rows (G = H): key = kx[row * x_stride + head * dn .. + dn) | kr[row * r_stride .. + dk - dn), value =
  // vx[row * x_stride + head * dv ..], row = base[s] + key position, below nrows
  const bf16_t *kx, *vx, *kr;
  long x_stride, r_stride;
  const int* base;
  int dn, nrows;
  // the walks of long tiles in nsplit stretches (rows: of the whole launch), fp32 part [rows, H, nsplit, dv + 4]; 0, 1: none
  int rows, nsplit;
  float* part;
};

// false: head sizes that no kernel holds.  max_q: an upper bound of a sequence's rows in this launch.
bool launch_chunk_attention(const ChunkArgs& a, int max_q, hipStream_t st);
// how many stretches serve a launch whose queries see `span` keys at most (0: not known)
int chunk_attention_splits(long rows, int S, int H, int G, int dk, int dv, long span);
// merges the records (maximum in log2 units, sum, two unused, output[width]) of rows: (token, head) pairs (latent_attention.hip)
bool launch_attention_combine(void* out, const float* part, long rows, int nsplit, int width, hipStream_t st);

// Single rows (row_attention.hip): dk, dv multiples of 8 up to 128, q and the cache's pieces 16-byte aligned, bs (a power of
// two) tokens a block, value rows vs apart.  nsplit stretches of the keys to a row, fp32 part [rows, H, nsplit, dv + 2] when
// there are more than one.
void launch_row_attention(const ChunkArgs& a, int rows, int bs, int vs, int nsplit, float* part, hipStream_t st);
// whether that form serves a launch whose longest chunk has max_q rows and whose rows see `span` keys at most
bool row_attention_serves(long rows, int max_q, int H, int G, long span);
// how many stretches serve rows of at most `span` visible keys
int row_attention_splits(long rows, int H, int G, long span);

// base[s]: row of key position 0 of sequence s when the keys its chunk sees (with window > 0: from the page of the first
// query's oldest one) lie back to back, offs[s]: its first row; offs[S]: rows in all.
void launch_latent_plan(int* base, int* offs, const int* qsl, const int* seq_lens, int S, int window, hipStream_t st);
// those rows of dk entries from pages of 16 at koff of a block, 16-byte pieces; at most n rows are written
void launch_latent_rows(bf16_t* out, const bf16_t* cache, long block_stride, const int* block_tables, int bt_stride,
                        const int* base, const int* offs, int S, int n, int koff, int dk, hipStream_t st);

}  // namespace mxs
