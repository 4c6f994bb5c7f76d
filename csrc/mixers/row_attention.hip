// Softmax attention of single rows (decoded tokens, chunks of a few rows) over the paged cache on the matrix cores
// (gfx950): bf16 queries, keys and values, head sizes up to 128, fp32 scores, weights and sums.
//
// A workgroup serves one row and up to 16 query heads of one kv head; its eight waves walk 32 keys at a time, each on its
// own, every eighth tile (and with `nsplit` stretches every nsplit * 8th), and are merged at the end.  No barrier stands in
// the walk: keys go from memory to the registers in the layout of the product, values through an LDS tile of the wave's own.
//   S = K Q^T      (v_mfma_f32_16x16x32_bf16) A = 16 keys, a lane's 8 entries are 16 bytes of a key row; columns = heads
//   O^T += V^T P^T A = V^T by the transposing LDS read, B = P as the accumulator leaves it, in three bf16 pieces: all 24 bits
//                  of the fp32 weight
// The next tile's keys and values and the page of the one after are in flight under a tile's products.  Bound by the cached
// bytes: 64 rows at 2,050 keys, 8 kv heads of 64, 32 heads: 208 -> 44.5 us (268 MB, 6.0 TB/s); 4 kv heads: 189 -> 25 us.  The form
// that it took these calls from scores with 8 lanes a key and 8 vector operations an entry and head (a workgroup holds 4 or 8
// heads whatever the group has) and has its waves wait for each other five times in 256 keys.
// A wave holds 4 tiles of 16 columns at most for its heads however few they are: with one head to a kv head the 32 products
// of a tile are still under the time of its bytes: 16 heads of 64 over 16: 182 -> 102 us.
#include "chunk_attention.h"
#include "mix_common.h"

#include <algorithm>

namespace mxs {

typedef __bf16 b8_t __attribute__((ext_vector_type(8)));
typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
typedef short s4_t __attribute__((ext_vector_type(4)));
typedef float f2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));

// Waves: eight with 64 entries a head; four with 128, where a wave's tile and registers are twice as large.
template <int DP> constexpr int kRowWaves = DP == 64 ? 8 : 4;

template <int DP>
__global__ void __launch_bounds__(64 * kRowWaves<DP>, DP == 64 ? 4 : 3) row_attention_kernel(ChunkArgs a, int hsplit, int shift, int vs, int nsplit,
                                                                          float* __restrict__ part) {
  constexpr int NW = kRowWaves<DP>;
  constexpr int KS = DP / 32, DT = DP / 16, VROW = DP + 8, NV = DP / 16;  // 16-byte value pieces a lane stages
  __shared__ __attribute__((aligned(16))) bf16_t lds[NW][32 * VROW];
  __shared__ float ms[NW][16], ls[NW][16];
  const int t = blockIdx.x, z = blockIdx.z;
  const int g = blockIdx.y / hsplit, hs = blockIdx.y - g * hsplit;
  const int R = a.H / a.G, h0 = g * R + hs * 16, nr = min(16, R - hs * 16);
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, c = lane & 15, qd = lane >> 4;
  const int dk = a.dk, dv = a.dv;
  const int s = seq_of_row(a.qsl, a.S, t);
  const int qlen = a.qsl[s + 1] - a.qsl[s], bs = 1 << shift;
  const int pos = min(max(a.seq_lens[s] - qlen + (t - a.qsl[s]), 0), a.bt_stride * bs - 1);
  const int lo = a.window > 0 ? max(pos - a.window + 1, 0) : 0;
  const int nA = a.window > 0 ? min(a.keep, lo) : 0;  // kept first tokens below the window
  const int nvis = nA + (pos - lo + 1);
  const int* bt = a.block_tables + static_cast<long>(s) * a.bt_stride;
  const bf16_t* kbase = a.cache + a.koff + static_cast<long>(g) * bs * dk;
  const bf16_t* vbase = a.cache + a.voff + static_cast<long>(g) * bs * vs;
  auto key_of = [&](int n) { n = min(n, nvis - 1); return n < nA ? n : lo + (n - nA); };

  b8_t qf[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    const int d = 32 * k + 8 * qd;
    uint4 raw = make_uint4(0, 0, 0, 0);
    if (c < nr && d < dk) raw = *reinterpret_cast<const uint4*>(a.q + static_cast<long>(t) * a.q_stride + (h0 + c) * dk + d);
    qf[k] = __builtin_bit_cast(b8_t, raw);
  }
  const int step = NW * nsplit * 32;
  int n0 = (z * NW + wid) * 32;
  uint4 kr[2][KS], vr[NV];
  int blk = 0;  // the block of key (lane % 32) of the tile to be fetched next
  auto fetch_blocks = [&](int n) { blk = bt[key_of(n + (lane & 31)) >> shift]; };
  auto fetch_keys = [&](int n) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bf16_t* p = kbase + static_cast<long>(__shfl(blk, 16 * u + c, 64)) * a.block_stride + (key_of(n + 16 * u + c) & (bs - 1)) * dk;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const int d = 32 * k + 8 * qd;
        kr[u][k] = make_uint4(0, 0, 0, 0);
        if (d < dk) kr[u][k] = *reinterpret_cast<const uint4*>(p + d);
      }
    }
  };
  constexpr int VP = DP / 8;  // lanes to a value row
  const int vrow = lane / VP, vcol = 8 * (lane % VP);
  auto fetch_values = [&](int n) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int r = vrow + i * (64 / VP);
      const int b = __shfl(blk, r, 64);  // every lane takes part in the exchange
      vr[i] = make_uint4(0, 0, 0, 0);
      if (vcol < dv && n + r < nvis)  // keys past the last: zeros
        vr[i] = *reinterpret_cast<const uint4*>(vbase + static_cast<long>(b) * a.block_stride + (key_of(n + r) & (bs - 1)) * vs + vcol);
    }
  };
  const float sinkv = a.sink && c < nr ? a.sink[h0 + c] : -INFINITY;
  float m = sinkv, l = 0.f;  // l: of this lane's keys
  f4_t acc[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) acc[i] = f4_t{0.f, 0.f, 0.f, 0.f};
  bf16_t* vt = lds[wid];
  if (n0 < nvis) {
    fetch_blocks(n0);
    fetch_keys(n0);
    fetch_values(n0);
    fetch_blocks(n0 + step);
  }
  for (; n0 < nvis; n0 += step) {
    f4_t sc[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      sc[u] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KS; ++k) sc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8_t, kr[u][k]), qf[k], sc[u], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) *reinterpret_cast<uint4*>(vt + (vrow + i * (64 / VP)) * VROW + vcol) = vr[i];
    const bool more = n0 + step < nvis;
    if (more) {
      fetch_keys(n0 + step);
      fetch_values(n0 + step);
      fetch_blocks(n0 + 2 * step);
    }
    float x[8], mx = m;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[4 * u + r] = n0 + 16 * u + 4 * qd + r < nvis ? sc[u][r] * a.scale : -INFINITY;
        mx = fmaxf(mx, x[4 * u + r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (__any(mx > m)) {
      const float corr = mx > m ? expf(m - mx) : 1.f;  // the first tile: exp(-inf) = 0
      l *= corr;
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] *= corr;
      m = mx;
    }
    b8_t p[3];
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      f2_t w;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        w[e] = n0 + 16 * (j / 4) + 4 * qd + j % 4 + e < nvis ? expf(x[j + e] - m) : 0.f;
        l += w[e];
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const b2_t h = __builtin_convertvector(w, b2_t);
        p[k][j] = h[0];
        p[k][j + 1] = h[1];
        const unsigned hb = __builtin_bit_cast(unsigned, h);
        w[0] -= bf2f_lo(hb);
        w[1] -= bf2f_hi(hb);
      }
    }
    wave_sync();
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      const bf16_t* at = vt + (4 * qd + (c >> 2)) * VROW + 16 * i + 4 * (c & 3);
      typedef __attribute__((address_space(3))) s4_t* lp;
      const s4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(at));
      const s4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(at + 16 * VROW));
      const b8_t vf = __builtin_bit_cast(b8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
      for (int k = 2; k >= 0; --k) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, p[k], acc[i], 0, 0, 0);
    }
    wave_sync();  // the tile is rewritten by the next round
  }

  // merge: the waves' sums lie head by head where their value tiles were
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  float* ow = reinterpret_cast<float*>(vt);  // [16][DP + 4]
  static_assert(16 * (DP + 4) * 4 <= 32 * VROW * 2, "the sums fit the tile");
#pragma unroll
  for (int i = 0; i < DT; ++i) *reinterpret_cast<f4_t*>(ow + c * (DP + 4) + 16 * i + 4 * qd) = acc[i];
  if (qd == 0) {
    ms[wid][c] = m;
    ls[wid][c] = l;
  }
  __syncthreads();
  for (int idx = tid; idx < nr * DP; idx += 64 * NW) {
    const int r = idx / DP, d = idx - r * DP;
    if (d >= dv) continue;
    float M = ms[0][r];
#pragma unroll
    for (int w = 1; w < NW; ++w) M = fmaxf(M, ms[w][r]);
    float L = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = ms[w][r] == M ? 1.f : expf(ms[w][r] - M);  // M = -inf: a stretch without keys, sums of zero
      L += f * ls[w][r];
      o += f * reinterpret_cast<const float*>(lds[w])[r * (DP + 4) + d];
    }
    const long at = static_cast<long>(t) * a.H + h0 + r;
    if (nsplit > 1) {
      float* pp = part + (at * nsplit + z) * (dv + 2);
      pp[d] = o;
      if (d == 0) {
        pp[dv] = M;
        pp[dv + 1] = L;
      }
    } else {
      if (a.sink) L += expf(a.sink[h0 + r] - M);
      a.out[at * dv + d] = f2bf(o / L);
    }
  }
}

constexpr int kMaxSplits = 16;

// the stretches of a (row, head), which begin at the sink's score as well
__global__ void __launch_bounds__(128) row_attention_merge_kernel(bf16_t* __restrict__ out, const float* __restrict__ part, int H, int dv,
                                                                  int nsplit, const float* __restrict__ sink) {
  const long at = blockIdx.x;
  const float* p = part + at * nsplit * (dv + 2);
  const int d = threadIdx.x;
  if (d >= dv) return;
  float m[kMaxSplits], l[kMaxSplits], v[kMaxSplits];  // all in flight together
#pragma unroll
  for (int z = 0; z < kMaxSplits; ++z) {
    const float* pz = p + min(z, nsplit - 1) * (dv + 2);
    v[z] = pz[d];
    m[z] = pz[dv];
    l[z] = pz[dv + 1];
  }
  float M = m[0], L = 0.f, o = 0.f;
#pragma unroll
  for (int z = 1; z < kMaxSplits; ++z) M = fmaxf(M, m[z]);
#pragma unroll
  for (int z = 0; z < kMaxSplits; ++z) {
    const float f = z < nsplit ? expf(m[z] - M) : 0.f;
    if (z < nsplit) {
      L += f * l[z];
      o += f * v[z];
    }
  }
  if (sink) L += expf(sink[at % H] - M);
  out[at * dv + d] = f2bf(o / L);
}

// Stretches: where the rows leave half of the chip's units without a workgroup, as many as give each unit two and a wave one
// tile at least.  One row of 2,050 keys, 8 kv heads: 157 us in the form before (one workgroup for 4 or 8 heads), 8.8 us here;
// 16 rows: 186 -> 18.7 us.  From 128 workgroups on the merge's launch costs what the split gives.
int row_attention_splits(long rows, int H, int G, long span) {
  const long groups = rows * G * ((H / G + 15) / 16);
  if (groups == 0 || groups > 128) return 1;
  return static_cast<int>(std::max(1L, std::min({static_cast<long>(kMaxSplits), 512 / groups, span / 256})));
}

// A chunk's rows have workgroups of their own here and read their keys again, in chunk_attention.hip 128 (row, head) pairs share
// them in one that takes longer to start.  Up to 512 workgroups the rows run side by side; with more, chunks of few rows do too.
// Rows / chunks, us, 8 kv heads of 64: 4 chunks of 15 7.3 / 8.1, behind 100 keys 8.2 / 9.5, behind 600 15.8 / 20.7; 16 chunks of
// 5 9.4 / 8.2, 10.3 / 9.6, 23.4 / 20.5, behind 2,000 57 / 29; 64 chunks of 15 53 / 8.5; 64 of 2 behind 600 30.4 / 25.7.  16 rows
// and more belong to the chunks (behind 2,000 keys 16 rows of 16 heads of 128 take 33 there) but where there is nothing to walk:
// a chunk of 16 alone 6.4 / 8.1.
bool row_attention_serves(long rows, int max_q, int H, int G, long span) {
  const long groups = rows * G * ((H / G + 15) / 16);
  return max_q <= 1 || (groups < 512 && (max_q < 16 || (max_q < 32 && span <= 64)));
}

void launch_row_attention(const ChunkArgs& a, int rows, int bs, int vs, int nsplit, float* part, hipStream_t st) {
  int shift = 0;
  while ((1 << shift) < bs) ++shift;
  const int hsplit = (a.H / a.G + 15) / 16;
  const dim3 grid(rows, a.G * hsplit, nsplit);
  if (a.dk <= 64 && a.dv <= 64)
    hipLaunchKernelGGL(row_attention_kernel<64>, grid, dim3(64 * kRowWaves<64>), 0, st, a, hsplit, shift, vs, nsplit, part);
  else
    hipLaunchKernelGGL(row_attention_kernel<128>, grid, dim3(64 * kRowWaves<128>), 0, st, a, hsplit, shift, vs, nsplit, part);
  if (nsplit > 1)
    hipLaunchKernelGGL(row_attention_merge_kernel, dim3(rows * a.H), dim3(128), 0, st, a.out, part, a.H, a.dv, nsplit, a.sink);
}

}  // namespace mxs
