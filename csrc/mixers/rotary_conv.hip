// Kernels around rotary attention, short causal convolutions and gated output norms (gfx950):
// scaled embedding rows into the fp32 stream, q/k head norm + rotary pairs + paged
// cache write in one launch, turning attention outputs back, the convolution with its carried
// inputs (alone, or with the query factor and the page write), and the norm of a recurrent mixer's read-out with its gate.  Activations and weights are
// bf16 or fp32; angles, norms, sums and activations are fp32 with one rounding at the store.
#include <algorithm>

#include "mix_common.h"

namespace mxs {

__device__ __forceinline__ float softplus_f(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

template <typename T>
__global__ void __launch_bounds__(256) embed_scaled_kernel(float* __restrict__ out, const int64_t* __restrict__ ids,
                                                           const T* __restrict__ table, int W, long vocab, float scale) {
  const long row = blockIdx.x;
  int64_t id = ids[row];
  id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);  // never outside the table, whatever the batch holds
  for (int c = threadIdx.x; c < W; c += blockDim.x) out[row * W + c] = ldf(table + id * W + c) * scale;
}

// One wave per (token, head): optional RMS norm over the head, interleaved rotary pairs (2i, 2i+1) on
// the first 2*nf dimensions, one store.  The grid's heads are the H query heads (rewritten in place),
// then G key heads and G value heads (into the paged cache; values have no norm and their own
// frequencies, possibly none).
template <typename T>
__global__ void __launch_bounds__(64) rope_qkv_cache_kernel(
    T* __restrict__ q, long q_stride, const T* __restrict__ k, long k_stride, const T* __restrict__ v, long v_stride,
    const int64_t* __restrict__ positions, const int64_t* __restrict__ slots, T* __restrict__ cache, long block_stride,
    int koff, int voff, int H, int G, int dk, int dv, int bs, const float* __restrict__ freqs, int nf,
    const T* __restrict__ q_norm, const T* __restrict__ k_norm, float eps, const float* __restrict__ v_freqs, int nvf) {
  const long t = blockIdx.x;
  const int hy = blockIdx.y, lane = threadIdx.x;
  const T* src;
  T* dst;
  const T* nw = nullptr;
  const float* fr = freqs;
  int dim = dk, nfr = nf;
  if (hy < H) {
    dst = q + t * q_stride + static_cast<long>(hy) * dk;
    src = dst;
    nw = q_norm;
  } else {
    const int64_t slot = slots[t];
    if (slot < 0) return;
    const long blk = slot / bs;
    const int off = static_cast<int>(slot % bs);
    if (hy < H + G) {
      const int g = hy - H;
      src = k + t * k_stride + static_cast<long>(g) * dk;
      dst = cache + blk * block_stride + koff + (static_cast<long>(g) * bs + off) * dk;
      nw = k_norm;
    } else {
      const int g = hy - H - G;
      src = v + t * v_stride + static_cast<long>(g) * dv;
      dst = cache + blk * block_stride + voff + (static_cast<long>(g) * bs + off) * dv;
      dim = dv;
      fr = v_freqs;
      nfr = nvf;
    }
  }
  float inv = 1.f;
  if (nw != nullptr) {
    float s = 0.f;
    for (int d = lane; d < dim; d += 64) { const float x = ldf(src + d); s += x * x; }
    inv = rsqrtf(wave_sum(s) / static_cast<float>(dim) + eps);
  }
  const float pos = static_cast<float>(positions[t]);
  for (int pr = lane; 2 * pr < dim; pr += 64) {
    const int d0 = 2 * pr;
    const bool two = d0 + 1 < dim;
    float a = ldf(src + d0) * inv, b = two ? ldf(src + d0 + 1) * inv : 0.f;
    if (nw != nullptr) { a *= ldf(nw + d0); if (two) b *= ldf(nw + d0 + 1); }
    if (pr < nfr) {
      float sn, cs;
      sincosf(pos * fr[pr], &sn, &cs);
      const float a2 = a * cs - b * sn;
      b = b * cs + a * sn;
      a = a2;
    }
    stf(dst + d0, a);
    if (two) stf(dst + d0 + 1, b);
  }
}

// out = scale * (x with the pairs of every head turned by sign * position * freqs); out rows may be
// a slice of a wider buffer.
template <typename T>
__global__ void __launch_bounds__(64) rope_rows_kernel(T* __restrict__ out, long out_stride, const T* __restrict__ x,
                                                       long x_stride, const int64_t* __restrict__ positions, int dim,
                                                       const float* __restrict__ freqs, int nf, float sign, float scale) {
  const long t = blockIdx.x;
  const int hd = blockIdx.y, lane = threadIdx.x;
  const T* src = x + t * x_stride + static_cast<long>(hd) * dim;
  T* dst = out + t * out_stride + static_cast<long>(hd) * dim;
  const float pos = static_cast<float>(positions[t]) * sign;
  for (int pr = lane; 2 * pr < dim; pr += 64) {
    const int d0 = 2 * pr;
    const bool two = d0 + 1 < dim;
    float a = ldf(src + d0), b = two ? ldf(src + d0 + 1) : 0.f;
    if (pr < nf) {
      float sn, cs;
      sincosf(pos * freqs[pr], &sn, &cs);
      const float a2 = a * cs - b * sn;
      b = b * cs + a * sn;
      a = a2;
    }
    stf(dst + d0, a * scale);
    if (two) stf(dst + d0 + 1, b * scale);
  }
}

// The same two for heads of whole, aligned pieces of 8 (key heads of 8 times a power of two, so that a norm is a sum over
// neighbouring lanes): a workgroup per token, which makes the token's turns once in LDS for all heads.  A wave per token
// and head turned 32 pairs on 2-byte accesses and made its sines itself.  4,096 tokens, 32 + 8 + 8 heads of 64 with
// norms: 54 -> 15.4 us; turning 32 heads back: 31 -> 8.2 us (10 and 7 us are their bytes).
template <typename T>
__device__ __forceinline__ void turn8(float* x, const float2* cs, int d, int nf) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int pr = d / 2 + i;
    if (pr < nf) {
      const float2 t = cs[pr];
      const float a = x[2 * i], b = x[2 * i + 1];
      x[2 * i] = a * t.x - b * t.y;
      x[2 * i + 1] = b * t.x + a * t.y;
    }
  }
}
__device__ __forceinline__ void make_turns(float2* cs, const float* freqs, int nf, float pos) {
  for (int i = threadIdx.x; i < nf; i += blockDim.x) {
    float sn, c;
    sincosf(pos * freqs[i], &sn, &c);
    cs[i] = make_float2(c, sn);
  }
}

template <typename T>
__global__ void __launch_bounds__(512) rope_qkv_cache_wide_kernel(
    T* __restrict__ q, long q_stride, const T* __restrict__ k, long k_stride, const T* __restrict__ v, long v_stride,
    const int64_t* __restrict__ positions, const int64_t* __restrict__ slots, T* __restrict__ cache, long block_stride,
    int koff, int voff, int H, int G, int dk, int dv, int bs, const float* __restrict__ freqs, int nf,
    const T* __restrict__ q_norm, const T* __restrict__ k_norm, float eps, const float* __restrict__ v_freqs, int nvf) {
  extern __shared__ float2 cs[];  // [nf] then [nvf]
  const long t = blockIdx.x;
  const int LP = dk / 8, nq = H * LP, nk = k ? G * LP : 0, n = nq + nk + (k ? G * dv / 8 : 0), step = blockDim.x * gridDim.y;
  int i = blockIdx.y * blockDim.x + threadIdx.x;
  float x[8];
  auto fetch = [&] {
    if (i < n) ld8f(i < nq ? q + t * q_stride + 8 * i : i < nq + nk ? k + t * k_stride + 8 * (i - nq) : v + t * v_stride + 8 * (i - nq - nk), x);
  };
  fetch();  // under way while the turns are made
  const int64_t slot = k ? slots[t] : -1;
  const float pos = static_cast<float>(positions[t]);
  make_turns(cs, freqs, nf, pos);
  make_turns(cs + nf, v_freqs, nvf, pos);
  __syncthreads();
  T* page = cache + (slot < 0 ? 0 : slot / bs) * block_stride;
  const int off = static_cast<int>(slot < 0 ? 0 : slot % bs);
  for (; i < n; i += step, fetch()) {
    if (i < nq + nk) {
      const bool isq = i < nq;
      const int j = isq ? i : i - nq, d = 8 * (j % LP), head = j / LP;
      const T* nw = isq ? q_norm : k_norm;
      if (nw) {
        float s = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) s += x[e] * x[e];
        for (int o = 1; o < LP; o <<= 1) s += __shfl_xor(s, o, 64);
        const float inv = rsqrtf(s / static_cast<float>(dk) + eps);
        float w[8];
        ld8f(nw + d, w);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = x[e] * inv * w[e];
      }
      turn8<T>(x, cs, d, nf);
      if (isq) st8f(q + t * q_stride + 8 * j, x);
      else if (slot >= 0) st8f(page + koff + (static_cast<long>(head) * bs + off) * dk + d, x);
    } else if (slot >= 0) {
      const int c = 8 * (i - nq - nk), g = c / dv, d = c - g * dv;
      turn8<T>(x, cs + nf, d, nvf);
      st8f(page + voff + (static_cast<long>(g) * bs + off) * dv + d, x);
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256) rope_rows_wide_kernel(T* __restrict__ out, long out_stride, const T* __restrict__ x,
                                                             long x_stride, const int64_t* __restrict__ positions, int heads,
                                                             int dim, const float* __restrict__ freqs, int nf, float sign,
                                                             float scale) {
  extern __shared__ float2 cs[];
  const long t = blockIdx.x;
  const int n = heads * dim / 8, step = blockDim.x * gridDim.y;
  int i = blockIdx.y * blockDim.x + threadIdx.x;
  float v[8];
  if (i < n) ld8f(x + t * x_stride + 8 * i, v);
  make_turns(cs, freqs, nf, static_cast<float>(positions[t]) * sign);
  __syncthreads();
  while (i < n) {
    turn8<T>(v, cs, 8 * i % dim, nf);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] *= scale;
    st8f(out + t * out_stride + 8 * i, v);
    if ((i += step) < n) ld8f(x + t * x_stride + 8 * i, v);
  }
}

// y[t, c] = act(bias[c] + sum_j w[j, c] x[t - (taps-1) + j, c]), w tap-major [taps, C]; inputs before the
// chunk come from the sequence's state rows [taps-1, C] (oldest first), zeros for a sequence's first
// tokens.  A thread takes V consecutive channels: V = 16 bytes' worth when rows, weights and channel
// count allow whole 16-byte pieces, else 1.  single: every sequence brings one row, and the thread that filtered its
// channels also replaces the carried inputs.
template <typename T> struct Piece;
template <> struct Piece<bf16_t> { static constexpr int N = 8; };
template <> struct Piece<float> { static constexpr int N = 4; };
__device__ __forceinline__ void load_piece(const bf16_t* p, float* o) {
  const uint4 a = *reinterpret_cast<const uint4*>(p);
  o[0] = bf2f_lo(a.x); o[1] = bf2f_hi(a.x); o[2] = bf2f_lo(a.y); o[3] = bf2f_hi(a.y);
  o[4] = bf2f_lo(a.z); o[5] = bf2f_hi(a.z); o[6] = bf2f_lo(a.w); o[7] = bf2f_hi(a.w);
}
__device__ __forceinline__ void load_piece(const float* p, float* o) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
}
__device__ __forceinline__ void store_piece(bf16_t* p, const float* o) {
  uint4 a;
  a.x = pack2(o[0], o[1]); a.y = pack2(o[2], o[3]); a.z = pack2(o[4], o[5]); a.w = pack2(o[6], o[7]);
  *reinterpret_cast<uint4*>(p) = a;
}
__device__ __forceinline__ void store_piece(float* p, const float* o) {
  *reinterpret_cast<float4*>(p) = make_float4(o[0], o[1], o[2], o[3]);
}

template <typename T, bool WIDE>
__global__ void __launch_bounds__(256) causal_conv_kernel(T* __restrict__ out, const T* __restrict__ x, long x_stride,
                                                          const T* __restrict__ w, const T* __restrict__ bias,
                                                          float* __restrict__ state, long state_stride,
                                                          const int* __restrict__ state_rows, long off,
                                                          const int* __restrict__ qsl, const int* __restrict__ seq_lens,
                                                          int S, int C, int taps, int silu, int single) {
  constexpr int V = WIDE ? Piece<T>::N : 1;
  const int t = blockIdx.x;
  const int c = (blockIdx.y * 256 + threadIdx.x) * V;
  if (c >= C) return;
  const int s = single ? t : seq_of_row(qsl, S, t);
  const int row0 = qsl[s], qlen = qsl[s + 1] - row0;
  const int i = t - row0;
  const bool fresh = seq_lens[s] - qlen <= 0;
  float* st = state + static_cast<long>(state_rows[s]) * state_stride + off;
  float acc[V], xv[V], wv[V];
  if constexpr (WIDE) {
    if (bias) load_piece(bias + c, acc);
    else for (int e = 0; e < V; ++e) acc[e] = 0.f;
  } else {
    acc[0] = bias ? ldf(bias + c) : 0.f;
  }
  for (int j = 0; j < taps; ++j) {
    const int src = i - (taps - 1 - j);
    if (src < 0 && fresh) continue;
    if constexpr (WIDE) {
      if (src >= 0) {
        load_piece(x + static_cast<long>(row0 + src) * x_stride + c, xv);
      } else {
        const float* sp = st + static_cast<long>(taps - 1 + src) * C + c;
#pragma unroll
        for (int e = 0; e < V; e += 4) load_piece(sp + e, xv + e);
      }
      load_piece(w + static_cast<long>(j) * C + c, wv);
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] += wv[e] * xv[e];
    } else {
      xv[0] = src >= 0 ? ldf(x + static_cast<long>(row0 + src) * x_stride + c) : st[static_cast<long>(taps - 1 + src) * C + c];
      acc[0] += ldf(w + static_cast<long>(j) * C + c) * xv[0];
    }
  }
  if (single && taps > 1) {  // xv holds this row's input (the last tap): the carried inputs move up by one
    for (int r = 0; r < taps - 1; ++r) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float nv = r == taps - 2 ? xv[e] : (fresh ? 0.f : st[static_cast<long>(r + 1) * C + c + e]);
        st[static_cast<long>(r) * C + c + e] = nv;
      }
    }
  }
  if (silu) {
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] = silu_f(acc[e]);
  }
  if constexpr (WIDE) store_piece(out + static_cast<long>(t) * C + c, acc);
  else stf(out + static_cast<long>(t) * C + c, acc[0]);
}

// The wide form for chunks: a thread takes its channels of 4 consecutive rows, so that a row is read once and not once per
// tap; what a row's filter reaches back to is carried from row to row, and taken anew where a sequence begins.  The terms
// of a sum are those of the kernel above, in its order.  4,096 rows of 6,144 channels, 4 taps: 46 -> 34 us.
constexpr int kConvRows = 4;
constexpr long kConvBytes = 7 << 20;
template <typename T, int TAPS>
__global__ void __launch_bounds__(256) causal_conv_rows_kernel(T* __restrict__ out, const T* __restrict__ x, long x_stride,
                                                               const T* __restrict__ w, const T* __restrict__ bias,
                                                               const float* __restrict__ state, long state_stride,
                                                               const int* __restrict__ state_rows, long off,
                                                               const int* __restrict__ qsl, const int* __restrict__ seq_lens,
                                                               int S, int rows, int C, int silu) {
  constexpr int V = Piece<T>::N;
  const int t0 = blockIdx.x * kConvRows;
  const int c = (blockIdx.y * 256 + threadIdx.x) * V;
  if (c >= C) return;
  uint4 raw[kConvRows];
#pragma unroll
  for (int r = 0; r < kConvRows; ++r)
    raw[r] = *reinterpret_cast<const uint4*>(x + static_cast<long>(min(t0 + r, rows - 1)) * x_stride + c);
  float wv[TAPS][V], bv[V], hist[TAPS - 1][V];
#pragma unroll
  for (int j = 0; j < TAPS; ++j) load_piece(w + static_cast<long>(j) * C + c, wv[j]);
#pragma unroll
  for (int e = 0; e < V; ++e) bv[e] = 0.f;
  if (bias) load_piece(bias + c, bv);
  int s = seq_of_row(qsl, S, t0);
  auto look_back = [&](int t) {  // the TAPS - 1 inputs before row t of sequence s
    const int row0 = qsl[s], i = t - row0;
    const bool fresh = seq_lens[s] - (qsl[s + 1] - row0) <= 0;
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) {
      const int src = i - (TAPS - 1) + j;
      if (src >= 0) {
        load_piece(x + static_cast<long>(row0 + src) * x_stride + c, hist[j]);
      } else if (fresh) {
#pragma unroll
        for (int e = 0; e < V; ++e) hist[j][e] = 0.f;
      } else {
        const float* sp = state + static_cast<long>(state_rows[s]) * state_stride + off + static_cast<long>(TAPS - 1 + src) * C + c;
#pragma unroll
        for (int e = 0; e < V; e += 4) load_piece(sp + e, hist[j] + e);
      }
    }
  };
  look_back(t0);
#pragma unroll
  for (int r = 0; r < kConvRows; ++r) {
    const int t = t0 + r;
    if (t >= rows) break;
    if (r > 0 && s + 1 < S && t == qsl[s + 1]) {  // rows past the last sequence go on as its own
      do ++s; while (s + 1 < S && qsl[s + 1] <= t);
      look_back(t);
    }
    float xv[V], acc[V];
    if constexpr (V == 8) {
      xv[0] = bf2f_lo(raw[r].x); xv[1] = bf2f_hi(raw[r].x); xv[2] = bf2f_lo(raw[r].y); xv[3] = bf2f_hi(raw[r].y);
      xv[4] = bf2f_lo(raw[r].z); xv[5] = bf2f_hi(raw[r].z); xv[6] = bf2f_lo(raw[r].w); xv[7] = bf2f_hi(raw[r].w);
    } else {
      xv[0] = __uint_as_float(raw[r].x); xv[1] = __uint_as_float(raw[r].y);
      xv[2] = __uint_as_float(raw[r].z); xv[3] = __uint_as_float(raw[r].w);
    }
#pragma unroll
    for (int e = 0; e < V; ++e) {
      acc[e] = bv[e];
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j) acc[e] += wv[j][e] * hist[j][e];
      acc[e] += wv[TAPS - 1][e] * xv[e];
      if (silu) acc[e] = silu_f(acc[e]);
    }
    store_piece(out + static_cast<long>(t) * C + c, acc);
#pragma unroll
    for (int j = 0; j + 1 < TAPS - 1; ++j)
#pragma unroll
      for (int e = 0; e < V; ++e) hist[j][e] = hist[j + 1][e];
#pragma unroll
    for (int e = 0; e < V; ++e) hist[TAPS - 2][e] = xv[e];
  }
}

// The convolution without activation, from the fused projection to what attention reads: u = x + bias, the
// filter over u, query columns (the first QC) times a factor that grows with the position, keys and values
// (per kv head dk and dv columns) into the token's page rows.  A thread takes V consecutive channels as above
// (WIDE: no piece crosses from one head to the next).  single: every sequence brings one row, and the thread
// that filtered its channels also replaces the carried inputs.
template <typename T, bool WIDE>
__global__ void __launch_bounds__(256) conv_qkv_cache_kernel(
    T* __restrict__ q, const T* __restrict__ x, long x_stride, const T* __restrict__ w, const T* __restrict__ bias,
    float* __restrict__ state, long state_stride, const int* __restrict__ state_rows, long off, const int* __restrict__ qsl,
    const int* __restrict__ seq_lens, int S, const int64_t* __restrict__ positions, const int64_t* __restrict__ slots,
    T* __restrict__ cache, long block_stride, int koff, int voff, int QC, int G, int dk, int dv, int bs, int taps,
    float temp_coef, float temp_every, int single) {
  constexpr int V = WIDE ? Piece<T>::N : 1;
  const int C = QC + G * (dk + dv);
  const int t = blockIdx.x;
  const int c = (blockIdx.y * 256 + threadIdx.x) * V;
  if (c >= C) return;
  const int s = single ? t : seq_of_row(qsl, S, t);
  const int row0 = qsl[s], qlen = qsl[s + 1] - row0;
  const int i = t - row0;
  const bool fresh = seq_lens[s] - qlen <= 0;
  float* st = state + static_cast<long>(state_rows[s]) * state_stride + off;
  float acc[V], xv[V], wv[V], bv[V];
#pragma unroll
  for (int e = 0; e < V; ++e) acc[e] = bv[e] = 0.f;
  if (bias) {
    if constexpr (WIDE) load_piece(bias + c, bv);
    else bv[0] = ldf(bias + c);
  }
  for (int j = 0; j < taps; ++j) {
    const int src = i - (taps - 1 - j);
    if (src < 0 && fresh) continue;
    if constexpr (WIDE) {
      if (src >= 0) {
        load_piece(x + static_cast<long>(row0 + src) * x_stride + c, xv);
#pragma unroll
        for (int e = 0; e < V; ++e) xv[e] += bv[e];
      } else {
        const float* sp = st + static_cast<long>(taps - 1 + src) * C + c;
#pragma unroll
        for (int e = 0; e < V; e += 4) load_piece(sp + e, xv + e);
      }
      load_piece(w + static_cast<long>(j) * C + c, wv);
    } else {
      xv[0] = src >= 0 ? ldf(x + static_cast<long>(row0 + src) * x_stride + c) + bv[0]
                       : st[static_cast<long>(taps - 1 + src) * C + c];
      wv[0] = ldf(w + static_cast<long>(j) * C + c);
    }
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] += wv[e] * xv[e];
  }
  if (single && taps > 1) {  // xv holds this row's u (the last tap): the carried inputs move up by one
    for (int r = 0; r < taps - 1; ++r) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float nv = r == taps - 2 ? xv[e] : (fresh ? 0.f : st[static_cast<long>(r + 1) * C + c + e]);
        st[static_cast<long>(r) * C + c + e] = nv;
      }
    }
  }
  T* dst;
  if (c < QC) {
    if (temp_coef != 0.f) {
      const float f = 1.f + temp_coef * logf(floorf((static_cast<float>(positions[t]) + 1.f) / temp_every) + 1.f);
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] *= f;
    }
    dst = q + static_cast<long>(t) * QC + c;
  } else {
    const int64_t slot = slots[t];
    if (slot < 0) return;
    const int nk = G * dk;
    const bool key = c < QC + nk;
    const int cc = key ? c - QC : c - QC - nk, d = key ? dk : dv;
    const int g = cc / d;
    dst = cache + (slot / bs) * block_stride + (key ? koff : voff) + (static_cast<long>(g) * bs + slot % bs) * d + (cc - g * d);
  }
  if constexpr (WIDE) store_piece(dst, acc);
  else stf(dst, acc[0]);
}

// The state after the step: the last taps-1 inputs (plus bias) of (old state ++ chunk).  Row r of the new state
// reads old row r + n or a chunk row, so one thread per channel walking r upwards never reads what it
// has already replaced.  Runs after causal_conv_kernel on the same stream.
template <typename T>
__global__ void __launch_bounds__(256) conv_state_kernel(const T* __restrict__ x, long x_stride, const T* __restrict__ bias,
                                                         float* __restrict__ state,
                                                         long state_stride, const int* __restrict__ state_rows, long off,
                                                         const int* __restrict__ qsl, const int* __restrict__ seq_lens,
                                                         int n_rows, int C, int taps) {
  const int s = blockIdx.x;
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= C) return;
  const int row0 = qsl[s];
  if (row0 < 0 || row0 >= n_rows) return;
  const int n = min(qsl[s + 1], n_rows) - row0;
  if (n <= 0) return;
  const bool fresh = seq_lens[s] - n <= 0;
  float* st = state + static_cast<long>(state_rows[s]) * state_stride + off;
  const float b = bias ? ldf(bias + c) : 0.f;
  for (int r = 0; r < taps - 1; ++r) {
    const int src = n - (taps - 1) + r;
    float xv = 0.f;
    if (src >= 0) xv = ldf(x + static_cast<long>(row0 + src) * x_stride + c) + b;
    else if (!fresh) xv = st[static_cast<long>(taps - 1 + src) * C + c];
    st[static_cast<long>(r) * C + c] = xv;
  }
}

// out = scale * [ RMSNorm_groups(o * act(gate)) * w ]            (gate_first)
//     = scale * [ RMSNorm_groups(o) * w * act(gate) ]            (otherwise)
// act = SiLU or sigmoid; w repeats with period wn; one wave per slice of the row (groups > 1) or the
// block for the whole row.
template <typename T>
__global__ void __launch_bounds__(256) gated_norm_kernel(T* __restrict__ out, long out_stride, const float* __restrict__ o,
                                                         const T* __restrict__ gate, long g_stride,
                                                         const T* __restrict__ w, int wn, int N, int groups, float eps,
                                                         int silu, int gate_first, float scale) {
  __shared__ float scratch[16];
  const long row = blockIdx.x;
  const float* orow = o + row * N;
  const T* grow = gate + row * g_stride;
  T* yrow = out + row * out_stride;
  auto act = [&](int c) { const float z = ldf(grow + c); return silu ? silu_f(z) : sigmoid_f(z); };
  if (groups == 1) {
    float s = 0.f;
    for (int c = threadIdx.x; c < N; c += blockDim.x) {
      const float v = gate_first ? orow[c] * act(c) : orow[c];
      s += v * v;
    }
    const float inv = rsqrtf(block_sum(s, scratch) / static_cast<float>(N) + eps);
    for (int c = threadIdx.x; c < N; c += blockDim.x)
      stf(yrow + c, orow[c] * act(c) * inv * ldf(w + c % wn) * scale);
    return;
  }
  const int n = N / groups, lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int g = wid; g < groups; g += nw) {
    float s = 0.f;
    for (int c = lane; c < n; c += 64) {
      const int i = g * n + c;
      const float v = gate_first ? orow[i] * act(i) : orow[i];
      s += v * v;
    }
    const float inv = rsqrtf(wave_sum(s) / static_cast<float>(n) + eps);
    for (int c = lane; c < n; c += 64) {
      const int i = g * n + c;
      stf(yrow + i, orow[i] * act(i) * inv * ldf(w + i % wn) * scale);
    }
  }
}

// The same for slices of 8 LP NP entries, LP a power of two up to 64: LP neighbouring lanes hold a slice, 8 entries a lane and
// step of LP lanes, from the activation to the store; a wave serves 64 / LP slices at once.  4,096 rows of 4,096, 8
// slices, SiLU first: 48.6 -> 28 us; 64 rows: 11.2 -> 4.5 us.
template <typename T, int NP>
__global__ void __launch_bounds__(256) gated_norm_wide_kernel(T* __restrict__ out, long out_stride, const float* __restrict__ o,
                                                              const T* __restrict__ gate, long g_stride,
                                                              const T* __restrict__ w, int wn, int N, int n, int LP, float eps,
                                                              int silu, int gate_first, float scale) {
  const long row = blockIdx.x;
  const int l = threadIdx.x & (LP - 1);  // LP divides 64
  for (int sl = threadIdx.x / LP; sl * n < N; sl += blockDim.x / LP) {
    float v[NP][8], g[NP][8];
    float s = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int c = sl * n + 8 * (l + p * LP);
      ld8f(o + row * N + c, v[p]);
      ld8f(gate + row * g_stride + c, g[p]);
    }
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float a = silu ? silu_f(g[p][e]) : sigmoid_f(g[p][e]);
        if (gate_first) v[p][e] *= a;
        s += v[p][e] * v[p][e];
        g[p][e] = gate_first ? 1.f : a;
      }
    for (int d = 1; d < LP; d <<= 1) s += __shfl_xor(s, d, 64);
    const float inv = rsqrtf(s / static_cast<float>(n) + eps);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int c = sl * n + 8 * (l + p * LP);
      float wv[8];
      ld8f(w + c % wn, wv);
#pragma unroll
      for (int e = 0; e < 8; ++e) wv[e] = v[p][e] * inv * wv[e] * g[p][e] * scale;
      st8f(out + row * out_stride + c, wv);
    }
  }
}

#define MIX_DISPATCH(bf, ...)                      \
  do {                                             \
    if (bf) { using T = bf16_t; __VA_ARGS__; }     \
    else { using T = float; __VA_ARGS__; }         \
  } while (0)

void launch_embed_scaled(float* out, const int64_t* ids, const void* table, int rows, int W, long vocab, float scale,
                         bool bf, hipStream_t st) {
  if (rows == 0) return;
  MIX_DISPATCH(bf, hipLaunchKernelGGL(embed_scaled_kernel<T>, dim3(rows), dim3(256), 0, st, out, ids, (const T*)table, W,
                                      vocab, scale));
  MXS_CHECK_LAUNCH();
}

// The form with a wave per token and head is faster while the chip holds all waves at once (7 tokens of 32 + 8 + 8 heads
// of 64 3.3 us, 4.0 here; 64 tokens 3.7 / 4.1; 200 tokens 5.2 / 4.2) or a token has no more pieces than a wave lanes (64
// tokens of 4 + 2 + 2 heads of 64 3.3 / 4.4; 4,096 tokens of one head of 8 6.1 / 7.1).  Up to kFewRows tokens, a token's pieces go over as many workgroups as hold them (64 tokens of
// 128 + 8 + 8 heads of 128: 7.1 us with one, 4.7).
constexpr int kFewRows = 256, kFewPieces = 64, kFewWaves = 4096;

void launch_rope_qkv_cache(void* q, long q_stride, const void* k, long k_stride, const void* v, long v_stride,
                           const int64_t* positions, const int64_t* slots, void* cache, long block_stride, int rows,
                           int koff, int voff, int H, int G, int dk, int dv, int bs, const float* freqs, int nf,
                           const void* q_norm, const void* k_norm, float eps, const float* v_freqs, int nvf, bool bf,
                           hipStream_t st) {
  if (rows == 0) return;
  auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const int LP = dk / 8, n = H * LP + (k ? G * (LP + dv / 8) : 0);  // pieces of a token
  if (n > kFewPieces && static_cast<long>(rows) * (H + (k ? 2 * G : 0)) > kFewWaves && dk % 8 == 0 && LP <= 64 && (LP & (LP - 1)) == 0 && q_stride % 8 == 0 && al(q) && al(q_norm) && al(k_norm) &&
      nf + nvf <= 4096 &&
      (k == nullptr || (dv % 8 == 0 && k_stride % 8 == 0 && v_stride % 8 == 0 && al(k) && al(v) && al(cache) && koff % 8 == 0 &&
                        voff % 8 == 0 && block_stride % 8 == 0))) {
    // few tokens: a lane for every piece, over several workgroups where one does not hold them; many: smaller workgroups pack
    // better (4,096 tokens 15.4 us, 18.3 with 512)
    const int threads = std::min(rows <= 1024 ? 512 : 256, (n + 63) / 64 * 64);
    const dim3 grid(rows, rows <= kFewRows ? (n + threads - 1) / threads : 1);
    MIX_DISPATCH(bf, hipLaunchKernelGGL(rope_qkv_cache_wide_kernel<T>, grid, dim3(threads), (nf + nvf) * sizeof(float2), st,
                                        (T*)q, q_stride, (const T*)k, k_stride, (const T*)v, v_stride, positions, slots,
                                        (T*)cache, block_stride, koff, voff, H, G, dk, dv, bs, freqs, nf, (const T*)q_norm,
                                        (const T*)k_norm, eps, v_freqs, nvf));
    MXS_CHECK_LAUNCH();
    return;
  }
  const dim3 grid(rows, H + (k != nullptr ? 2 * G : 0));
  MIX_DISPATCH(bf, hipLaunchKernelGGL(rope_qkv_cache_kernel<T>, grid, dim3(64), 0, st, (T*)q, q_stride, (const T*)k,
                                      k_stride, (const T*)v, v_stride, positions, slots, (T*)cache, block_stride, koff,
                                      voff, H, G, dk, dv, bs, freqs, nf, (const T*)q_norm, (const T*)k_norm, eps, v_freqs,
                                      nvf));
  MXS_CHECK_LAUNCH();
}

void launch_rope_rows(void* out, long out_stride, const void* x, long x_stride, const int64_t* positions, int rows,
                      int heads, int dim, const float* freqs, int nf, float sign, float scale, bool bf, hipStream_t st) {
  if (rows == 0) return;
  auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (static_cast<long>(rows) * heads > kFewWaves && dim % 8 == 0 && x_stride % 8 == 0 && out_stride % 8 == 0 && al(x) && al(out) && nf <= 4096) {
    const int n = heads * dim / 8, threads = std::min(256, (n + 63) / 64 * 64);
    const dim3 grid(rows, rows <= kFewRows ? (n + threads - 1) / threads : 1);
    MIX_DISPATCH(bf, hipLaunchKernelGGL(rope_rows_wide_kernel<T>, grid, dim3(threads), nf * sizeof(float2), st, (T*)out, out_stride,
                                        (const T*)x, x_stride, positions, heads, dim, freqs, nf, sign, scale));
    MXS_CHECK_LAUNCH();
    return;
  }
  MIX_DISPATCH(bf, hipLaunchKernelGGL(rope_rows_kernel<T>, dim3(rows, heads), dim3(64), 0, st, (T*)out, out_stride,
                                      (const T*)x, x_stride, positions, dim, freqs, nf, sign, scale));
  MXS_CHECK_LAUNCH();
}

void launch_causal_conv(void* out, const void* x, long x_stride, const void* w, const void* bias, float* state,
                        long state_stride, const int* state_rows, long off, const int* qsl, const int* seq_lens, int S,
                        int rows, int C, int taps, int silu, bool single, bool bf, hipStream_t st) {
  if (rows == 0 || S == 0) return;
  const int cb = (C + 255) / 256;
  // whole 16-byte pieces everywhere: rows, weights, bias, output, and the fp32 state rows
  const int v = bf ? 8 : 4;
  auto al = [](const void* ptr) { return reinterpret_cast<uintptr_t>(ptr) % 16 == 0; };
  const bool wide = C % v == 0 && x_stride % v == 0 && al(x) && al(w) && al(out) && (bias == nullptr || al(bias)) &&
                    al(state) && state_stride % 4 == 0 && off % 4 == 0;
  // Four rows a thread where the bytes count: below some 7 MB of rows a quarter of the workgroups and a chain of four rows take
  // longer than reading rows again, most of all for few channels (bf16, 4 taps, one row a thread / four: 4,096 rows of 64
  // 7.9 / 16.0 us, 2,048 of 1,024 8.0 / 10.1, 1,024 of 3,072 10.3 / 10.6, 700 of 5,120 12.3 / 12.2, 2,048 of 2,048 13.1 / 11.1,
  // 4,096 of 6,144 46.1 / 34.4; fp32, 2,048 of 512 6.6 / 7.3, 512 of 3,072 8.5 / 7.8).  Two taps read too little twice: 4,096 of
  // 3,072 20.4 / 21.3.
  if (wide && !single && (taps == 3 || taps == 4) && static_cast<long>(rows) * C * (16 / v) >= kConvBytes) {
    const dim3 grid((rows + kConvRows - 1) / kConvRows, (C / v + 255) / 256);
#define MIX_CONV(TAPS)                                                                                                    \
  MIX_DISPATCH(bf, hipLaunchKernelGGL((causal_conv_rows_kernel<T, TAPS>), grid, dim3(256), 0, st, (T*)out, (const T*)x,   \
                                      x_stride, (const T*)w, (const T*)bias, state, state_stride, state_rows, off, qsl,  \
                                      seq_lens, S, rows, C, silu))
    if (taps == 3) MIX_CONV(3);
    else MIX_CONV(4);
#undef MIX_CONV
  } else if (wide) {
    const int cw = (C / v + 255) / 256;
    MIX_DISPATCH(bf, hipLaunchKernelGGL((causal_conv_kernel<T, true>), dim3(rows, cw), dim3(256), 0, st, (T*)out,
                                        (const T*)x, x_stride, (const T*)w, (const T*)bias, state, state_stride,
                                        state_rows, off, qsl, seq_lens, S, C, taps, silu, single ? 1 : 0));
  } else {
    MIX_DISPATCH(bf, hipLaunchKernelGGL((causal_conv_kernel<T, false>), dim3(rows, cb), dim3(256), 0, st, (T*)out,
                                        (const T*)x, x_stride, (const T*)w, (const T*)bias, state, state_stride,
                                        state_rows, off, qsl, seq_lens, S, C, taps, silu, single ? 1 : 0));
  }
  MXS_CHECK_LAUNCH();
  if (taps > 1 && !single) {
    MIX_DISPATCH(bf, hipLaunchKernelGGL(conv_state_kernel<T>, dim3(S, cb), dim3(256), 0, st, (const T*)x, x_stride,
                                        (const T*)nullptr, state, state_stride, state_rows, off, qsl, seq_lens, rows, C, taps));
    MXS_CHECK_LAUNCH();
  }
}

void launch_conv_qkv_cache(void* q, const void* x, long x_stride, const void* w, const void* bias, float* state,
                           long state_stride, const int* state_rows, long off, const int* qsl, const int* seq_lens, int S,
                           int rows, const int64_t* positions, const int64_t* slots, void* cache, long block_stride, int koff,
                           int voff, int QC, int G, int dk, int dv, int bs, int taps, float temp_coef, float temp_every,
                           bool single, bool bf, hipStream_t st) {
  if (rows == 0 || S == 0) return;
  const int C = QC + G * (dk + dv), v = bf ? 8 : 4;
  auto al = [](const void* ptr) { return reinterpret_cast<uintptr_t>(ptr) % 16 == 0; };
  const bool wide = QC % v == 0 && dk % v == 0 && dv % v == 0 && x_stride % v == 0 && koff % v == 0 && voff % v == 0 &&
                    block_stride % v == 0 && al(x) && al(w) && al(q) && al(cache) && (bias == nullptr || al(bias)) &&
                    al(state) && state_stride % 4 == 0 && off % 4 == 0;
  const dim3 grid(rows, ((wide ? C / v : C) + 255) / 256);
  if (wide) {
    MIX_DISPATCH(bf, hipLaunchKernelGGL((conv_qkv_cache_kernel<T, true>), grid, dim3(256), 0, st, (T*)q, (const T*)x, x_stride,
                                        (const T*)w, (const T*)bias, state, state_stride, state_rows, off, qsl, seq_lens, S,
                                        positions, slots, (T*)cache, block_stride, koff, voff, QC, G, dk, dv, bs, taps,
                                        temp_coef, temp_every, single ? 1 : 0));
  } else {
    MIX_DISPATCH(bf, hipLaunchKernelGGL((conv_qkv_cache_kernel<T, false>), grid, dim3(256), 0, st, (T*)q, (const T*)x, x_stride,
                                        (const T*)w, (const T*)bias, state, state_stride, state_rows, off, qsl, seq_lens, S,
                                        positions, slots, (T*)cache, block_stride, koff, voff, QC, G, dk, dv, bs, taps,
                                        temp_coef, temp_every, single ? 1 : 0));
  }
  MXS_CHECK_LAUNCH();
  if (taps > 1 && !single) {
    MIX_DISPATCH(bf, hipLaunchKernelGGL(conv_state_kernel<T>, dim3(S, (C + 255) / 256), dim3(256), 0, st, (const T*)x, x_stride,
                                        (const T*)bias, state, state_stride, state_rows, off, qsl, seq_lens, rows, C, taps));
    MXS_CHECK_LAUNCH();
  }
}

void launch_gated_norm(void* out, long out_stride, const float* o, const void* gate, long g_stride, const void* w, int wn,
                       int rows, int N, int groups, float eps, int silu, int gate_first, float scale, bool bf,
                       hipStream_t st) {
  if (rows == 0) return;
  auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const int n = N / groups, LP = n % 8 == 0 ? std::min(64, n / 8) : 0, np = LP ? n / 8 / LP : 0;
  // up to four short slices have a wave each in the form above: 64 rows of two slices of 64 3.3 / 3.8 us, of 32 slices of 8
  // 10.7 / 3.7
  if ((N > 256 || groups > 4) && LP && (LP & (LP - 1)) == 0 && 8 * LP * np == n && (np == 1 || np == 2 || np == 4 || np == 8) && wn % 8 == 0 && N % 8 == 0 &&
      g_stride % 8 == 0 && out_stride % 8 == 0 && al(out) && al(o) && al(gate) && al(w)) {
    const int threads = std::min(256, (N / 8 / np + 63) / 64 * 64);
#define MIX_GN(NP)                                                                                                     \
  MIX_DISPATCH(bf, hipLaunchKernelGGL((gated_norm_wide_kernel<T, NP>), dim3(rows), dim3(threads), 0, st, (T*)out, out_stride, o, \
                                      (const T*)gate, g_stride, (const T*)w, wn, N, n, LP, eps, silu, gate_first, scale))
    if (np == 1) MIX_GN(1);
    else if (np == 2) MIX_GN(2);
    else if (np == 4) MIX_GN(4);
    else MIX_GN(8);
#undef MIX_GN
    MXS_CHECK_LAUNCH();
    return;
  }
  MIX_DISPATCH(bf, hipLaunchKernelGGL(gated_norm_kernel<T>, dim3(rows), dim3(256), 0, st, (T*)out, out_stride, o,
                                      (const T*)gate, g_stride, (const T*)w, wn, N, groups, eps, silu, gate_first, scale));
  MXS_CHECK_LAUNCH();
}

}  // namespace mxs
