// K13: fused sampling. One workgroup per row of logits (vocab up to ~152k):
//   temperature <= 0        -> argmax (lowest index on ties)
//   otherwise               -> Gumbel-max over softmax(z / T) restricted to the top-k / top-p set:
//                              argmax_v (z_v / T + g_v), g_v = -log(-log u_v),
//                              u_v = hash(seed, step, v)  (counter-based: reproducible per request,
//                              graph-capturable, no RNG state).  No sort: the top-k and top-p
//                              thresholds come from a histogram of the row (select_threshold).
// The hash matches mxserve/ops/reference.py::_hash_u32 bit for bit.
#include <cstdlib>

#include "common.h"

namespace mxs {

__device__ __forceinline__ uint32_t hash_u32(uint32_t x) {
  x = (x ^ (x >> 16)) * 0x7FEB352Du;
  x = (x ^ (x >> 15)) * 0x846CA68Bu;
  return x ^ (x >> 16);
}

struct ArgMax {
  float v;
  int i;
};

__device__ __forceinline__ ArgMax better(ArgMax a, ArgMax b) {
  if (b.v > a.v || (b.v == a.v && b.i < a.i)) return b;
  return a;
}

__device__ ArgMax block_argmax(ArgMax a, float* sv, int* si) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgMax b{__shfl_xor(a.v, o, 64), __shfl_xor(a.i, o, 64)};
    a = better(a, b);
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if (lane == 0) {
    sv[wid] = a.v;
    si[wid] = a.i;
  }
  __syncthreads();
  ArgMax r{sv[0], si[0]};
  for (int w = 1; w < nw; ++w) r = better(r, ArgMax{sv[w], si[w]});
  return r;
}

__device__ __forceinline__ float ld(const float* p, int v) { return p[v]; }
__device__ __forceinline__ float ld(const bf16_t* p, int v) { return bf2f(p[v]); }

// 8 consecutive logits starting at v (v % 8 == 0, row 16-byte aligned)
__device__ __forceinline__ void ld8(const bf16_t* p, int v, float (&o)[8]) {
  const uint4 w = *reinterpret_cast<const uint4*>(p + v);
  const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    o[2 * k] = bf2f_lo(u[k]);
    o[2 * k + 1] = bf2f_hi(u[k]);
  }
}
__device__ __forceinline__ void ld8(const float* p, int v, float (&o)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(p + v), b = *reinterpret_cast<const float4*>(p + v + 4);
  o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
}

// Gumbel noise in base-2 units: argmax_v (z_v / T + G_v) with G = -ln(-ln u) is argmax_v of
// (z_v / T + G_v) log2(e) = z_v log2(e) / T - log2(-log2 u) + const, so the scores are taken as
// x * (log2(e) / T) + gumbel2(u) with two native v_log_f32 (log2) per logit instead of two
// full-precision logf (u is in [2^-25, 1 - 2^-25]: both logarithms see normal inputs).  The final
// Gumbel-max pass over a 128k-vocab row is the sampling kernel's dominant cost (79 us per 448-row
// decode step with logf, profiles/r5/headline).
__device__ __forceinline__ float gumbel2(uint32_t key, int v) {
  const uint32_t h = hash_u32(key ^ hash_u32(static_cast<uint32_t>(v) + 0x632BE5ABu));
  const float u = (static_cast<float>(h >> 8) + 0.5f) * (1.f / 16777216.f);
  return -__builtin_amdgcn_logf(-__builtin_amdgcn_logf(u));
}
constexpr float kSLog2e = 1.4426950408889634f;

// ---- a row's logits, wherever they are.  each(f) calls f(logit, index) for every logit this thread owns (slots past the
// row: -inf with an index >= V).  Register forms: the workgroup loads its row ONCE, 8 neighbouring logits per thread and
// step of 1024 threads, and every pass runs on registers; rows that do not fit or are not 16-byte aligned are read again
// by each pass.
template <int NE>
struct RegRow16 {  // bf16, packed pairs
  using T = bf16_t;
  uint32_t r[NE / 2];
  __device__ __forceinline__ RegRow16(const bf16_t* z, int V, bool) {
#pragma unroll
    for (int q = 0; q < NE / 8; ++q) {
      const int v0 = 8 * (static_cast<int>(threadIdx.x) + 1024 * q);
      uint4 w = make_uint4(0xFF80FF80u, 0xFF80FF80u, 0xFF80FF80u, 0xFF80FF80u);  // -inf pairs
      if (v0 < V) w = *reinterpret_cast<const uint4*>(z + v0);
      r[4 * q] = w.x;
      r[4 * q + 1] = w.y;
      r[4 * q + 2] = w.z;
      r[4 * q + 3] = w.w;
    }
  }
  template <class F>
  __device__ __forceinline__ void each(F f) {
    // an empty asm "modifying" the packed row at the top of each pass: keeps hipcc from carrying all unpacked
    // floats from one pass to the next, which would spill
#pragma unroll
    for (int i = 0; i < NE / 2; ++i) asm volatile("" : "+v"(r[i]));
    int first = 8 * static_cast<int>(threadIdx.x);
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      if ((e & 7) == 0) asm volatile("" : "+v"(first));  // nor all indices
      f((e & 1) ? bf2f_hi(r[e >> 1]) : bf2f_lo(r[e >> 1]), first + 8192 * (e >> 3) + (e & 7));
      if ((e & 3) == 3) __builtin_amdgcn_sched_barrier(0);  // a few independent chains in flight, not the whole row
    }
  }
};

template <int NE>
struct RegRow32 {
  using T = float;
  float r[NE];
  __device__ __forceinline__ RegRow32(const float* z, int V, bool) {
#pragma unroll
    for (int q = 0; q < NE / 8; ++q) {
      const int v0 = 8 * (static_cast<int>(threadIdx.x) + 1024 * q);
      float x[8] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY, -INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (v0 < V) ld8(z, v0, x);
#pragma unroll
      for (int i = 0; i < 8; ++i) r[8 * q + i] = x[i];
    }
  }
  template <class F>
  __device__ __forceinline__ void each(F f) {
#pragma unroll
    for (int i = 0; i < NE; ++i) asm volatile("" : "+v"(r[i]));
    int first = 8 * static_cast<int>(threadIdx.x);
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      if ((e & 7) == 0) asm volatile("" : "+v"(first));
      f(r[e], first + 8192 * (e >> 3) + (e & 7));
      if ((e & 3) == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
};

template <typename T_>
struct MemRow {
  using T = T_;
  const T* z;
  int V;
  bool vec;
  __device__ __forceinline__ MemRow(const T* z_, int V_, bool vec_) : z(z_), V(V_), vec(vec_) {}
  template <class F>
  __device__ __forceinline__ void each(F f) {
    if (vec) {
      constexpr int W = 8 * 1024, D = 8 / sizeof(T);  // D pieces of 8 in flight (one row of 128,256 fp32: 21.0 -> 9.9 us)
      for (int v = 8 * static_cast<int>(threadIdx.x); v < V; v += D * W) {
        float x[D][8];
#pragma unroll
        for (int g = 0; g < D; ++g)
          if (g == 0 || v + g * W < V) ld8(z, v + g * W, x[g]);
#pragma unroll
        for (int g = 0; g < D; ++g) {
          if (g > 0 && v + g * W >= V) break;
#pragma unroll
          for (int u = 0; u < 8; ++u) f(x[g][u], v + g * W + u);
        }
      }
    } else {
#pragma unroll 4
      for (int v = threadIdx.x; v < V; v += 1024) f(ld(z, v), v);
    }
  }
};

// Thresholds of the top-k / top-p sets.  "The largest logit x with weight({z >= x}) >= target", weight 1 for top-k and
// the logit's share of the softmax for top-p, is found from a histogram of weights over kSelBins equal steps of [lo, hi]:
// the bin in which the sum from the top reaches the target is known after one pass, its logits (some hundred of a
// 128k row) are collected and ranked against each other; a fuller bin is cut again.  Two passes over the row where a
// bisection over value took 32, each with an exponential per logit: that was what a row's time went into, and a row is
// one workgroup, so a step with few sampled rows waits for it (MI355X, 128,256 bf16 logits, 13 rows: 275 us; 32,000
// fp32 logits, 64 rows: 177 us.  Now 61 us and 23 us).  Shares (at most 1) are 2^-46 fixed point, what 64-bit sums of
// 2^17 of them hold, with a bit less for each doubling of the row beyond: the sums do not depend on the order of the LDS
// atomics, so a request's tokens stay reproducible.  A share loses less than a step, a row 2^-29 of its sum, where an fp32
// sum rounds at 2^-24 (one word of 32 bits a share, 2^-15 of a row: 2 us less of 60).
constexpr int kSelBins = 2048, kSelList = 512;
struct SelLds {
  unsigned long long hist[kSelBins];
  unsigned long long wave[16];
  unsigned long long above;
  unsigned long long lw[kSelList];
  float list[kSelList];
  int n, bin;
};

// by_share: weight 2^32 hscale exp2((x - mx) * invt2), target `goal` of the whole; otherwise weight 1, target goal itself.
// lo <= hi finite; logits outside [lo, hi] have no weight.  -inf when even all of them stay below the target.
template <class Row>
__device__ __forceinline__ float select_threshold(Row& R, SelLds& L, float* sv, bool by_share, double goal, float mx,
                                                  float invt2, float hscale, float lo, float hi) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  auto weight = [&](float x) -> unsigned long long {
    if (!by_share) return 1ull;
    const float a = __builtin_amdgcn_exp2f((x - mx) * invt2) * hscale;
    const uint32_t up = static_cast<uint32_t>(a);  // both words are exact
    const uint32_t low = static_cast<uint32_t>(__builtin_amdgcn_fractf(a) * 4294967296.f);
    return static_cast<unsigned long long>(up) << 32 | low;
  };
  unsigned long long above = 0, target = 0;
  for (int level = 0; level < 8; ++level) {
    if (!(hi > lo)) return lo;
    __syncthreads();  // the level before is done with the bins
    for (int i = tid; i < kSelBins; i += 1024) L.hist[i] = 0;
    if (tid == 0) {
      L.n = 0;
      L.bin = -1;
    }
    __syncthreads();
    const float scale = fminf(kSelBins / (hi - lo), 3e38f);
    auto bin_of = [&](float x) -> int {
      return min(static_cast<int>(fminf((hi - x) * scale, static_cast<float>(kSelBins))), kSelBins - 1);
    };
    R.each([&](float x, int) {
      if (x >= lo && x <= hi) atomicAdd(&L.hist[bin_of(x)], weight(x));
    });
    __syncthreads();
    // the bin that reaches the target: sums from the top, two bins a thread
    const unsigned long long a = L.hist[2 * tid], b = L.hist[2 * tid + 1];
    unsigned long long s = a + b;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned long long t = __shfl_up(s, o, 64);
      if (lane >= o) s += t;
    }
    if (lane == 63) L.wave[wid] = s;
    __syncthreads();
    unsigned long long before = above, total = 0;
#pragma unroll 2
    for (int w = 0; w < 16; ++w) {
      if (w < wid) before += L.wave[w];
      total += L.wave[w];
    }
    if (level == 0) {
      const double t = by_share ? ceil(goal * static_cast<double>(total)) : goal;
      target = t < 1.0 ? 1ull : static_cast<unsigned long long>(t);
    }
    const unsigned long long e0 = before + s - a - b, e1 = e0 + a;
    if (e0 < target && e1 >= target) {
      L.bin = 2 * tid;
      L.above = e0;
    } else if (e1 < target && e1 + b >= target) {
      L.bin = 2 * tid + 1;
      L.above = e1;
    }
    __syncthreads();
    const int bin = L.bin;
    if (bin < 0) return -INFINITY;
    above = L.above;
    // its logits
    float bmn = INFINITY, bmx = -INFINITY;
    R.each([&](float x, int) {
      const bool in = x >= lo && x <= hi && bin_of(x) == bin;
      const unsigned long long m = __ballot(in);
      if (m != 0) {
        const int first = __builtin_ctzll(m);
        int at = 0;
        if (lane == first) at = atomicAdd(&L.n, static_cast<int>(__popcll(m)));
        at = __shfl(at, first, 64) + __popcll(m & ((1ull << lane) - 1));
        if (in) {
          bmn = fminf(bmn, x);
          bmx = fmaxf(bmx, x);
          if (at < kSelList) L.list[at] = x;
        }
      }
    });
    __syncthreads();
    const int n = L.n;
    if (n <= kSelList) {
      if (tid < n) L.lw[tid] = weight(L.list[tid]);
      __syncthreads();
      float best = -INFINITY;
      if (tid < n) {
        const float x = L.list[tid];
        unsigned long long sum = above;
#pragma unroll 4
        for (int j = 0; j < n; ++j) sum += L.list[j] >= x ? L.lw[j] : 0ull;
        if (sum >= target) best = x;
      }
      return block_max(best, sv);
    }
    lo = -block_max(-bmn, sv);
    hi = block_max(bmx, sv);
  }
  return lo;
}

template <class Row>
__global__ void __launch_bounds__(1024) sample_kernel(int64_t* __restrict__ out,
                                                      const typename Row::T* __restrict__ logits, int V, long row_stride,
                                                      bool vec, const float* __restrict__ temperature,
                                                      const float* __restrict__ top_p, const int* __restrict__ top_k,
                                                      const int64_t* __restrict__ seeds,
                                                      const int64_t* __restrict__ steps) {
  __shared__ float sv[16];
  __shared__ int si[16];
  __shared__ SelLds L;
  using T = typename Row::T;
  const int row = blockIdx.x;
  const T* z = logits + row * row_stride;
  const float t = temperature[row];
  const int k = top_k[row];
  const float p = top_p[row];
  const bool drawn = t > 0.f, cut = drawn && ((k > 0 && k < V) || p < 1.f);
  const float invt2 = 1.f / t * kSLog2e;
  const uint32_t key = hash_u32(static_cast<uint32_t>(static_cast<uint64_t>(seeds[row]) * 0x9E3779B1ull +
                                                      static_cast<uint64_t>(steps[row])));
  auto finish = [&](const ArgMax& a) {
    const ArgMax r = block_argmax(a, sv, si);
    if (threadIdx.x == 0) out[row] = r.i;
  };
  auto draw = [&](auto& from, float thr) {
    ArgMax a{-INFINITY, 0x7FFFFFFF};
    from.each([&](float x, int v) {
      if (v < V && x >= thr) a = better(a, ArgMax{x * invt2 + gumbel2(key, v), v});
    });
    finish(a);
  };
  if (!cut) {  // one pass: registers would give nothing.  One greedy row of 151,936 bf16: 20.4 us held first, 12.1 us
    MemRow<T> M(z, V, vec);
    if (drawn) {
      draw(M, -INFINITY);
    } else {
      ArgMax a{-INFINITY, 0x7FFFFFFF};
      M.each([&](float x, int v) { a = better(a, ArgMax{x, v}); });
      finish(a);
    }
    return;
  }
  Row R(z, V, vec);
  float thr = -INFINITY, mx = -INFINITY, mn = INFINITY;
  R.each([&](float x, int) {
    mx = fmaxf(mx, x);
    if (x != -INFINITY) mn = fminf(mn, x);
  });
  mx = block_max(mx, sv);
  mn = -block_max(-mn, sv);
  if (mx == INFINITY) {  // nothing below an infinite logit has a share
    thr = mx;
  } else if (mx > -INFINITY) {
    // a share of 1 is 2^32 hscale; the row's shares together stay below 2^63
    const float hscale = V <= 1 << 17 ? 16384.f : static_cast<float>(1u << max(__clz(V - 1) - 1, 0));
    for (int by_share = 0; by_share < 2; ++by_share) {
      if (by_share ? p < 1.f : k > 0 && k < V)
        thr = fmaxf(thr, select_threshold(R, L, sv, by_share != 0, by_share ? static_cast<double>(p) : static_cast<double>(k),
                                          mx, invt2, hscale, by_share ? fmaxf(mn, mx - 88.f * t) : mn, mx));
    }
  }
  draw(R, thr);
}

void launch_sample(int64_t* out, const void* logits, bool bf16, int B, int V, long row_stride,
                   const float* temperature, const float* top_p, const int* top_k, const int64_t* seeds,
                   const int64_t* steps, hipStream_t s) {
  if (B == 0) return;
  const bool vec = V % 8 == 0 && row_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(logits) & 15) == 0;
  auto run = [&](auto kernel, auto* z) {
    hipLaunchKernelGGL(kernel, dim3(B), dim3(1024), 0, s, out, z, V, row_stride, vec, temperature, top_p, top_k, seeds, steps);
  };
  static const bool reg_ok = [] {  // MXS_SAMPLE_REG=0: rows are read again by each pass (the same tokens)
    const char* e = std::getenv("MXS_SAMPLE_REG");
    return e == nullptr || e[0] != '0';
  }();
  // registers hold a row up to what 1024 threads of 128 VGPRs have room for: 160 bf16 or 64 fp32 logits a thread
  const int fit = vec && reg_ok ? V : 1 << 30;
  if (bf16) {
    const auto* z = static_cast<const bf16_t*>(logits);
    if (fit <= 1024 * 32) run(sample_kernel<RegRow16<32>>, z);
    else if (fit <= 1024 * 128) run(sample_kernel<RegRow16<128>>, z);
    else if (fit <= 1024 * 160) run(sample_kernel<RegRow16<160>>, z);
    else run(sample_kernel<MemRow<bf16_t>>, z);
  } else {
    const auto* z = static_cast<const float*>(logits);
    if (fit <= 1024 * 32) run(sample_kernel<RegRow32<32>>, z);
    else if (fit <= 1024 * 64) run(sample_kernel<RegRow32<64>>, z);
    else run(sample_kernel<MemRow<float>>, z);
  }
  MXS_CHECK_LAUNCH();
}

// Log-probabilities for the rows that asked for them (OpenAI `logprobs` / `top_logprobs`).
// One workgroup per selected row: one pass for the row's log-sum-exp (online max / rescaled sum,
// merged across lanes and waves), then the sampled token's log-prob and the K best tokens by K
// block-argmax passes, each excluding everything at or above the previous pick in (value desc,
// index asc) order.  K <= 20, and only requesting rows are touched, so the extra reads are a few
// hundred KB of L2-resident logits per row.  Log-probs are of the raw model distribution (before
// temperature / top-k / top-p), as vLLM reports them.
template <typename T>
__global__ void __launch_bounds__(1024) logprobs_kernel(float* __restrict__ tok_lp, int64_t* __restrict__ top_ids,
                                                        float* __restrict__ top_lp, const T* __restrict__ logits,
                                                        int V, long row_stride, const int64_t* __restrict__ rows,
                                                        const int64_t* __restrict__ tokens, int K) {
  __shared__ float sv[16];
  __shared__ int si[16];
  __shared__ float sm[16], ss[16];
  const int b = blockIdx.x;
  const T* z = logits + rows[b] * row_stride;
  float m = -INFINITY, s = 0.f;
  for (int v = threadIdx.x; v < V; v += blockDim.x) {
    const float x = ld(z, v);
    if (x > m) {
      s = s * __expf(m - x) + 1.f;
      m = x;
    } else {
      s += __expf(x - m);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float m2 = __shfl_xor(m, o, 64), s2 = __shfl_xor(s, o, 64);
    const float M = fmaxf(m, m2);
    s = (M == -INFINITY) ? 0.f : s * __expf(m - M) + s2 * __expf(m2 - M);
    m = M;
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if (lane == 0) {
    sm[wid] = m;
    ss[wid] = s;
  }
  __syncthreads();
  float M = sm[0];
  for (int w = 1; w < nw; ++w) M = fmaxf(M, sm[w]);
  float S = 0.f;
  for (int w = 0; w < nw; ++w) S += sm[w] == -INFINITY ? 0.f : ss[w] * __expf(sm[w] - M);
  const float lse = M + logf(S);
  if (threadIdx.x == 0) tok_lp[b] = ld(z, static_cast<int>(tokens[b])) - lse;
  ArgMax prev{INFINITY, -1};
  for (int j = 0; j < K; ++j) {
    ArgMax a{-INFINITY, 0x7FFFFFFF};
    for (int v = threadIdx.x; v < V; v += blockDim.x) {
      const float x = ld(z, v);
      if (x < prev.v || (x == prev.v && v > prev.i)) a = better(a, ArgMax{x, v});
    }
    const ArgMax r = block_argmax(a, sv, si);
    if (threadIdx.x == 0) {
      top_ids[b * K + j] = r.i < V ? r.i : 0;
      top_lp[b * K + j] = r.v - lse;
    }
    prev = r;
  }
}

void launch_logprobs(float* tok_lp, int64_t* top_ids, float* top_lp, const void* logits, bool bf16, int n, int V,
                     long row_stride, const int64_t* rows, const int64_t* tokens, int K, hipStream_t s) {
  if (n == 0) return;
  if (bf16)
    hipLaunchKernelGGL(logprobs_kernel<bf16_t>, dim3(n), dim3(1024), 0, s, tok_lp, top_ids, top_lp,
                       static_cast<const bf16_t*>(logits), V, row_stride, rows, tokens, K);
  else
    hipLaunchKernelGGL(logprobs_kernel<float>, dim3(n), dim3(1024), 0, s, tok_lp, top_ids, top_lp,
                       static_cast<const float*>(logits), V, row_stride, rows, tokens, K);
  MXS_CHECK_LAUNCH();
}

// Sampling penalties (OpenAI frequency_penalty / presence_penalty, vLLM repetition_penalty),
// applied in place to the logits rows before sampling.  One workgroup per sampled row; rows with
// neutral penalties exit at once (the kernel sits in every decode graph).  The row's token history
// (prompt then generated tokens, written on the device every step) is hist[row, 0:hlen):
//   prompt tokens    -> LDS presence bitmap (V <= 163840 bits = 20 KiB)
//   generated tokens -> per-token counts in a global int32 scratch row (V x 4 B; LDS cannot hold
//                       counts for a 128k-152k vocab), zeroed first, atomics at L2, read back with
//                       atomic loads so no stale L1 line is used
// then for every v:  seen = in prompt or count > 0
//   repetition: z = seen ? (z > 0 ? z / rep : z * rep) : z;   z -= count * freq + (count > 0) * pres
constexpr int kPenMaxVocab = 163840;

template <typename T>
__device__ __forceinline__ void st(T* p, float v);
template <>
__device__ __forceinline__ void st<float>(float* p, float v) { *p = v; }
template <>
__device__ __forceinline__ void st<bf16_t>(bf16_t* p, float v) { *p = f2bf(v); }

template <typename T>
__global__ void __launch_bounds__(1024) penalties_kernel(T* __restrict__ logits, int V, long row_stride,
                                                         const int* __restrict__ hist, long hist_stride,
                                                         const int64_t* __restrict__ srows,
                                                         const int* __restrict__ hlen, const int* __restrict__ plen,
                                                         const float* __restrict__ rep,
                                                         const float* __restrict__ freq,
                                                         const float* __restrict__ pres, int* __restrict__ counts) {
  __shared__ unsigned bits[kPenMaxVocab / 32];
  const int b = blockIdx.x;
  const float rp = rep[b], fp = freq[b], pp = pres[b];
  if (rp == 1.f && fp == 0.f && pp == 0.f) return;
  T* z = logits + b * row_stride;
  int* cnt = counts + static_cast<long>(b) * V;
  const int* h = hist + srows[b] * hist_stride;
  const int n = hlen[b], np = min(plen[b], n);
  for (int w = threadIdx.x; w < (V + 31) / 32; w += blockDim.x) bits[w] = 0u;
  for (int v = threadIdx.x; v < V; v += blockDim.x) cnt[v] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int t = h[i];
    if (t < 0 || t >= V) continue;
    if (i < np)
      atomicOr(&bits[t >> 5], 1u << (t & 31));
    else
      atomicAdd(&cnt[t], 1);
  }
  __syncthreads();
  for (int v = threadIdx.x; v < V; v += blockDim.x) {
    const int c = __hip_atomic_load(&cnt[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool seen = c > 0 || ((bits[v >> 5] >> (v & 31)) & 1u);
    if (!seen) continue;
    float x = ld(z, v);
    if (rp != 1.f) x = x > 0.f ? x / rp : x * rp;
    if (c > 0) x -= static_cast<float>(c) * fp + pp;
    st(z + v, x);
  }
}

void launch_penalties(void* logits, bool bf16, int B, int V, long row_stride, const int* hist, long hist_stride,
                      const int64_t* srows, const int* hlen, const int* plen, const float* rep, const float* freq,
                      const float* pres, int* counts, hipStream_t s) {
  if (B == 0) return;
  if (bf16)
    hipLaunchKernelGGL(penalties_kernel<bf16_t>, dim3(B), dim3(1024), 0, s, static_cast<bf16_t*>(logits), V,
                       row_stride, hist, hist_stride, srows, hlen, plen, rep, freq, pres, counts);
  else
    hipLaunchKernelGGL(penalties_kernel<float>, dim3(B), dim3(1024), 0, s, static_cast<float*>(logits), V, row_stride,
                       hist, hist_stride, srows, hlen, plen, rep, freq, pres, counts);
  MXS_CHECK_LAUNCH();
}

}  // namespace mxs
