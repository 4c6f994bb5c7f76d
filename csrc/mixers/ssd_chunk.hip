// The selective state space of column_scan.h over chunks of 64 tokens on the matrix cores (gfx950): bf16 x, B, C, fp32 state,
// decays and sums.  With c_t the sum of the decay exponents up to token t of the chunk and S the state at its start,
//     y_t   = exp(c_t) S^T C_t + sum_{s <= t} (C_t . B_s) exp(c_t - c_s) dt_s x_s + D x_t
//     S_end = exp(c_64) S      + sum_s exp(c_64 - c_s) dt_s B_s x_s^T
// are four matrix products.  x, B and C enter as they are; what is fp32 (the weights of a (t, s) pair, the state, the weighted
// x) enters in three bf16 pieces, all 24 bits of it, in three products.  c is summed in 64 bits and kept as a multiple of 2^-8
// and a rest, so that a difference is good to fp32 however far the sum has run (an exponent above 128 is a decay of zero).
//
// A wave owns 32 columns of one head's state [N, 32] in its accumulators for the whole walk, where it is the second operand of
// S^T C as it lies, and needs nothing from other waves but the staged tiles: a workgroup is four waves, 128 columns of 1 to 4
// heads of a B/C group, which share the 64 rows of B, C and x in LDS.  The next tile's pieces are in flight in registers under
// the products of the state.  Long chunks are cut into pieces as in column_scan.hip (its modes and its chain).
// Bound by instruction issue (138 matrix instructions a chunk and wave beside some 2,000 others): 4,096 tokens, 64 heads of
// 64, state 128, both passes: 720 us token by token on the vector units, 114 us here.  Error against 64 bits, of a head's outputs /
// its state after 96 tokens, by tokens -> here: half lives of thousands of tokens 3.1e-7 -> 1.25e-7 / 4.3e-7 -> 1.1e-7, of some
// tokens 7.9e-8 -> 7.0e-8 / 8.1e-8 -> 5.9e-8, of a fraction of one 6.6e-8 -> 6.4e-8 / 7.9e-8 -> 5.8e-8.
#include <algorithm>
#include <limits>

#include "mix_common.h"
#include "column_scan.h"

namespace mxs {

typedef __bf16 b8_t __attribute__((ext_vector_type(8)));
typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
typedef short s4_t __attribute__((ext_vector_type(4)));
typedef float f2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef float f16_t __attribute__((ext_vector_type(16)));

namespace {

constexpr int kTok = 64;

// eight fp32 numbers as three bf16 vectors whose sum is the number
struct Split {
  b8_t p[3];
  template <typename F> __device__ __forceinline__ explicit Split(F&& at) {
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      f2_t w = {at(j), at(j + 1)};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const b2_t h = __builtin_convertvector(w, b2_t);
        p[k][j] = h[0];
        p[k][j + 1] = h[1];
        const unsigned u = __builtin_bit_cast(unsigned, h);
        w[0] -= bf2f_lo(u);
        w[1] -= bf2f_hi(u);
      }
    }
  }
};

__device__ __forceinline__ b8_t pair4(s4_t a, s4_t b) {
  return __builtin_bit_cast(b8_t, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}
// entries 0..3 and 8..11 from p on: the order in which an accumulator's rows lie in a lane
__device__ __forceinline__ b8_t row_perm(const bf16_t* p) {
  return pair4(*reinterpret_cast<const s4_t*>(p), *reinterpret_cast<const s4_t*>(p + 8));
}
// the same order down a column of a row-major tile: 16 lanes turn 4 rows x 16 columns (p: the lane's place in them)
__device__ __forceinline__ b8_t col_perm(const bf16_t* p, int pitch) {
  typedef __attribute__((address_space(3))) s4_t* lp;
  return pair4(__builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(p)), __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(p + 8 * pitch)));
}
__device__ __forceinline__ f16_t mm(b8_t a, b8_t b, f16_t c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
typedef unsigned short u2_t __attribute__((ext_vector_type(2)));
// running maximum of 16 bytes of bf16 magnitudes, two by two: 0x7F80 and above are no numbers
__device__ __forceinline__ u2_t widest(u2_t top, const uint4& w) {
  for (const unsigned v : {w.x, w.y, w.z, w.w}) top = __builtin_elementwise_max(top, __builtin_bit_cast(u2_t, v & 0x7FFF7FFFu));
  return top;
}
// softplus(a + b) = max(z, 0) + log(1 + exp(-|z|)) to one rounding: every step keeps what it rounds away.  Everything that a
// token writes and shows goes through this number, so that its error, unlike a sum's, does not average out.  The exponential
// by its series after a whole power of two is taken out, the logarithm as 2 atanh(e / (2 + e)) by its series.
__device__ __forceinline__ float softplus_sum(float a, float b) {
  const float z = a + b, zb = z - a, u = fminf(fabsf(z), 200.f);
  const float zl = u < 200.f ? (a - (z - zb)) + (b - zb) : 0.f, n = rintf(u * -1.44269504f);
  const float r0 = fmaf(n, -0.693145752f, -u);                    // 16 bits of ln 2: exact
  const float r1 = fmaf(n, -1.42860677e-6f, z > 0.f ? -zl : zl);  // and the rest of it
  const float r = r0 + r1, rl = (r0 - r) + r1;
  const float p = r * r * fmaf(r, fmaf(r, fmaf(r, fmaf(r, fmaf(r, fmaf(r, 1.f / 40320, 1.f / 5040), 1.f / 720), 1.f / 120), 1.f / 24), 1.f / 6), 0.5f);
  const float q = p + rl, s = r + q, sl = (r - s) + q, eh = 1.f + s;
  const float e = ldexpf(eh, static_cast<int>(n)), el = ldexpf(((1.f - eh) + s) + sl, static_cast<int>(n));
  const float t = 2.f + e, tl = (e - (t - 2.f)) + el, rc = __builtin_amdgcn_rcpf(t);
  const float h = e * rc, hl = (fmaf(-h, t, e) + fmaf(-h, tl, el)) * rc, h2 = h * h;
  const float k = h2 * fmaf(h2, fmaf(h2, fmaf(h2, fmaf(h2, fmaf(h2, fmaf(h2, fmaf(h2, 1.f / 17, 1.f / 15), 1.f / 13), 1.f / 11), 1.f / 9), 1.f / 7), 1.f / 5), 1.f / 3);
  const float L = 2.f * h, Ll = 2.f * fmaf(h, k, fmaf(hl, h2, hl));
  const float m = z < 0.f ? 0.f : z, y = m + L, yb = y - m;
  return m < 1e30f ? y + ((m - (y - yb)) + (L - yb) + (Ll + (z > 0.f ? zl : 0.f))) : m;
}
// row of accumulator entry i (plus 4 in the upper half of the wave)
__device__ __forceinline__ constexpr int arow(int i) { return 8 * (i / 4) + i % 4; }

}  // namespace

// NT: N / 32.  OUT: outputs are wanted (modes 0 and 2).
template <int NT, bool OUT>
__global__ void __launch_bounds__(256, 2) ssd_chunk_kernel(const ScanArgs p) {
  constexpr int N = 32 * NT, NP = N + 8, XP = 128 + 8;  // rows padded by 16 bytes
  constexpr int NB = kTok * N / 8 / 256, NX = kTok * 128 / 8 / 256;  // 16-byte pieces a thread stages
  __shared__ __attribute__((aligned(16))) bf16_t sB[kTok * NP];
  __shared__ __attribute__((aligned(16))) bf16_t sC[OUT ? kTok * NP : 8];
  __shared__ __attribute__((aligned(16))) bf16_t sX[kTok * XP];
  __shared__ int bad[128];  // per column: the first token so far whose x is no number
  __shared__ __attribute__((aligned(16))) float tok[4][5][kTok];  // per wave: c's multiple and rest, dt, end weight, exp(c)
  const int mode = p.mode, np = p.npieces, P = p.dv, H = p.H;
  const int s = blockIdx.z / np, pc = blockIdx.z - s * np;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, c = lane & 31, hi = lane >> 5;
  const int h0 = blockIdx.x * (128 / P), col0 = wid * 32, hd = h0 + col0 / P, pcol = col0 % P + c;
  int row0 = p.qsl[s];
  if (row0 < 0 || row0 >= p.n_rows) return;
  const int qlen_all = min(p.qsl[s + 1], p.n_rows) - row0;
  const int tb = mode == 0 ? 0 : pc * p.piece, te = mode == 0 ? qlen_all : min(qlen_all, tb + p.piece);
  if (te <= tb) return;
  row0 += tb;
  const int qlen = te - tb, kh = h0 / (H / p.G);
  const long per_head = static_cast<long>(P) * N, sc_at = (static_cast<long>(s) * np + pc) * (H * per_head);
  float* slot = p.state + static_cast<long>(p.state_rows[s]) * p.state_stride + p.off;
  const bool fresh = mode == 1 || (mode == 0 && p.seq_lens[s] - qlen_all <= 0);
  const long mine = (static_cast<long>(hd) * P + pcol) * N + 4 * hi;  // the lane's column, its half's rows
  f16_t S[NT];
  {
    const float* in = (mode == 2 ? p.sc_start + sc_at : slot) + mine;
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        f4_t v = {0.f, 0.f, 0.f, 0.f};
        if (!fresh) v = *reinterpret_cast<const f4_t*>(in + 32 * n + arow(i));
#pragma unroll
        for (int e = 0; e < 4; ++e) S[n][i + e] = v[e];
      }
  }
  const bf16_t* Bp = static_cast<const bf16_t*>(p.k) + kh * N;
  const bf16_t* Cp = static_cast<const bf16_t*>(p.q) + kh * N;
  const bf16_t* Xp = static_cast<const bf16_t*>(p.v) + h0 * P;
  const bf16_t* dtp = static_cast<const bf16_t*>(p.beta) + hd;
  const float eA = expf(p.A_log[hd]), bias = p.dt_bias[hd], Dh = p.D[hd];
  uint4 rB[NB], rC[OUT ? NB : 1], rX[NX];
  float rdt = 0.f;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int id = tid + 256 * i, t = id / (N / 8), at = 8 * (id % (N / 8));
      const bool ok = t0 + t < qlen;
      const long row = row0 + t0 + (ok ? t : 0);
      rB[i] = make_uint4(0, 0, 0, 0);
      if (ok) rB[i] = *reinterpret_cast<const uint4*>(Bp + row * p.k_stride + at);
      if constexpr (OUT) {
        rC[i] = make_uint4(0, 0, 0, 0);
        if (ok) rC[i] = *reinterpret_cast<const uint4*>(Cp + row * p.q_stride + at);
      }
    }
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int id = tid + 256 * i, t = id / 16, at = 8 * (id % 16);
      rX[i] = make_uint4(0, 0, 0, 0);
      if (t0 + t < qlen) rX[i] = *reinterpret_cast<const uint4*>(Xp + (row0 + t0 + t) * p.v_stride + at);
    }
    rdt = t0 + lane < qlen ? bf2f(dtp[(row0 + t0 + lane) * p.beta_stride]) : 0.f;
  };
  if (tid < 128) bad[tid] = std::numeric_limits<int>::max();
  float* my = &tok[wid][0][0];
  double total = 0.0;  // decay exponents of the walk, times log2 e
  fetch(0);
  for (int t0 = 0; t0 < qlen; t0 += kTok) {
    __syncthreads();  // the last tile's reads are done
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int id = tid + 256 * i, at = id / (N / 8) * NP + 8 * (id % (N / 8));
      *reinterpret_cast<uint4*>(sB + at) = rB[i];
      if constexpr (OUT) *reinterpret_cast<uint4*>(sC + at) = rC[i];
    }
    u2_t top = {0, 0};
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int id = tid + 256 * i;
      *reinterpret_cast<uint4*>(sX + id / 16 * XP + 8 * (id % 16)) = rX[i];
      top = widest(top, rX[i]);
    }
    // A weight of zero, which later tokens' x have in a token's sum, makes NaN of an x that is no number.  It goes in as zero,
    // and what its column gives from there on, the state at the end among it, is NaN, as it is token by token.
    if (max(top[0], top[1]) >= 0x7F80) {
#pragma unroll 1
      for (int k = 0; k < 8 * NX; ++k) {
        const int id = tid + 256 * (k / 8), t = id / 16, at = 8 * (id % 16) + k % 8;
        if ((sX[t * XP + at] & 0x7F80) == 0x7F80) {
          sX[t * XP + at] = 0;
          atomicMin(bad + at, t0 + t);
        }
      }
    }
    float eL;
    {  // lane = token
      const bool in = t0 + lane < qlen;
      const float dt = in ? softplus_sum(rdt, bias) : 0.f;
      double cum = in ? -fmin(static_cast<double>(eA) * dt, 128.0) * 1.4426950408889634 : 0.0;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const double up = __shfl_up(cum, o, 64);
        if (lane >= o) cum += up;
      }
      const double end = __shfl(cum, 63, 64), part = rint(cum * 256.0) * (1.0 / 256.0);
      my[lane] = static_cast<float>(part);
      my[kTok + lane] = static_cast<float>(cum - part);
      my[2 * kTok + lane] = dt;
      my[3 * kTok + lane] = __builtin_amdgcn_exp2f(static_cast<float>(end - cum)) * dt;
      my[4 * kTok + lane] = __builtin_amdgcn_exp2f(static_cast<float>(cum));
      eL = __builtin_amdgcn_exp2f(static_cast<float>(end));
      total += end;
    }
    __syncthreads();

    // the wave's columns of x as the second operand, 16 tokens at a time
    const int tr = 4 * hi + ((lane & 15) >> 2), tc = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    b8_t xf[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) xf[j] = col_perm(sX + (16 * j + tr) * XP + col0 + tc, XP);

    const bool two = qlen - t0 > 32;  // the chunk's second half holds tokens
    if constexpr (OUT) {
      f16_t acc[2];
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.f;
      // S^T C
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          __builtin_amdgcn_sched_barrier(0);  // keeps the reads of later steps from piling up in registers
          const Split sp([&](int e) { return S[n][8 * j + e]; });
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            if (t == 1 && !two) continue;
            const b8_t cf = row_perm(sC + (32 * t + c) * NP + 32 * n + 16 * j + 4 * hi);
#pragma unroll
            for (int k = 2; k >= 0; --k) acc[t] = mm(cf, sp.p[k], acc[t]);
          }
        }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
          const f4_t ec = *reinterpret_cast<const f4_t*>(my + 4 * kTok + 32 * t + arow(i) + 4 * hi);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[t][i + e] *= ec[e];
        }
      // pairs within the chunk, s by s tile
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (t == 1 && !two) continue;
        const float ct = my[32 * t + c], rt = my[kTok + 32 * t + c];
#pragma unroll
        for (int u = 0; u <= t; ++u) {
          __builtin_amdgcn_sched_barrier(0);
          f16_t g, g2;  // two sums where the registers hold them: half as many roundings at the size of the whole
          constexpr bool kTwo = NT == 2;
#pragma unroll
          for (int i = 0; i < 16; ++i) g[i] = g2[i] = 0.f;
#pragma unroll
          for (int j = 0; j < 2 * NT; ++j) {
            if (j % 2 == 0) __builtin_amdgcn_sched_barrier(0);
            f16_t& sum = kTwo && j % 2 ? g2 : g;
            sum = mm(row_perm(sB + (32 * u + c) * NP + 16 * j + 4 * hi), row_perm(sC + (32 * t + c) * NP + 16 * j + 4 * hi), sum);
          }
          if constexpr (kTwo) g += g2;
#pragma unroll
          for (int i = 0; i < 16; i += 4) {
            __builtin_amdgcn_sched_barrier(0);
            const int s0 = 32 * u + arow(i) + 4 * hi;
            const f4_t cs = *reinterpret_cast<const f4_t*>(my + s0), rs = *reinterpret_cast<const f4_t*>(my + kTok + s0);
            const f4_t ds = *reinterpret_cast<const f4_t*>(my + 2 * kTok + s0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float m = g[i + e] * (__builtin_amdgcn_exp2f((ct - cs[e]) + (rt - rs[e])) * ds[e]);
              if (u == t) {
                const int d = arow(i) + e + 4 * hi - c;  // s - t
                m = d > 0 ? 0.f : d == 0 ? m + Dh : m;
              }
              g[i + e] = m;
            }
          }
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            __builtin_amdgcn_sched_barrier(0);
            const Split sp([&](int e) { return g[8 * j + e]; });
#pragma unroll
            for (int k = 2; k >= 0; --k) acc[t] = mm(sp.p[k], xf[2 * u + j], acc[t]);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      float* op = p.out + static_cast<long>(row0 + t0 + 4 * hi) * (H * P) + hd * P + pcol;
      const int left = qlen - t0 - 4 * hi, lost = bad[col0 + c] - t0 - 4 * hi;
      if (__builtin_amdgcn_ballot_w64(lost < kTok) != 0) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (32 * t + arow(i) >= lost) acc[t][i] = NAN;
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          if (32 * t + arow(i) < left) op[(32 * t + arow(i)) * (H * P)] = acc[t][i];
        }
    }

    // the state at the chunk's end, under which the next chunk's pieces come in (earlier they would not fit the registers)
    __builtin_amdgcn_sched_barrier(0);
    if (t0 + kTok < qlen) fetch(t0 + kTok);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) S[n][i] *= eL;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j >= 2 && !two) continue;
      __builtin_amdgcn_sched_barrier(0);
      const f4_t w0 = *reinterpret_cast<const f4_t*>(my + 3 * kTok + 16 * j + 4 * hi);
      const f4_t w1 = *reinterpret_cast<const f4_t*>(my + 3 * kTok + 16 * j + 4 * hi + 8);
      const Split sp([&](int e) { return static_cast<float>(xf[j][e]) * (e < 4 ? w0[e & 3] : w1[e & 3]); });
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const b8_t bf = col_perm(sB + (16 * j + tr) * NP + 32 * n + tc, NP);
#pragma unroll
        for (int k = 2; k >= 0; --k) S[n] = mm(bf, sp.p[k], S[n]);
      }
    }
  }
  if (mode == 1 && col0 % P == 0 && lane == 0)  // carries a state across the piece
    p.sc_decay[(static_cast<long>(s) * np + pc) * H + hd] = static_cast<float>(-total * 0.6931471805599453);
  if (mode != 2 || te == qlen_all) {
    const bool lost = bad[col0 + c] < qlen;
    float* o = (mode == 1 ? p.sc_local + sc_at : slot) + mine;
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int i = 0; i < 16; i += 4)
        *reinterpret_cast<f4_t*>(o + 32 * n + arow(i)) = lost ? f4_t{NAN, NAN, NAN, NAN} : f4_t{S[n][i], S[n][i + 1], S[n][i + 2], S[n][i + 3]};
  }
}

// Whole tiles and 16-byte pieces: state 64 or 128, heads of 32, 64 or 128 that fill a workgroup's 128 columns within a group of
// B and C.  From 64 rows and 8 rows a sequence on: a chunk of fewer tokens costs what a full one does.  64 heads of 64, state
// 128, token by token against here: one chunk of 64 tokens 22.4 / 17.7 us; 32 chunks of 16 58 / 35; a chunk beside 32 single
// tokens: of 257 232 / 165, of 400 148 / 111.  Chunks of fewer than 32 tokens only where the heads fill the chip, as token by
// token they are short walks: 16 chunks of 8, 8 heads 8.8 / 13.8, 32 heads 16.7 / 16.3, 64 heads 27.6 / 21.1; 8 of 24, 8 heads
// 12.9 / 13.8, 32 heads 17.9 / 14.9; 8 of 32, 8 heads 14.5 / 14.0.
bool ssd_chunk_fits(const ScanArgs& a, int S) {
  auto al = [](const void* p, long n) { return reinterpret_cast<uintptr_t>(p) % n == 0; };
  const int P = a.dv;
  const int longest = a.max_q > 1 ? a.max_q : a.n_rows - S + 1;
  if (longest < 32 && static_cast<long>(a.n_rows) * a.H * P < 1 << 18) return false;
  if (a.n_rows < 64 || a.n_rows < 8L * S || (a.dk != 64 && a.dk != 128) || (P != 32 && P != 64 && P != 128)) return false;
  if ((a.H / a.G) % (128 / P) != 0) return false;
  return a.k_stride % 8 == 0 && a.q_stride % 8 == 0 && a.v_stride % 8 == 0 && al(a.k, 16) && al(a.q, 16) && al(a.v, 16) &&
         al(a.state, 16) && a.state_stride % 4 == 0 && a.off % 4 == 0 && (a.npieces <= 1 || (al(a.sc_local, 16) && al(a.sc_start, 16)));
}

bool launch_ssd_chunk(const ScanArgs& a, int S, hipStream_t st) {
  const dim3 grid(a.H / (128 / a.dv), 1, S * a.npieces);
  if (grid.z > 65535u) return false;
  if (a.dk == 128) {
    if (a.mode == 1) hipLaunchKernelGGL((ssd_chunk_kernel<4, false>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((ssd_chunk_kernel<4, true>), grid, dim3(256), 0, st, a);
  } else {
    if (a.mode == 1) hipLaunchKernelGGL((ssd_chunk_kernel<2, false>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((ssd_chunk_kernel<2, true>), grid, dim3(256), 0, st, a);
  }
  MXS_CHECK_LAUNCH();
  return true;
}

}  // namespace mxs
