// The gated delta rule of column_scan.h over chunks of 32 tokens (gfx950): bf16 operands, everything else fp32.
//
// With g the decays (per key channel), E_t their product over the chunk's tokens up to t, F_i that of those behind i, S the
// state at the chunk's start and A[t, i], Q[t, i] = sum_d {k, q}_t k_i g_{i+1} .. g_t (the decays of channel d), the writes
// u_t = b_t (v_t - S~_t^T k_t) of a chunk solve
//     u_t + b_t sum_{i < t} A[t, i] u_i = b_t (v_t - S^T (E_t k_t))
// a lower triangle that does not know S.  Its solutions for v and for E k give u = U0 - W S, and with them
//     o = (E q - Q W) S + Q U0,        S_end = E_32 S + sum_i (F_i k_i) u_i^T.
// delta_prepare: a workgroup per chunk and head makes W, U0, E q - Q W, Q U0 (into the outputs) and F k.  A and Q come from
//   products of decays as the token-by-token form has them, never from a quotient: 16 lanes hold the 16 parts of a key, 2 keys
//   each, and walk the tokens.  A thread then solves one of the 128 + 128 columns in its registers.
// delta_walk: a workgroup per head and 16 value columns walks the chunks; each of its four waves holds a quarter of the
//   state's rows and adds its part of W S and (E q - Q W) S (v_mfma_f32_16x16x4_f32; the state is the second operand as the
//   accumulators hold it), the parts meet in LDS over one barrier a chunk.
// Bound by the walk's chain (48 matrix instructions of 32 cycles, a turn through LDS, and one wave a SIMD to hide them).  4,096
// tokens, 16 heads of 128 x 128: 1,480 us token by token (in pieces of 256, each carrying its transition matrix of 128 more
// columns, twice, with library products in between), 432 us here, 156 of them the preparation.  Error against 64 bits, of a
// head's outputs / its state after 96 tokens, by tokens -> here: half lives of a thousand tokens 3.6e-7 -> 1.8e-7 / 4.5e-7 ->
// 2.0e-7, of some tokens 1.36e-7 -> 1.25e-7 / 1.07e-7 -> 1.02e-7, of a tenth of a token 1.21e-7 -> 1.13e-7 / 8.5e-8 -> 7.9e-8.
#include <algorithm>

#include "mix_common.h"
#include "column_scan.h"

namespace mxs {

typedef float f4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int kDC = 32;  // tokens of a chunk

__device__ __forceinline__ float softplus_d(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }
__device__ __forceinline__ float row16(float v) {  // sum over 16 lanes of a DPP row, the same bits in every lane
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, false));
  return v;
}
// What scales a whole row is not rounded before it does, or once: a chunk's sums round a little more often than a walk by tokens,
// and where decays are fast, so that nothing else is left, that was 2 to 7 % of the error.
__device__ __forceinline__ double unit_of(float square, float scale) { return static_cast<double>(scale) / sqrt(static_cast<double>(square)); }
__device__ __forceinline__ float strength(float z) { return static_cast<float>(1.0 / (1.0 + exp(-static_cast<double>(z)))); }
// a barrier for LDS alone: __syncthreads would wait for the loads of the chunks to come as well
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// R neighbouring elements as fp32
template <int R> __device__ __forceinline__ void run_of(const bf16_t* p, float* o, bool vec) {
  if (vec && R == 8) {
    load16(p, o);
  } else if (vec) {
    const uint2 a = *reinterpret_cast<const uint2*>(p);
    o[0] = bf2f_lo(a.x); o[1] = bf2f_hi(a.x); o[2] = bf2f_lo(a.y); o[3] = bf2f_hi(a.y);
  } else {
#pragma unroll
    for (int i = 0; i < R; ++i) o[i] = bf2f(p[i]);
  }
}

// what delta_prepare leaves of a (chunk, head): offsets in floats
template <int DK> struct Slab {
  static constexpr int W = 0, Q = kDC * DK, K = 2 * kDC * DK, E = 3 * kDC * DK, U = 3 * kDC * DK + DK;
  static __host__ __device__ long size(int dv) { return U + static_cast<long>(kDC) * dv; }
};
// first slab row of a sequence whose first row is row0: chunks of earlier ones never reach it
__device__ __forceinline__ int first_chunk(int row0, int s) { return row0 / kDC + s; }

}  // namespace

template <int DK>
__global__ void __launch_bounds__(256) delta_prepare_kernel(const ScanArgs p, float* __restrict__ work, int S, int flags) {
  constexpr int R = DK / 16;
  __shared__ __attribute__((aligned(16))) float ks[kDC][DK], qs[kDC][DK], gs[kDC][DK], ls[kDC][DK];  // gs = exp(-ls)
  __shared__ __attribute__((aligned(16))) float As[kDC][kDC], Qs[kDC][kDC];
  __shared__ float bs[kDC];
  const int tid = threadIdx.x, hd = blockIdx.x, slot = blockIdx.y, H = p.H, dv = p.dv, kh = hd / (H / p.G);
  int s;
  {
    int lo = 0, hi = S - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (first_chunk(p.qsl[mid], mid) <= slot) lo = mid; else hi = mid - 1;
    }
    s = lo;
  }
  int row0 = p.qsl[s];
  if (row0 < 0 || row0 >= p.n_rows) return;
  const int qlen = min(p.qsl[s + 1], p.n_rows) - row0, t0 = (slot - first_chunk(row0, s)) * kDC;
  if (t0 < 0 || t0 >= qlen) return;
  row0 += t0;
  const int nt = min(kDC, qlen - t0);
  const int part = tid & 15, grp = tid >> 4;
  const float eA = expf(p.A_log[hd]);
  // unit keys and queries, decays
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int t = grp + 16 * h;
    const long row = row0 + min(t, nt - 1);
    float k[R], q[R], a[R], sk = 0.f, sq = 0.f;
    run_of<R>(static_cast<const bf16_t*>(p.k) + row * p.k_stride + kh * DK + part * R, k, flags & 1);
    run_of<R>(static_cast<const bf16_t*>(p.q) + row * p.q_stride + kh * DK + part * R, q, flags & 2);
    run_of<R>(static_cast<const bf16_t*>(p.a) + row * p.a_stride + hd * DK + part * R, a, flags & 4);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      sk += k[i] * k[i];
      sq += q[i] * q[i];
    }
    const bool in = t < nt;
    const double ik = unit_of(row16(sk) + p.unit_eps, 1.f), iq = unit_of(row16(sq) + p.unit_eps, p.q_scale);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int d = part * R + i;
      ks[t][d] = in ? static_cast<float>(k[i] * ik) : 0.f;
      qs[t][d] = in ? static_cast<float>(q[i] * iq) : 0.f;
      const float l = in ? eA * softplus_d(a[i] + p.dt_bias[hd * DK + d]) : 0.f;
      ls[t][d] = l;
      gs[t][d] = expf(-l);
    }
    if (part == 0) bs[t] = in ? strength(bf2f(static_cast<const bf16_t*>(p.beta)[row * p.beta_stride + hd])) : 0.f;
  }
  __syncthreads();
  {  // A and Q of keys grp and grp + 16
    float w0[R], w1[R];
#pragma unroll
    for (int i = 0; i < R; ++i) w0[i] = w1[i] = 0.f;
    for (int t = 0; t < nt; ++t) {
      float g[R], k[R], q[R];
#pragma unroll
      for (int i = 0; i < R; i += 4) {
        *reinterpret_cast<f4_t*>(g + i) = *reinterpret_cast<const f4_t*>(&gs[t][part * R + i]);
        *reinterpret_cast<f4_t*>(k + i) = *reinterpret_cast<const f4_t*>(&ks[t][part * R + i]);
        *reinterpret_cast<f4_t*>(q + i) = *reinterpret_cast<const f4_t*>(&qs[t][part * R + i]);
      }
      float sa[2] = {0.f, 0.f}, sq[2] = {0.f, 0.f}, a1 = 0.f, q1 = 0.f;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        w0[i] = t == grp ? k[i] : w0[i] * g[i];  // zero before the key's own token
        sa[i & 1] += w0[i] * k[i];
        sq[i & 1] += w0[i] * q[i];
      }
      const float a0 = row16(sa[0] + sa[1]), q0 = row16(sq[0] + sq[1]);
      if (t >= 16) {
        sa[0] = sa[1] = sq[0] = sq[1] = 0.f;
#pragma unroll
        for (int i = 0; i < R; ++i) {
          w1[i] = t == grp + 16 ? k[i] : w1[i] * g[i];
          sa[i & 1] += w1[i] * k[i];
          sq[i & 1] += w1[i] * q[i];
        }
        a1 = row16(sa[0] + sa[1]);
        q1 = row16(sq[0] + sq[1]);
      }
      if (part == 0) {
        As[t][grp] = a0;
        Qs[t][grp] = q0;
        As[t][grp + 16] = a1;
        Qs[t][grp + 16] = q1;
      }
    }
  }
  for (int t = nt + grp; t < kDC; t += 16) {  // rows that no token has
    As[t][2 * part] = As[t][2 * part + 1] = 0.f;
    Qs[t][2 * part] = Qs[t][2 * part + 1] = 0.f;
  }
  __syncthreads();
  float* mine = work + (static_cast<long>(slot) * H + hd) * Slab<DK>::size(dv);
  const bool keys = tid >= 128;
  const int col = tid & 127;
  if (keys ? col >= DK : col >= std::max(dv, DK)) return;  // no barrier below
  if (keys || col < dv) {
    float x[kDC];
    if (keys) {
      float e = 0.f;  // sums of the exponents: one rounding for a product of decays, however many tokens it spans
#pragma unroll
      for (int t = 0; t < kDC; ++t) {
        e += ls[t][col];
        x[t] = ks[t][col] * expf(-e);
      }
      mine[Slab<DK>::E + col] = expf(-e);
    } else {
      const bf16_t* vp = static_cast<const bf16_t*>(p.v) + hd * dv + col;
#pragma unroll
      for (int t = 0; t < kDC; ++t) x[t] = bf2f(vp[(row0 + min(t, nt - 1)) * p.v_stride]);  // past the last: bs is zero
    }
    int z = 0;
#pragma unroll
    for (int t = 0; t < kDC; ++t) {
      // a row's coefficients are read two rows ahead and no earlier: all of them would fill the registers twice
      asm volatile("" : "+v"(z) : "v"(x[t < 2 ? 0 : t - 2]));
      float r[4] = {0.f, 0.f, 0.f, 0.f};  // the sum apart: small terms first, one rounding at the size of the value
#pragma unroll
      for (int i = 0; i < t; i += 4) {
        const f4_t a = *reinterpret_cast<const f4_t*>(&As[t][i + z]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (i + e < t) r[e] += a[e] * x[i + e];
      }
      x[t] = t < nt ? bs[t] * (x[t] - ((r[0] + r[1]) + (r[2] + r[3]))) : 0.f;
    }
    asm volatile("" ::: "memory");  // decays and keys are read again: kept, they would not fit the registers
    float e = 0.f;
#pragma unroll
    for (int t = 0; t < kDC; ++t) {
      asm volatile("" : "+v"(z) : "v"(e));
      float r[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i <= t; i += 4) {
        const f4_t a = *reinterpret_cast<const f4_t*>(&Qs[t][i + z]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (i + j <= t) r[j] += a[j] * x[i + j];
      }
      const float y = (r[0] + r[1]) + (r[2] + r[3]);
      if (keys) {
        e += ls[t][col];
        mine[Slab<DK>::W + t * DK + col] = x[t];
        mine[Slab<DK>::Q + t * DK + col] = qs[t][col] * expf(-e) - y;
      } else if (t < nt) {
        p.out[static_cast<long>(row0 + t) * (H * dv) + hd * dv + col] = y;
      }
    }
    if (!keys) {  // 16 columns as an accumulator holds them: lane 16 (t % 16 / 4) + column, entry t % 4
      float* u = mine + Slab<DK>::U + (col / 16) * (kDC * 16) + (col % 16) * 4;
#pragma unroll
      for (int t = 0; t < kDC; t += 4) *reinterpret_cast<f4_t*>(u + t * 16) = f4_t{x[t], x[t + 1], x[t + 2], x[t + 3]};
    }
  }
  asm volatile("" ::: "memory");
  if (!keys && col < DK) {
    float f = 0.f;
    float* kp = mine + Slab<DK>::K + col * kDC;
#pragma unroll
    for (int t = kDC - 4; t >= 0; t -= 4) {
      f4_t v;
#pragma unroll
      for (int e = 3; e >= 0; --e) {
        v[e] = ks[t + e][col] * expf(-f);
        f += ls[t + e][col];
      }
      *reinterpret_cast<f4_t*>(kp + t) = v;
    }
  }
}

template <int DK>
__global__ void __launch_bounds__(256, 1) delta_walk_kernel(const ScanArgs p, const float* __restrict__ work) {
  constexpr int DT = DK / 64;  // tiles of 16 state rows a wave holds
  __shared__ __attribute__((aligned(16))) float lds[2][4][2][2][64][4];  // parity, wave, U | O, token tile, lane, entry
  const int hd = blockIdx.x, cb = blockIdx.y, s = blockIdx.z, H = p.H, dv = p.dv;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = lane & 15, qd = lane >> 4;
  const int row0 = p.qsl[s];
  if (row0 < 0 || row0 >= p.n_rows) return;
  const int qlen = min(p.qsl[s + 1], p.n_rows) - row0;
  if (qlen <= 0) return;
  float* slot = p.state + static_cast<long>(p.state_rows[s]) * p.state_stride + p.off +
                (static_cast<long>(hd) * dv + cb * 16 + c) * DK + w * (DK / 4) + 4 * qd;
  f4_t St[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) {
    St[d] = f4_t{0.f, 0.f, 0.f, 0.f};
    if (p.seq_lens[s] - qlen > 0) St[d] = *reinterpret_cast<const f4_t*>(slot + 16 * d);
  }
  const long size = Slab<DK>::size(dv);
  const float* slab = work + (static_cast<long>(first_chunk(row0, s)) * H + hd) * size;
  struct Piece {  // what a wave reads of a chunk
    f4_t w[2][DT], q[2][DT], k[DT][2], e[DT], u[2];
    float o[2];
  };
  const int orow = 8 * w + (lane >> 3), ocol = 2 * (lane & 7);  // of the outputs this lane writes
  float* op = p.out + static_cast<long>(row0 + orow) * (H * dv) + hd * dv + cb * 16 + ocol;
  const int nchunk = (qlen + kDC - 1) / kDC;
  // the loads stand in no branch (past the last chunk that one again): a wait then counts those that came after its own
  auto fetch = [&](Piece& b, int i0) {
    i0 = min(i0, nchunk - 1);
    const float* at = slab + static_cast<long>(i0) * (H * size);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        const int i = (16 * t + c) * DK + w * (DK / 4) + 16 * d + 4 * qd;
        b.w[t][d] = *reinterpret_cast<const f4_t*>(at + Slab<DK>::W + i);
        b.q[t][d] = *reinterpret_cast<const f4_t*>(at + Slab<DK>::Q + i);
        b.k[d][t] = *reinterpret_cast<const f4_t*>(at + Slab<DK>::K + (w * (DK / 4) + 16 * d + c) * kDC + 16 * t + 4 * qd);
      }
#pragma unroll
    for (int d = 0; d < DT; ++d) b.e[d] = *reinterpret_cast<const f4_t*>(at + Slab<DK>::E + w * (DK / 4) + 16 * d + 4 * qd);
#pragma unroll
    for (int t = 0; t < 2; ++t) b.u[t] = *reinterpret_cast<const f4_t*>(at + Slab<DK>::U + cb * (kDC * 16) + t * 256 + lane * 4);
    const float* o = op + static_cast<long>(min(i0 * kDC, qlen - 1 - orow)) * (H * dv);  // rows past the last: that one
    b.o[0] = o[0];
    b.o[1] = o[1];
  };
  auto step = [&](const Piece& b, int i0, int par) {
    const int t0 = i0 * kDC;
    f4_t u[2], us[2][DT], os[2][DT];  // short sums: their roundings are fewer
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int d = 0; d < DT; ++d) us[t][d] = os[t][d] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          us[t][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.w[t][d][r], St[d][r], us[t][d], 0, 0, 0);
          os[t][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.q[t][d][r], St[d][r], os[t][d], 0, 0, 0);
        }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f4_t su = us[t][0], so = os[t][0];
#pragma unroll
      for (int d = 1; d < DT; ++d) {
        su += us[t][d];
        so += os[t][d];
      }
      *reinterpret_cast<f4_t*>(&lds[par][w][0][t][lane][0]) = su;
      *reinterpret_cast<f4_t*>(&lds[par][w][1][t][lane][0]) = so;
    }
#pragma unroll
    for (int d = 0; d < DT; ++d) St[d] *= b.e[d];
    lds_barrier();  // the one of a chunk: the other parity's sums are read before this and written after it
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f4_t part[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) part[v] = *reinterpret_cast<const f4_t*>(&lds[par][v][0][t][lane][0]);
      u[t] = b.u[t] - ((part[0] + part[1]) + (part[2] + part[3]));
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int d = 0; d < DT; ++d) St[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.k[d][t][r], u[t][r], St[d], 0, 0, 0);
    if (t0 + orow < qlen) {  // row orow = entry orow % 4 of lanes 16 (orow % 16 / 4) + column
      const int l = 16 * (orow % 16 / 4) + ocol;
      float x[4], y[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        x[v] = lds[par][v][1][orow / 16][l][orow & 3];
        y[v] = lds[par][v][1][orow / 16][l + 1][orow & 3];
      }
      float* o = op + static_cast<long>(t0) * (H * dv);
      o[0] = b.o[0] + ((x[0] + x[1]) + (x[2] + x[3]));
      o[1] = b.o[1] + ((y[0] + y[1]) + (y[2] + y[3]));
    }
  };
  // three chunks are on their way or in work: a chunk takes less than its loads
  Piece b[3];
  int i0 = 0, par = 0;
  if (nchunk >= 3) {
    fetch(b[0], 0);
    fetch(b[1], 1);
    for (; i0 + 3 <= nchunk; i0 += 3) {
#pragma unroll
      for (int i = 0; i < 3; ++i, par ^= 1) {
        fetch(b[(i + 2) % 3], i0 + i + 2);
        step(b[i], i0 + i, par);
      }
    }
  } else {
    fetch(b[0], 0);
    if (nchunk > 1) fetch(b[1], 1);
  }
  if (i0 < nchunk) step(b[0], i0, par);
  if (i0 + 1 < nchunk) step(b[1], i0 + 1, par ^ 1);
#pragma unroll
  for (int d = 0; d < DT; ++d) *reinterpret_cast<f4_t*>(slot + 16 * d) = St[d];
}

// floats of scratch per (chunk, head), 0: sizes that these kernels do not hold.  Chunks: T / 32 + sequences.
long delta_chunk_floats(int dk, int dv) {
  if ((dk != 64 && dk != 128) || dv % 16 != 0 || dv < 16 || dv > 128) return 0;
  return dk == 64 ? Slab<64>::size(dv) : Slab<128>::size(dv);
}

bool launch_delta_chunk(const ScanArgs& a, int S, float* work, hipStream_t st) {
  auto al = [](const void* p, long n) { return reinterpret_cast<uintptr_t>(p) % n == 0; };
  if (!al(a.state, 16) || a.state_stride % 4 != 0 || a.off % 4 != 0 || !al(work, 16)) return false;
  const int slots = a.n_rows / kDC + S;
  if (S > 65535 || slots > 65535) return false;
  const int R = a.dk / 16;
  auto run = [&](const void* p, long stride) { return al(p, 2 * R) && stride % R == 0; };
  const int flags = (run(a.k, a.k_stride) ? 1 : 0) | (run(a.q, a.q_stride) ? 2 : 0) | (run(a.a, a.a_stride) ? 4 : 0);
  const dim3 prep(a.H, slots), walk(a.H, a.dv / 16, S);  // a head's workgroups on one chiplet where 8 divides H: its slabs are in one L2
  if (a.dk == 128) {
    hipLaunchKernelGGL(delta_prepare_kernel<128>, prep, dim3(256), 0, st, a, work, S, flags);
    hipLaunchKernelGGL(delta_walk_kernel<128>, walk, dim3(256), 0, st, a, work);
  } else {
    hipLaunchKernelGGL(delta_prepare_kernel<64>, prep, dim3(256), 0, st, a, work, S, flags);
    hipLaunchKernelGGL(delta_walk_kernel<64>, walk, dim3(256), 0, st, a, work);
  }
  MXS_CHECK_LAUNCH();
  return true;
}

}  // namespace mxs
