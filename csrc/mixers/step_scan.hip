// The recurrences of column_scan.h for steps of single tokens (gfx950): a read and a write of the state and little else.
//
// A column of the state (one value's dk entries, back to back in memory) belongs to dk / 4 neighbouring lanes with 16 bytes
// each, so that a wave's access is one whole stretch of memory; a wave holds eight of those and works alone: its key, query
// and decays are four entries a lane, sums go over the column's lanes, and there is neither LDS nor a barrier.  Bound by the
// state's bytes: 64 sequences, 64 heads of 64 x 128 (268 MB both ways): 99 us in the staged form of column_scan.hip, which
// reads 32 bytes a lane in halves and waits for its workgroup, 51 us here; delta rule, 16 heads of 128 x 128 (134 MB): 72 and
// 32 us.
#include <algorithm>
#include <type_traits>

#include "mix_common.h"
#include "column_scan.h"

namespace mxs {

typedef float f4_t __attribute__((ext_vector_type(4)));

namespace {

__device__ __forceinline__ float softplus_s(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

// sum over L neighbouring lanes, the same bits in each
template <int L> __device__ __forceinline__ float lanes_sum(float v) {
  if constexpr (L >= 16) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, false));
    if constexpr (L >= 32) v += __shfl_xor(v, 16, 64);
    if constexpr (L >= 64) v += __shfl_xor(v, 32, 64);
  } else {
#pragma unroll
    for (int o = 1; o < L; o <<= 1) v += __shfl_xor(v, o, 64);
  }
  return v;
}

struct Four {
  float v[4];
  __device__ __forceinline__ float& operator[](int i) { return v[i]; }
  __device__ __forceinline__ float operator[](int i) const { return v[i]; }
};
__device__ __forceinline__ Four four(const bf16_t* p, bool vec) {
  if (vec) {
    const uint2 a = *reinterpret_cast<const uint2*>(p);
    return Four{{bf2f_lo(a.x), bf2f_hi(a.x), bf2f_lo(a.y), bf2f_hi(a.y)}};
  }
  return Four{{bf2f(p[0]), bf2f(p[1]), bf2f(p[2]), bf2f(p[3])}};
}
__device__ __forceinline__ Four four(const float* p, bool vec) {
  if (vec) {
    const f4_t a = *reinterpret_cast<const f4_t*>(p);
    return Four{{a[0], a[1], a[2], a[3]}};
  }
  return Four{{p[0], p[1], p[2], p[3]}};
}
__device__ __forceinline__ float dot4(const Four& a, const Four& b) { return (a[0] * b[0] + a[1] * b[1]) + (a[2] * b[2] + a[3] * b[3]); }

}  // namespace

constexpr int kStepCols = 8;  // columns of a lane

template <typename T, int KIND, int L>
__global__ void __launch_bounds__(256, 4) step_scan_kernel(const ScanArgs p, int flags) {
  constexpr int PER = 64 / L, CW = kStepCols * PER, DK = 4 * L;  // columns of an access, of a wave
  constexpr bool DELTA = KIND == kDeltaRule, GLA = KIND == kGatedLinear;
  using A = typename std::conditional<GLA, float, T>::type;
  const int s = blockIdx.y, lane = threadIdx.x & 63, part = lane % L, H = p.H, dv = p.dv;
  const int nb = (dv + CW - 1) / CW, unit = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= H * nb) return;
  const int hd = unit / nb, c0 = (unit - hd * nb) * CW + lane / L;  // the lane's first column; the next is PER on
  int row = p.qsl[s];
  if (row < 0 || row >= p.n_rows) return;
  const int qlen = min(p.qsl[s + 1], p.n_rows) - row;
  if (qlen <= 0) return;
  float* slot = p.state + static_cast<long>(p.state_rows[s]) * p.state_stride + p.off + (static_cast<long>(hd) * dv + c0) * DK + 4 * part;
  const bool fresh = p.seq_lens[s] - qlen <= 0;
  Four S[kStepCols];
#pragma unroll
  for (int i = 0; i < kStepCols; ++i) {
    S[i] = Four{{0.f, 0.f, 0.f, 0.f}};
    if (!fresh && c0 + i * PER < dv) S[i] = four(slot + static_cast<long>(i) * PER * DK, true);
  }
  const int kh = hd / (H / p.G);
  const T* kp = static_cast<const T*>(p.k) + kh * DK + 4 * part;
  const T* qp = static_cast<const T*>(p.q) + kh * DK + 4 * part;
  const T* vp = static_cast<const T*>(p.v) + hd * dv;
  const A* ap = static_cast<const A*>(p.a) + (KIND != kStateSpace ? hd * DK + 4 * part : 0);
  const float eA = GLA ? 0.f : expf(p.A_log[hd]);
#pragma unroll 1
  for (const int end = row + qlen; row < end; ++row) {
    Four k = four(kp + row * p.k_stride, flags & 1), q = four(qp + row * p.q_stride, flags & 2), g = {{0.f, 0.f, 0.f, 0.f}};
    float v[kStepCols], o[kStepCols];
#pragma unroll
    for (int i = 0; i < kStepCols; ++i) v[i] = ldf(vp + row * p.v_stride + min(c0 + i * PER, dv - 1));
    if constexpr (KIND != kStateSpace) g = four(ap + row * p.a_stride, flags & 4);
    if constexpr (DELTA) {
      const float b = sigmoid_f(ldf(static_cast<const T*>(p.beta) + row * p.beta_stride + hd));
      const float ik = rsqrtf(lanes_sum<L>(dot4(k, k)) + p.unit_eps), iq = rsqrtf(lanes_sum<L>(dot4(q, q)) + p.unit_eps) * p.q_scale;
      const Four bias = four(p.dt_bias + hd * DK + 4 * part, false);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        k[e] *= ik;
        q[e] *= iq;
        g[e] = expf(-eA * softplus_s(g[e] + bias[e]));
      }
#pragma unroll
      for (int i = 0; i < kStepCols; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) S[i][e] *= g[e];
        const float u = b * (v[i] - lanes_sum<L>(dot4(S[i], k)));
#pragma unroll
        for (int e = 0; e < 4; ++e) S[i][e] += k[e] * u;
        o[i] = lanes_sum<L>(dot4(S[i], q));
      }
    } else if constexpr (GLA) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        g[e] = expf(g[e]);
        q[e] *= p.q_scale;
      }
#pragma unroll
      for (int i = 0; i < kStepCols; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) S[i][e] = g[e] * S[i][e] + k[e] * v[i];
        o[i] = lanes_sum<L>(dot4(S[i], q));
      }
    } else {
      const float dt = softplus_s(ldf(static_cast<const T*>(p.beta) + row * p.beta_stride + hd) + p.dt_bias[hd]);
      const float a = expf(-eA * dt), D = p.D[hd];
#pragma unroll
      for (int i = 0; i < kStepCols; ++i) {
        const float x = dt * v[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) S[i][e] = a * S[i][e] + k[e] * x;
        o[i] = lanes_sum<L>(dot4(S[i], q)) + D * v[i];
      }
    }
    float mine = 0.f;  // lane `part` of a column's lanes writes column i = part
#pragma unroll
    for (int i = 0; i < kStepCols; ++i) mine = part == i ? o[i] : mine;
    const int col = c0 + part * PER;
    if (part < kStepCols && col < dv) p.out[static_cast<long>(row) * (H * dv) + hd * dv + col] = mine;
  }
#pragma unroll
  for (int i = 0; i < kStepCols; ++i)
    if (c0 + i * PER < dv) *reinterpret_cast<f4_t*>(slot + static_cast<long>(i) * PER * DK) = f4_t{S[i][0], S[i][1], S[i][2], S[i][3]};
}

template <typename T, int KIND>
static bool launch_step(const ScanArgs& a, int S, hipStream_t st) {
  if (reinterpret_cast<uintptr_t>(a.state) % 16 != 0 || a.state_stride % 4 != 0 || a.off % 4 != 0 || S > 65535) return false;
  auto fits = [&](const void* p, long stride, size_t e) { return reinterpret_cast<uintptr_t>(p) % (4 * e) == 0 && stride % 4 == 0; };
  const int flags = (fits(a.k, a.k_stride, sizeof(T)) ? 1 : 0) | (fits(a.q, a.q_stride, sizeof(T)) ? 2 : 0) |
                    (KIND != kStateSpace && fits(a.a, a.a_stride, KIND == kGatedLinear ? 4 : sizeof(T)) ? 4 : 0);
#define MIX_STEP(L)                                                                                                    \
  do {                                                                                                                 \
    const int cw = kStepCols * (64 / L), units = a.H * ((a.dv + cw - 1) / cw);                                         \
    hipLaunchKernelGGL((step_scan_kernel<T, KIND, L>), dim3((units + 3) / 4, S), dim3(256), 0, st, a, flags);          \
  } while (0)
  if (a.dk == 32) MIX_STEP(8);
  else if (a.dk == 64) MIX_STEP(16);
  else if (a.dk == 128) MIX_STEP(32);
  else if (a.dk == 256) MIX_STEP(64);
  else return false;
#undef MIX_STEP
  MXS_CHECK_LAUNCH();
  return true;
}

bool launch_step_scan(const ScanArgs& a, int S, int kind, bool bf, hipStream_t st) {
  if (kind == kDeltaRule) return bf ? launch_step<bf16_t, kDeltaRule>(a, S, st) : launch_step<float, kDeltaRule>(a, S, st);
  if (kind == kGatedLinear) return bf ? launch_step<bf16_t, kGatedLinear>(a, S, st) : launch_step<float, kGatedLinear>(a, S, st);
  return bf ? launch_step<bf16_t, kStateSpace>(a, S, st) : launch_step<float, kStateSpace>(a, S, st);
}

}  // namespace mxs
