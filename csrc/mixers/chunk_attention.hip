// Softmax attention of prompt chunks on the 32-wide matrix instructions (gfx950), bf16 keys and values, fp32 scores,
// weights and sums.
//
// A workgroup serves 128 (query, head) pairs of one kv head: the query heads of a kv head lie side by side, so that the
// columns of a tile are full for single rows too and a key tile is staged once for all of them.  Its four waves hold 32
// pairs each and walk the visible keys together, in tiles of KT through two LDS buffers: the next tile's 16-byte pieces
// are in flight in registers under the current tile's products.  Per 32 keys and wave:
//   S^T = K Q^T  (v_mfma_f32_32x32x16_bf16)  A = key rows from LDS (16-byte reads), B = Q^T in registers.  A lane holds 16
//                keys of one query: maximum and sum are its own work plus one exchange with the lane 32 away.
//   O^T += V^T P^T   B = P^T as the accumulator leaves it, every weight in two bf16 halves (p = hi + lo, two products: 16
//                mantissa bits of the fp32 weight); A = V^T straight from the token-major rows through the transposing
//                LDS read (ds_read_b64_tr_b16: 16 lanes turn 4 keys x 16 values), in the key order that the accumulator has.
// Bound by instruction issue: for 64-wide heads a 64-key tile costs a wave about 270 vector instructions, 32 of them
// exponentials, and 24 matrix instructions, and the two kinds hardly overlap (interleaving them by hand, four waves a SIMD,
// walks paired long with short, and walks that begin at different keys all measured the same or slower).
// 4,096 rows, 32 heads of 64 over 8 kv heads: 1,127 us with one wave per 16 rows of a head on the 16-wide instructions and
// 2-byte reads of V (the form that this one replaced), 125 us; window 1,024: 72 us; 16 heads of 128: 192 us.  Keys of 128 + 64
// and values of 128 expanded from latent rows of 576, 16 heads, 4,096 rows: 189 us and 50 us for gathering and expanding, against
// 1,142 us over the rows themselves with folded queries.
#include "chunk_attention.h"
#include "chunk_walk.h"
#include "mix_common.h"

#include <algorithm>

namespace mxs {

typedef __bf16 b8_t __attribute__((ext_vector_type(8)));
typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
typedef short s4_t __attribute__((ext_vector_type(4)));
typedef float f2_t __attribute__((ext_vector_type(2)));
typedef float f16_t __attribute__((ext_vector_type(16)));

// plain v_max: fmaxf on a matrix instruction's result makes the compiler canonicalise its operands first
__device__ __forceinline__ float vmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float vmax3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float across(float v, bool sum) {  // with the lane 32 away
  const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  const float a = __uint_as_float(sw[0]), b = __uint_as_float(sw[1]);
  return sum ? a + b : fmaxf(a, b);
}

constexpr int kSplitKeys = 768;  // shorter walks are one stretch's alone

// DKP, DVP: head sizes the registers are laid out for (smaller ones ride in zeroed columns); KT: keys of a tile; PAGED:
// where keys and values are; WHOLE: a third piece of every weight, all 24 bits.
template <int DKP, int DVP, int KT, bool PAGED, bool SPLIT, bool WHOLE>
__global__ void __launch_bounds__(256, DKP + DVP <= 128 ? 3 : 2) chunk_attention_kernel(ChunkArgs a) {
  constexpr int KS = DKP / 16, DT = DVP / 32, KU = KT / 32;
  constexpr int KROW = DKP + 8, VROW = DVP + 8;  // padded by 16 bytes: neighbouring rows start in other banks
  constexpr int NK = KT * DKP / 8 / 256, NV = KT * DVP / 8 / 256;  // 16-byte pieces a thread stages
  static_assert(NK * 256 * 8 == KT * DKP && NV * 256 * 8 == KT * DVP, "tile");
  __shared__ __attribute__((aligned(16))) bf16_t lds[2][KT * (KROW + VROW)];
  const int g = blockIdx.x, s = SPLIT ? blockIdx.z / a.nsplit : blockIdx.z, stretch = SPLIT ? blockIdx.z - s * a.nsplit : 0;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int c = lane & 31, hi = lane >> 5;
  const int row0 = a.qsl[s], qlen = a.qsl[s + 1] - row0;
  const int R = a.H / a.G;
  const int npairs = qlen * R, tile = gridDim.y - 1 - blockIdx.y, first = tile * 128;  // the longest walks first
  if (first >= npairs) return;
  const int past = max(a.seq_lens[s] - qlen, 0);
  const int dk = a.dk, dv = a.dv;
  // pairs and positions of the workgroup, the wave, the lane
  const int glast = past + (min(first + 128, npairs) - 1) / R;
  const int wfirst = first + wid * 32;
  const bool live = wfirst < npairs;  // a wave without pairs stages and waits with the others
  const int wlo = past + min(wfirst, npairs - 1) / R, whi = past + min(wfirst + 31, npairs - 1) / R;
  const int pair = min(wfirst + c, npairs - 1);
  const bool qok = wfirst + c < npairs;
  const int qi = pair / R, head = g * R + (pair - qi * R), pos = past + qi;

  // what this thread stages of a tile: a wave takes a page of 16 keys (or half of one), its base is uniform and the lane's
  // pieces stay where they are inside it
  constexpr int PT = KT / 16, WPP = 4 / PT;  // pages a tile, waves a page
  const int wv = __builtin_amdgcn_readfirstlane(wid), wpage = wv / WPP;
  const int kpr = dk >> 3, vpr = dv >> 3;  // pieces a row
  int krow[NK], vrow[NV], kat[NK], vat[NV];  // row inside the page (-1: none), place in LDS
  int kfrom[NK], vfrom[NV];                  // element offset from the page's base
  bool kown[NK];                             // of a key in rows: the head's own part
#pragma unroll
  for (int i = 0; i < NK; ++i) {
    const int idx = lane + 64 * (i * WPP + wv % WPP), r = idx / kpr, col = 8 * (idx - r * kpr);
    krow[i] = r < 16 ? r : -1;
    kat[i] = (wpage * 16 + r) * KROW + col;
    kfrom[i] = PAGED ? 8 * idx : col < a.dn ? r * static_cast<int>(a.x_stride) + col : r * static_cast<int>(a.r_stride) + col - a.dn;
    kown[i] = col < a.dn;
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int idx = lane + 64 * (i * WPP + wv % WPP), r = idx / vpr, col = 8 * (idx - r * vpr);
    vrow[i] = r < 16 ? r : -1;
    vat[i] = KT * KROW + (wpage * 16 + r) * VROW + col;
    vfrom[i] = PAGED ? 8 * idx : r * static_cast<int>(a.x_stride) + col;
  }
  if (dk < DKP || dv < DVP) {  // columns that no piece ever writes
    for (int i = tid; i < 2 * KT * (KROW + VROW) / 8; i += 256) reinterpret_cast<uint4*>(&lds[0][0])[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();
  }

  const ChunkWalk walk = chunk_walk(past + first / R, glast, a.window, a.keep, KT);
  const int ntile = walk.ntile;
  auto start_of = [&](int it) { return walk.start(it); };

  // this workgroup's tiles: all, or its stretch of a long walk (short walks are the first stretch's alone)
  int it0 = 0, itn = ntile;
  float* pp = nullptr;
  if constexpr (SPLIT) {
    pp = a.part + ((static_cast<long>(row0 + qi) * a.H + head) * a.nsplit + stretch) * (dv + 4);
    if (ntile * KT >= kSplitKeys) {
      it0 = ntile * stretch / a.nsplit;
      itn = ntile * (stretch + 1) / a.nsplit;
    } else if (stretch > 0) {
      if (qok && hi == 0) {
        pp[0] = -INFINITY;
        pp[1] = 0.f;
      }
      return;
    }
  }

  const int* bt = PAGED ? a.block_tables + static_cast<long>(s) * a.bt_stride : nullptr;
  const int lastpage = PAGED ? min(glast >> 4, a.bt_stride - 1) : 0;
  const int dense0 = PAGED ? 0 : a.base[s], low0 = PAGED ? 0 : first_gathered(past, a.window);
  const int kmax = PAGED ? glast : min(glast, a.nrows - 1 - dense0);  // the last key that may be read
  int page = 0;  // of the tile to be fetched next
  auto fetch_page = [&](int k0) {
    if constexpr (PAGED) page = bt[min((k0 >> 4) + wpage, lastpage)];
  };
  uint4 kst[NK], vst[NV];
  auto fetch_tile = [&](int k0) {
    const int key0 = k0 + 16 * wpage;
    const bf16_t *kb, *vb, *rb = nullptr;
    if constexpr (PAGED) {
      const bf16_t* blk = a.cache + static_cast<long>(page) * a.block_stride;
      kb = blk + a.koff + g * 16 * dk;
      vb = blk + a.voff + g * 16 * dv;
    } else {
      const long r = dense0 + key0;
      kb = a.kx + r * a.x_stride + g * a.dn;
      vb = a.vx + r * a.x_stride + g * dv;
      rb = a.kr + r * a.r_stride;
    }
    // keys past the last one anybody here sees may hold anything, and there are no rows before the first gathered one: zeros
    const int left = PAGED ? kmax - key0 : gathered_left(key0, low0, kmax);
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      kst[i] = make_uint4(0, 0, 0, 0);
      if (krow[i] >= 0 && krow[i] <= left) {
        const bf16_t* from = kb;
        if constexpr (!PAGED) from = kown[i] ? kb : rb;
        kst[i] = *reinterpret_cast<const uint4*>(from + kfrom[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      vst[i] = make_uint4(0, 0, 0, 0);
      if (vrow[i] >= 0 && vrow[i] <= left) vst[i] = *reinterpret_cast<const uint4*>(vb + vfrom[i]);
    }
  };
  auto put_tile = [&](bf16_t* buf) {
#pragma unroll
    for (int i = 0; i < NK; ++i)
      if (krow[i] >= 0) *reinterpret_cast<uint4*>(buf + kat[i]) = kst[i];
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (vrow[i] >= 0) *reinterpret_cast<uint4*>(buf + vat[i]) = vst[i];
  };
  fetch_page(start_of(it0));
  fetch_tile(start_of(it0));
  if (it0 + 1 < itn) fetch_page(start_of(it0 + 1));

  // Q^T: 8 entries of the lane's query per step of 16; a negative scale turns the query's sign
  const uint32_t flip = a.scale < 0.f ? 0x80008000u : 0u;
  const float sl2 = fmaxf(fabsf(a.scale) * 1.4426950408889634f, 1e-30f);
  b8_t qf[KS];
  {
    const bf16_t* qp = a.q + static_cast<long>(row0 + qi) * a.q_stride + head * dk + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint2 x = make_uint2(0, 0), y = x;
      if (qok && 16 * ks < dk) {
        x = *reinterpret_cast<const uint2*>(qp + 16 * ks);
        y = *reinterpret_cast<const uint2*>(qp + 16 * ks + 4);
      }
      qf[ks] = __builtin_bit_cast(b8_t, make_uint4(x.x ^ flip, x.y ^ flip, y.x ^ flip, y.y ^ flip));
    }
  }
  // m in log2 units; l is the lane's share of the sum: the sink's 1 goes to the lower half
  const bool sunk = a.sink && stretch == 0;
  float m = sunk ? a.sink[head] * 1.4426950408889634f : -INFINITY, l = (sunk && hi == 0) ? 1.f : 0.f;
  f16_t o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f16_t{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const int low = a.window > 0 ? pos - a.window : -1;  // the window's keys lie above it
  // the lane's corner of a transposing read: its 16-lane group turns 4 keys x 16 values
  const int trow = 4 * hi + ((lane & 15) >> 2), tcol = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

  put_tile(lds[it0 & 1]);
  for (int it = it0; it < itn; ++it) {
    __syncthreads();  // this tile is whole, and nobody reads the other buffer any more
    if (it + 1 < itn) {
      fetch_tile(start_of(it + 1));
      if (it + 2 < itn) fetch_page(start_of(it + 2));
    }
    const int k0 = start_of(it);
    const bf16_t* kl = lds[it & 1];
    const bf16_t* vl = kl + KT * KROW;
    if (live && k0 <= whi && (a.window <= 0 || k0 + KT > wlo - a.window + 1 || k0 < a.keep)) {
      f16_t acc[KU];
#pragma unroll
      for (int u = 0; u < KU; ++u) {
        acc[u] = f16_t{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const b8_t kf = __builtin_bit_cast(b8_t, *reinterpret_cast<const uint4*>(kl + (u * 32 + c) * KROW + 16 * ks + 8 * hi));
          acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], acc[u], 0, 0, 0);
        }
      }
      // a tile that every query of the wave sees whole (the usual case) needs no mask
      if (!(k0 + KT - 1 <= wlo && (a.window <= 0 || k0 > whi - a.window || k0 + KT - 1 < a.keep))) {
#pragma unroll
        for (int u = 0; u < KU; ++u)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int j = k0 + u * 32 + (i & 3) + 8 * (i >> 2) + 4 * hi;
            const bool seen = (j <= pos) & ((j > low) | (j < a.keep));
            acc[u][i] = seen ? acc[u][i] : -INFINITY;
          }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int u = 0; u < KU; ++u) {
        const f16_t& x = acc[u];
        const float p = vmax3(vmax3(x[0], x[1], x[2]), vmax3(x[3], x[4], x[5]), vmax3(x[6], x[7], x[8]));
        mx = vmax3(mx, vmax3(p, vmax3(x[9], x[10], x[11]), x[12]), vmax3(x[13], x[14], x[15]));
      }
      // m is a reference, not the maximum: weights may reach 2^6 before everything is rescaled to a new one, which
      // after the first tiles of a walk is seldom (a true maximum moves for some query of 32 in most tiles)
      const float m_new = across(mx, false) * sl2;
      if (__builtin_amdgcn_ballot_w64(m_new > m + 6.f) != 0) {
        const float to = vmax(m, m_new), corr = to == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - to);
        l *= corr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[dt][i] *= corr;
        m = to;
      }
      const float mneg = m == -INFINITY ? 0.f : -m;  // nothing seen yet: exp2(-inf) stays 0
#pragma unroll
      for (int n = 0; n < 2 * KU; ++n) {  // 16 keys
        uint32_t ph[4], pl[4], pr[4];
        float ls = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float p0 = __builtin_amdgcn_exp2f(fmaf(acc[n >> 1][8 * (n & 1) + 2 * j], sl2, mneg));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(acc[n >> 1][8 * (n & 1) + 2 * j + 1], sl2, mneg));
          ls += p0 + p1;
          // p = hi + lo: hi the upper 16 bits (exact), lo = p - hi rounded to bf16
          const uint32_t u0 = __float_as_uint(p0), u1 = __float_as_uint(p1);
          ph[j] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
          const f2_t lo = {p0 - __uint_as_float(u0 & 0xFFFF0000u), p1 - __uint_as_float(u1 & 0xFFFF0000u)};
          pl[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(lo, b2_t));
          if constexpr (WHOLE) {
            const f2_t rest = {lo[0] - bf2f_lo(pl[j]), lo[1] - bf2f_hi(pl[j])};
            pr[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, b2_t));
          }
        }
        l += ls;
        const b8_t bh = __builtin_bit_cast(b8_t, make_uint4(ph[0], ph[1], ph[2], ph[3]));
        const b8_t bl = __builtin_bit_cast(b8_t, make_uint4(pl[0], pl[1], pl[2], pl[3]));
        const bf16_t* vp = vl + (16 * n + trow) * VROW + tcol;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          typedef __attribute__((address_space(3))) s4_t* lds_s4;
          const s4_t x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(vp + 32 * dt));
          const s4_t y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(vp + 8 * VROW + 32 * dt));
          const short8 xy = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
          const b8_t vf = __builtin_bit_cast(b8_t, xy);
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, bh, o[dt], 0, 0, 0);
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, bl, o[dt], 0, 0, 0);
          if constexpr (WHOLE) {
            const b8_t br = __builtin_bit_cast(b8_t, make_uint4(pr[0], pr[1], pr[2], pr[3]));
            o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, br, o[dt], 0, 0, 0);
          }
        }
      }
    }
    if (it + 1 < itn) put_tile(lds[(it + 1) & 1]);
  }
  // A weight of zero makes NaN of a value that is no number, in queries that do not see its key: entries that came out as no
  // numbers are summed again key by key over the keys that their query does see, until no number can come of them any more.
  float odd = 0.f;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) odd = fmaf(o[dt][i], 0.f, odd);
  if (__builtin_amdgcn_ballot_w64(odd != 0.f) != 0) {
    f16_t r[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) r[dt][i] = 0.f;
    bool open = true;
#pragma unroll 1
    for (int n = it0 * KT; n < itn * KT && open; ++n) {
      const int j = start_of(n / KT) + n % KT;
      if (j < low0 || j > min(kmax, whi)) continue;
      const bf16_t *kj, *vj, *rj = nullptr;
      if constexpr (PAGED) {
        const bf16_t* blk = a.cache + static_cast<long>(bt[min(j >> 4, lastpage)]) * a.block_stride;
        kj = blk + a.koff + (g * 16 + (j & 15)) * dk;
        vj = blk + a.voff + (g * 16 + (j & 15)) * dv;
      } else {
        const long row = dense0 + j;
        kj = a.kx + row * a.x_stride + g * a.dn;
        vj = a.vx + row * a.x_stride + g * dv;
        rj = a.kr + row * a.r_stride - a.dn;
      }
      float sc = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int d = 16 * ks + 8 * hi;
        if (d >= dk) continue;
        float x[8];
        load16((PAGED || d < a.dn ? kj : rj) + d, x);
#pragma unroll
        for (int e = 0; e < 8; ++e) sc = fmaf(static_cast<float>(qf[ks][e]), x[e], sc);
      }
      sc = across(sc, true);
      const bool seen = (j <= pos) & ((j > low) | (j < a.keep));
      const float w = __builtin_amdgcn_exp2f(fmaf(sc, sl2, m == -INFINITY ? 0.f : -m));
      open = false;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int d = 32 * dt + 8 * b + 4 * hi;
          if (d >= dv) continue;
          const uint2 v = *reinterpret_cast<const uint2*>(vj + d);
          const float x[4] = {bf2f_lo(v.x), bf2f_hi(v.x), bf2f_lo(v.y), bf2f_hi(v.y)};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = 4 * b + e;
            if (seen) r[dt][i] = fmaf(w, x[e], r[dt][i]);
            open |= !(fabsf(o[dt][i]) < INFINITY) && fabsf(r[dt][i]) < INFINITY;
          }
        }
      open = __builtin_amdgcn_ballot_w64(open) != 0;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (!(fabsf(o[dt][i]) < INFINITY)) o[dt][i] = r[dt][i];
  }
  l = across(l, true);
  if (!qok) return;
  if constexpr (SPLIT) {
    if (hi == 0) {
      pp[0] = m;
      pp[1] = l;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        if (32 * dt + 8 * b < dv)
          *reinterpret_cast<float4*>(pp + 4 + 32 * dt + 8 * b + 4 * hi) =
              make_float4(o[dt][4 * b], o[dt][4 * b + 1], o[dt][4 * b + 2], o[dt][4 * b + 3]);
    return;
  }
  const float inv = 1.f / l;
  bf16_t* op = a.out + static_cast<long>(row0 + qi) * (a.H * dv) + head * dv + 4 * hi;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int d = 32 * dt + 8 * b;  // dims d + 4 hi .. + 3; dv is a multiple of 16
      if (d < dv) {
        uint2 w;
        w.x = pack2(o[dt][4 * b] * inv, o[dt][4 * b + 1] * inv);
        w.y = pack2(o[dt][4 * b + 2] * inv, o[dt][4 * b + 3] * inv);
        *reinterpret_cast<uint2*>(op + d) = w;
      }
    }
  }
}

bool launch_chunk_attention(const ChunkArgs& a, int max_q, hipStream_t st) {
  const bool paged = a.kx == nullptr;
  if (a.dk % 16 || a.dv % 16 || a.dv > 128 || a.dk > (paged ? 128 : 192) || (!paged && (a.dn % 8 || a.dn > a.dk || a.G != a.H)))
    return false;
  const int n = a.nsplit > 1 ? a.nsplit : 1;
  const dim3 grid(a.G, (static_cast<long>(max_q) * (a.H / a.G) + 127) / 128, a.S * n), block(256);
  if (grid.z > 65535u) return false;
#define MIX_CHUNK(WHOLE, ...)                                                                                                \
  do {                                                                                                                       \
    if (n > 1) hipLaunchKernelGGL((chunk_attention_kernel<__VA_ARGS__, true, WHOLE>), grid, block, 0, st, a);                \
    else hipLaunchKernelGGL((chunk_attention_kernel<__VA_ARGS__, false, WHOLE>), grid, block, 0, st, a);                     \
  } while (0)
  // chunks of fewer than 16 rows keep all bits of a weight, as the forms for rows do
  const bool whole = paged && max_q < 16, small = a.dk <= 64 && a.dv <= 64;
  if (!paged) MIX_CHUNK(false, 192, 128, 32, false);
  else if (small && whole) MIX_CHUNK(true, 64, 64, 64, true);
  else if (small) MIX_CHUNK(false, 64, 64, 64, true);
  else if (whole) MIX_CHUNK(true, 128, 128, 32, true);
  else MIX_CHUNK(false, 128, 128, 32, true);
#undef MIX_CHUNK
  MXS_CHECK_LAUNCH();
  return n == 1 || launch_attention_combine(a.out, a.part, static_cast<long>(a.rows) * a.H, n, a.dv, st);
}

// Stretches pay where the longest walk counts and not the chip: a key costs a walk some 0.022 us (heads of 64; 0.04 with 128
// entries), a stretch's records their bytes twice at 2 TB/s, the merge 6 us.  Whole against split, 32 heads of 64 over 8:
// 64 rows behind 2,000 keys 49.7 / 21.6 us, 512 rows behind 2,000 62.3 / 44.7, behind 1,000 39.6 / 37.6; 1,024 rows with
// nothing behind them 29.1 / 47.2 (two stretches, not chosen); 16 heads of 128 over 4:
// 512 rows behind 2,000 105 / 49.  Up to about
// two workgroups a unit, stretches of 512 keys or more.
int chunk_attention_splits(long rows, int S, int H, int G, int dk, int dv, long span) {
  const long tiles = G * (rows * (H / G) / 128 + S);
  if (tiles == 0 || span < 1024) return 1;
  int best = 1;
  double gain = 0.;
  for (int n = 2; n <= 4 && n * tiles <= 1024 && 512L * n <= span && S * n <= 65535; ++n) {
    const double walk = static_cast<double>(span) * (dk + dv <= 128 ? 0.022 : 0.04);
    const double g = walk * (1. - 1. / n) - 2. * 4. * (dv + 4) * rows * H * n / 2e6 - 6.;
    if (g > gain) {
      gain = g;
      best = n;
    }
  }
  return best;
}

// One workgroup: the sequences' row counts summed 256 at a time.
__global__ void __launch_bounds__(256) latent_plan_kernel(int* __restrict__ base, int* __restrict__ offs,
                                                          const int* __restrict__ qsl, const int* __restrict__ seq_lens,
                                                          int S, int window) {
  __shared__ int sum[256];
  int before = 0;
  for (int s0 = 0; s0 < S; s0 += 256) {
    const int s = s0 + threadIdx.x;
    int n = 0, firstkey = 0;
    if (s < S) {
      const int qlen = qsl[s + 1] - qsl[s], past = max(seq_lens[s] - qlen, 0);
      firstkey = first_gathered(past, window);
      n = qlen > 0 ? past + qlen - firstkey : 0;
    }
    sum[threadIdx.x] = n;
    __syncthreads();
    for (int o = 1; o < 256; o <<= 1) {
      const int t = threadIdx.x >= o ? sum[threadIdx.x - o] : 0;
      __syncthreads();
      sum[threadIdx.x] += t;
      __syncthreads();
    }
    if (s < S) {
      offs[s] = before + sum[threadIdx.x] - n;
      base[s] = offs[s] - firstkey;
    }
    before += sum[255];
    __syncthreads();
  }
  if (threadIdx.x == 0) offs[S] = before;
}

void launch_latent_plan(int* base, int* offs, const int* qsl, const int* seq_lens, int S, int window, hipStream_t st) {
  hipLaunchKernelGGL(latent_plan_kernel, dim3(1), dim3(256), 0, st, base, offs, qsl, seq_lens, S, window);
  MXS_CHECK_LAUNCH();
}

__global__ void __launch_bounds__(256) latent_rows_kernel(uint4* __restrict__ out, const bf16_t* __restrict__ cache, long block_stride,
                                                          const int* __restrict__ block_tables, int bt_stride,
                                                          const int* __restrict__ base, const int* __restrict__ offs, int S,
                                                          int n, int koff, int pieces) {
  const long i = blockIdx.x * 256l + threadIdx.x;
  const int row = static_cast<int>(i / pieces), piece = static_cast<int>(i - static_cast<long>(row) * pieces);
  if (row >= min(n, offs[S])) return;
  const int s = seq_of_row(offs, S, row), key = row - base[s];
  const int page = block_tables[static_cast<long>(s) * bt_stride + min(key >> 4, bt_stride - 1)];
  out[i] = *reinterpret_cast<const uint4*>(cache + page * block_stride + koff + ((key & 15) * pieces + piece) * 8);
}

void launch_latent_rows(bf16_t* out, const bf16_t* cache, long block_stride, const int* block_tables, int bt_stride,
                        const int* base, const int* offs, int S, int n, int koff, int dk, hipStream_t st) {
  if (n == 0) return;
  const int pieces = dk / 8;
  hipLaunchKernelGGL(latent_rows_kernel, dim3((static_cast<long>(n) * pieces + 255) / 256), dim3(256), 0, st,
                     reinterpret_cast<uint4*>(out), cache, block_stride, block_tables, bt_stride, base, offs, S, n, koff, pieces);
  MXS_CHECK_LAUNCH();
}

}  // namespace mxs
