// torch bindings of the mixer kernels (mxserve/_M): shape and dtype checks on the host, so that a
// launch never reads or writes outside what the kernels and their grids assume.
#include <limits>

#include "chunk_attention.h"
#include "bind_util.h"
#include "column_scan.h"
#include "differential_attention.h"

namespace mxs {
void launch_resid_update(float*, const void*, long, const void*, const void*, long, const void*, const void*, int,
                         const void*, void*, int, int, float, float, float, float, bool, hipStream_t);
void launch_embed_normed(float*, float*, void*, const int64_t*, const void*, const void*, int, int, long, float, float, bool,
                         hipStream_t);
bool launch_depth_mix(float*, long, int, const float*, void*, int, int, bool, hipStream_t);
void launch_xielu(void*, const void*, long, const float*, bool, hipStream_t);
void launch_qkv_prep_cache(void*, long, const void*, long, const void*, long, const int64_t*, const int64_t*, void*, long,
                           int, int, int, int, int, int, int, int, const float*, int, float, bool, const void*, const void*,
                           const void*, const void*, const void*, float, int, bool, hipStream_t);
bool launch_talking_attention(void*, const void*, long, const void*, long, const int*, int, const int*, const int*, int,
                              int, int, int, int, int, int, int, int, float, int, int, int, const float*, const float*, float*,
                              int, bool, hipStream_t);
void launch_cast_into(void*, long, const float*, int, int, bool, hipStream_t);
void launch_relu_sq(void*, const void*, long, bool, hipStream_t);
void launch_softcap(float*, const void*, long, int, int, float, bool, hipStream_t);
void launch_gated_rms_norm(void*, const float*, const void*, long, const void*, int, int, int, float, bool, hipStream_t);
void launch_gate_linear(float*, const void*, long, const void*, const void*, int, int, int, bool, hipStream_t);
void launch_kv_write(void*, long, const void*, long, const void*, long, const int64_t*, int, int, int, int, int, int,
                     int, bool, hipStream_t);
bool launch_window_attention(void*, const void*, long, const void*, long, const int*, int, const int*, const int*, int,
                             int, int, int, int, int, int, int, int, float, int, int, int, bool, const float*, int, int,
                             float*, bool, hipStream_t);
bool launch_matrix_scan(float*, const void*, long, const void*, long, const void*, long, const float*, const float*,
                        float*, long, const int*, long, const int*, const int*, int, int, int, int, int, int, float,
                        float, bool, bool, int, int, float*, float*, long, hipStream_t);
void launch_embed_scaled(float*, const int64_t*, const void*, int, int, long, float, bool, hipStream_t);
void launch_rope_qkv_cache(void*, long, const void*, long, const void*, long, const int64_t*, const int64_t*, void*, long,
                           int, int, int, int, int, int, int, int, const float*, int, const void*, const void*, float,
                           const float*, int, bool, hipStream_t);
void launch_rope_rows(void*, long, const void*, long, const int64_t*, int, int, int, const float*, int, float, float, bool,
                      hipStream_t);
void launch_causal_conv(void*, const void*, long, const void*, const void*, float*, long, const int*, long, const int*,
                        const int*, int, int, int, int, int, bool, bool, hipStream_t);
void launch_gated_norm(void*, long, const float*, const void*, long, const void*, int, int, int, int, float, int, int,
                       float, bool, hipStream_t);
bool launch_column_scan(const ScanArgs&, int, int, bool, hipStream_t);
bool launch_decay_lowrank(float*, const void*, long, const void*, const void*, int, int, int, float, bool, hipStream_t);
bool launch_streams(float*, int, const void*, long, const int64_t*, long, const void*, const void*, const float*, const void*,
                    void*, int, int, float, float, bool, hipStream_t);
void launch_act(void*, const void*, long, int, int, int, bool, bool, hipStream_t);
void launch_conv_qkv_cache(void*, const void*, long, const void*, const void*, float*, long, const int*, long, const int*,
                           const int*, int, int, const int64_t*, const int64_t*, void*, long, int, int, int, int, int, int,
                           int, int, float, float, bool, bool, hipStream_t);
int differential_tiles(int, int);
bool launch_differential_attention(const DiffArgs&, int, int, bool, hipStream_t);
bool launch_route_grouped(float*, int*, const float*, const float*, int, int, int, int, int, float, bool, bool, hipStream_t);
bool launch_latent_attention(void*, float*, const void*, long, const void*, long, const int*, int, const int*, const int*,
                             int, int, int, int, int, int, int, float, int, const float*, int, bool, int, hipStream_t);
void launch_latent_prep(void*, const void*, long, const void*, long, const int64_t*, const int64_t*, void*, long, int, int,
                        int, int, int, int, const float*, const void*, const void*, float, bool, float, bool, hipStream_t);
void launch_rope_half_into(void*, long, const void*, long, const int64_t*, int, int, int, int, int, int, const float*, int,
                           bool, float, bool, hipStream_t);
void launch_route_topk(float*, int*, const float*, int, int, int, bool, bool, hipStream_t);
void launch_capped_glu(void*, const void*, long, int, int, float, float, bool, hipStream_t);
bool launch_expert_align(int*, int*, const int*, int, int, hipStream_t);
void launch_gather_scaled(void*, const void*, long, const float*, const int*, int, int, int, const int*, const int*, int, int,
                          int*, bool, hipStream_t);
void launch_spread_scaled(void*, const void*, long, const float*, const int*, int, int, int, int, bool, hipStream_t);
void launch_expert_combine(void*, const void*, const int*, int, int, long, const void*, long, int, const float*, bool, bool,
                           hipStream_t);
}  // namespace mxs

using namespace mxs_bind;

namespace {

void resid_update(at::Tensor x, OptT a, OptT wa, OptT b, OptT wb, OptT bias, bool assign, OptT norm_w, OptT h,
                  double eps, double a_scale, double w_offset, double wa_offset) {
  float* xp = f32(x, "x");
  TORCH_CHECK(x.dim() == 2, "x: [T, W]");
  const int64_t T = x.size(0), W = x.size(1);
  const at::Tensor* any = a.has_value() ? &*a : (norm_w.has_value() ? &*norm_w : (h.has_value() ? &*h : nullptr));
  if (any == nullptr || T == 0) return;
  const bool bf = is_bf(*any);
  const void* ap = a.has_value() ? mat(*a, bf, T, W, "a") : nullptr;
  const void* bp = b.has_value() ? mat(*b, bf, T, W, "b") : nullptr;
  TORCH_CHECK(!b.has_value() || (a.has_value() && wa.has_value() && wb.has_value()), "two branches need both weights");
  TORCH_CHECK(!assign || a.has_value(), "assign needs a");
  TORCH_CHECK(!norm_w.has_value() || h.has_value(), "norm_w needs h (h alone: the updated x, cast)");
  void* hp = nullptr;
  if (h.has_value()) {
    TORCH_CHECK(h->is_cuda() && h->is_contiguous() && h->dim() == 2 && h->size(0) == T && h->size(1) == W &&
                is_bf(*h) == bf, "h: contiguous [T, W] of the operands' dtype");
    hp = h->data_ptr();
  }
  mxs::launch_resid_update(xp, ap, a.has_value() ? a->stride(0) : 0, vec(wa, bf, W, "wa"), bp,
                           b.has_value() ? b->stride(0) : 0, vec(wb, bf, W, "wb"), vec(bias, bf, W, "bias"), assign,
                           vec(norm_w, bf, W, "norm_w"), hp, static_cast<int>(T), static_cast<int>(W),
                           static_cast<float>(eps), static_cast<float>(a_scale), static_cast<float>(w_offset),
                           static_cast<float>(wa_offset), bf, stream());
}

void cast_into(at::Tensor dst, at::Tensor x) {
  const float* xp = f32(x, "x");
  TORCH_CHECK(x.dim() == 2 && dst.is_cuda() && dst.dim() == 2 && dst.size(0) == x.size(0) && dst.size(1) >= x.size(1) &&
              dst.stride(1) == 1, "dst: [T, >= W] with contiguous rows");
  mxs::launch_cast_into(dst.data_ptr(), dst.stride(0), xp, static_cast<int>(x.size(0)), static_cast<int>(x.size(1)),
                        is_bf(dst), stream());
}

void relu_sq(at::Tensor out, at::Tensor x) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && out.is_contiguous() && out.numel() == x.numel() &&
              out.scalar_type() == x.scalar_type(), "relu_sq: contiguous tensors of one dtype");
  mxs::launch_relu_sq(out.data_ptr(), x.data_ptr(), x.numel(), is_bf(x), stream());
}

void softcap(at::Tensor out, at::Tensor x, double cap) {
  float* op = f32(out, "out");
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1 && out.dim() == 2 && out.size(0) == x.size(0) &&
              out.size(1) == x.size(1), "softcap: [n, V]");
  mxs::launch_softcap(op, x.data_ptr(), x.stride(0), static_cast<int>(x.size(0)), static_cast<int>(x.size(1)),
                      static_cast<float>(cap), is_bf(x), stream());
}

void gated_rms_norm(at::Tensor out, at::Tensor o, at::Tensor gate, at::Tensor w, double eps, int64_t groups) {
  const float* opn = f32(o, "o");
  TORCH_CHECK(o.dim() == 2, "o: [T, N]");
  const int64_t T = o.size(0), N = o.size(1);
  const bool bf = is_bf(out);
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && out.dim() == 2 && out.size(0) == T && out.size(1) == N, "out: [T, N]");
  TORCH_CHECK(groups >= 1 && N % groups == 0, "groups must divide N");
  mxs::launch_gated_rms_norm(out.data_ptr(), opn, mat(gate, bf, T, N, "gate"), gate.stride(0), vec(OptT(w), bf, N, "w"),
                             static_cast<int>(T), static_cast<int>(N), static_cast<int>(groups), static_cast<float>(eps),
                             bf, stream());
}

void gate_linear(at::Tensor out, at::Tensor h, at::Tensor w, OptT bias) {
  float* op = f32(out, "out");
  TORCH_CHECK(h.is_cuda() && h.dim() == 2 && h.stride(1) == 1 && w.is_cuda() && w.dim() == 2 && w.is_contiguous() &&
              w.size(1) == h.size(1) && out.dim() == 2 && out.size(0) == h.size(0) && out.size(1) == w.size(0),
              "gate_linear: h [T, W], w [N, W], out [T, N]");
  const bool bf = is_bf(h);
  TORCH_CHECK(is_bf(w) == bf, "w: dtype differs from h");
  mxs::launch_gate_linear(op, h.data_ptr(), h.stride(0), w.data_ptr(), vec(bias, bf, w.size(0), "bias"),
                          static_cast<int>(h.size(0)), static_cast<int>(w.size(0)), static_cast<int>(w.size(1)), bf,
                          stream());
}

void kv_write(at::Tensor cache, at::Tensor k, at::Tensor v, at::Tensor slots, int64_t koff, int64_t voff, int64_t G,
              int64_t dk, int64_t dv, int64_t bs) {
  const bool bf = is_bf(k);
  const int64_t T = k.size(0);
  check_cache(cache, bf, koff, voff, G, dk, dv, bs);
  TORCH_CHECK(slots.is_cuda() && slots.scalar_type() == at::kLong && slots.is_contiguous() && slots.numel() == T,
              "slot_mapping: int64 [T]");
  mxs::launch_kv_write(cache.data_ptr(), cache.stride(0), mat(k, bf, T, G * dk, "k"), k.stride(0),
                       mat(v, bf, T, G * dv, "v"), v.stride(0), slots.data_ptr<int64_t>(), static_cast<int>(T),
                       static_cast<int>(koff), static_cast<int>(voff), static_cast<int>(G), static_cast<int>(dk),
                       static_cast<int>(dv), static_cast<int>(bs), bf, stream());
}

void window_attention(at::Tensor out, at::Tensor q, at::Tensor cache, at::Tensor block_tables, at::Tensor qsl,
                      at::Tensor seq_lens, int64_t koff, int64_t voff, int64_t H, int64_t G, int64_t dk, int64_t dv,
                      int64_t bs, double scale, int64_t window, int64_t keep, int64_t max_query_len, OptT sink,
                      int64_t v_stride, int64_t max_seq_len) {
  const bool bf = is_bf(q);
  const float* sinkp = nullptr;
  if (sink.has_value()) {
    sinkp = f32(*sink, "sink");
    TORCH_CHECK(sink->numel() == H, "sink: fp32 [H]");
  }
  const int64_t T = q.size(0), S = seq_lens.numel();
  if (v_stride > 0 && v_stride != dv) {  // values are a slice of a wider cached row of the one kv head
    TORCH_CHECK(G == 1 && v_stride >= dv, "strided value rows: one kv head, stride >= dv");
    check_cache(cache, bf, koff, voff, G, dk, 0, bs);
    TORCH_CHECK(voff >= 0 && voff + (bs - 1) * v_stride + dv <= cache.size(1), "value rows reach past the cache block");
  } else {
    check_cache(cache, bf, koff, voff, G, dk, dv, bs);
  }
  TORCH_CHECK(G >= 1 && H % G == 0, "query heads must divide over kv heads");
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && out.dim() == 2 && out.size(0) == T && out.size(1) == H * dv &&
              is_bf(out) == bf, "out: [T, H*dv]");
  TORCH_CHECK(block_tables.is_cuda() && block_tables.scalar_type() == at::kInt && block_tables.dim() == 2 &&
              block_tables.size(0) >= S && block_tables.stride(1) == 1, "block_tables: int32 [S, max_blocks]");
  // a step of few rows, and the long walks of few chunks, split their keys over workgroups
  const int64_t table = block_tables.stride(0) * bs, seen = window > 0 ? window + std::max<int64_t>(keep, 0) : table;
  const int h = static_cast<int>(H), g = static_cast<int>(G);
  const int64_t span = std::min(max_seq_len > 0 ? std::min(max_seq_len, table) : table, seen);
  const int max_q = static_cast<int>(std::min<int64_t>(max_query_len, T));
  const bool by_rows = mxs::row_attention_serves(T, max_q, h, g, span);
  const int nsplit = !bf || dk > 128 || dv > 128 ? 1 :
      by_rows ? mxs::row_attention_splits(T, h, g, std::min(table, seen)) :
      mxs::chunk_attention_splits(T, static_cast<int>(S), h, g, static_cast<int>(dk), static_cast<int>(dv), std::min(max_seq_len, seen));
  at::Tensor part;
  if (nsplit > 1) part = at::empty({T * H * nsplit * (dv + 4)}, out.options().dtype(at::kFloat));
  const bool ok = mxs::launch_window_attention(
      out.data_ptr(), mat(q, bf, T, H * dk, "q"), q.stride(0), cache.data_ptr(), cache.stride(0),
      block_tables.data_ptr<int>(), static_cast<int>(block_tables.stride(0)), i32(qsl, S + 1, "qsl"),
      i32(seq_lens, S, "seq_lens"), static_cast<int>(S), static_cast<int>(T), static_cast<int>(koff),
      static_cast<int>(voff), static_cast<int>(H), static_cast<int>(G), static_cast<int>(dk), static_cast<int>(dv),
      static_cast<int>(bs), static_cast<float>(scale), static_cast<int>(window), static_cast<int>(keep),
      max_q, by_rows, sinkp, static_cast<int>(v_stride), nsplit,
      nsplit > 1 ? part.data_ptr<float>() : nullptr, bf, stream());
  TORCH_CHECK(ok, "window_attention: head sizes beyond what the kernel holds (dv <= 512)");
}

void scan(bool mlstm, at::Tensor out, at::Tensor q, at::Tensor k, at::Tensor v, const float* decay, const float* gates,
          at::Tensor state, at::Tensor state_rows, int64_t off, at::Tensor qsl, at::Tensor seq_lens, int64_t H,
          int64_t dk, int64_t dv, bool silu, double cap, double q_scale, int64_t piece, int64_t npieces, OptT sc_local,
          OptT sc_start) {
  const bool bf = is_bf(q);
  const int64_t T = q.size(0), S = seq_lens.numel();
  float* op = f32(out, "out");
  TORCH_CHECK(out.dim() == 2 && out.size(0) == T && out.size(1) == H * dv, "out: fp32 [T, H*dv]");
  float* sp = f32(state, "state");
  const int64_t need = mlstm ? H * (dk * dv + dk + 1) : H * dk * dv;
  TORCH_CHECK(state.dim() == 2 && off >= 0 && off + need <= state.size(1), "state slot too small for this layer");
  // time-split launches: two scratch pools of [S, npieces, sc_floats] (a piece's end state; mLSTM: plus [H] sums)
  const int64_t sc_floats = need + (mlstm ? H : 0);
  float *scl = nullptr, *scs = nullptr;
  if (npieces > 1) {
    TORCH_CHECK(piece >= 16 && sc_local.has_value() && sc_start.has_value(), "a split scan needs its scratch pools");
    scl = f32(*sc_local, "sc_local");
    scs = f32(*sc_start, "sc_start");
    TORCH_CHECK(sc_local->numel() >= S * npieces * sc_floats && sc_start->numel() >= S * npieces * sc_floats,
                "scratch pools smaller than [S, npieces, state]");
  } else {
    piece = 1;
    npieces = 1;
  }
  const bool ok = mxs::launch_matrix_scan(
      op, mat(q, bf, T, H * dk, "q"), q.stride(0), mat(k, bf, T, H * dk, "k"), k.stride(0), mat(v, bf, T, H * dv, "v"),
      v.stride(0), decay, gates, sp, state.stride(0), i32(state_rows, S, "state_rows"), off, i32(qsl, S + 1, "qsl"),
      i32(seq_lens, S, "seq_lens"), static_cast<int>(S), static_cast<int>(T), static_cast<int>(H), static_cast<int>(dk),
      static_cast<int>(dv), silu ? 1 : 0, static_cast<float>(cap), static_cast<float>(q_scale), mlstm, bf,
      static_cast<int>(piece), static_cast<int>(npieces), scl, scs, sc_floats, stream());
  TORCH_CHECK(ok, "matrix scan: key size beyond 256");
}

void decay_scan(at::Tensor out, at::Tensor q, at::Tensor k, at::Tensor v, at::Tensor decay, at::Tensor state,
                at::Tensor state_rows, int64_t off, at::Tensor qsl, at::Tensor seq_lens, int64_t H, int64_t dk,
                int64_t dv, bool silu, int64_t piece, int64_t npieces, OptT sc_local, OptT sc_start) {
  TORCH_CHECK(decay.numel() == H, "decay: fp32 [H]");
  scan(false, out, q, k, v, f32(decay, "decay"), nullptr, state, state_rows, off, qsl, seq_lens, H, dk, dv, silu, 0.0, 1.0,
       piece, npieces, sc_local, sc_start);
}

void mlstm_scan(at::Tensor out, at::Tensor q, at::Tensor k, at::Tensor v, at::Tensor gates, at::Tensor state,
                at::Tensor state_rows, int64_t off, at::Tensor qsl, at::Tensor seq_lens, int64_t H, int64_t dk,
                int64_t dv, double cap, double q_scale, int64_t piece, int64_t npieces, OptT sc_local, OptT sc_start) {
  TORCH_CHECK(gates.dim() == 2 && gates.size(0) == q.size(0) && gates.size(1) == 2 * H, "gates: fp32 [T, 2H]");
  scan(true, out, q, k, v, nullptr, f32(gates, "gates"), state, state_rows, off, qsl, seq_lens, H, dk, dv, false, cap,
       q_scale, piece, npieces, sc_local, sc_start);
}

// ---- rotary attention, convolutions, column scans
void embed_scaled(at::Tensor out, at::Tensor ids, at::Tensor table, double scale) {
  float* op = f32(out, "out");
  TORCH_CHECK(table.is_cuda() && table.dim() == 2 && table.is_contiguous(), "table: contiguous [vocab, W]");
  const int64_t T = ids.numel(), W = table.size(1);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == T && out.size(1) == W, "out: fp32 [T, W]");
  mxs::launch_embed_scaled(op, i64(ids, T, "ids"), table.data_ptr(), static_cast<int>(T), static_cast<int>(W),
                           table.size(0), static_cast<float>(scale), is_bf(table), stream());
}

void rope_qkv_cache(at::Tensor q, OptT k, OptT v, at::Tensor positions, at::Tensor slots, at::Tensor cache, int64_t koff,
                    int64_t voff, int64_t H, int64_t G, int64_t dk, int64_t dv, int64_t bs, at::Tensor freqs, OptT q_norm,
                    OptT k_norm, double eps, OptT v_freqs) {
  const bool bf = is_bf(q);
  const int64_t T = q.size(0);
  TORCH_CHECK(k.has_value() == v.has_value(), "k and v go together");
  const void *kp = nullptr, *vp = nullptr;
  if (k.has_value()) {
    check_cache(cache, bf, koff, voff, G, dk, dv, bs);
    kp = mat(*k, bf, T, G * dk, "k");
    vp = mat(*v, bf, T, G * dv, "v");
  }
  const int64_t nf = freqs.numel(), nvf = v_freqs.has_value() ? v_freqs->numel() : 0;
  TORCH_CHECK(2 * nf <= dk && 2 * nvf <= dv, "more rotary pairs than the head has dimensions");
  mxs::launch_rope_qkv_cache(const_cast<void*>(mat(q, bf, T, H * dk, "q")), q.stride(0), kp, k.has_value() ? k->stride(0) : 0,
                             vp, v.has_value() ? v->stride(0) : 0, i64(positions, T, "positions"),
                             i64(slots, T, "slot_mapping"), cache.data_ptr(), cache.stride(0), static_cast<int>(T),
                             static_cast<int>(koff), static_cast<int>(voff), static_cast<int>(H), static_cast<int>(G),
                             static_cast<int>(dk), static_cast<int>(dv), static_cast<int>(bs), f32(freqs, "freqs"),
                             static_cast<int>(nf), vec(q_norm, bf, dk, "q_norm"), vec(k_norm, bf, dk, "k_norm"),
                             static_cast<float>(eps), f32n(v_freqs, nvf, "v_freqs"), static_cast<int>(nvf), bf, stream());
}

void rope_rows(at::Tensor out, at::Tensor x, at::Tensor positions, int64_t heads, int64_t dim, at::Tensor freqs,
               double sign, double scale) {
  const bool bf = is_bf(x);
  const int64_t T = x.size(0);
  TORCH_CHECK(2 * freqs.numel() <= dim, "more rotary pairs than the head has dimensions");
  mxs::launch_rope_rows(const_cast<void*>(mat(out, bf, T, heads * dim, "out")), out.stride(0), mat(x, bf, T, heads * dim, "x"),
                        x.stride(0), i64(positions, T, "positions"), static_cast<int>(T), static_cast<int>(heads),
                        static_cast<int>(dim), f32(freqs, "freqs"), static_cast<int>(freqs.numel()),
                        static_cast<float>(sign), static_cast<float>(scale), bf, stream());
}

void causal_conv(at::Tensor out, at::Tensor x, at::Tensor w, OptT bias, at::Tensor state, at::Tensor state_rows,
                 int64_t off, at::Tensor qsl, at::Tensor seq_lens, bool silu, int64_t max_q) {
  const bool bf = is_bf(x);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && w.is_cuda() && w.is_contiguous() && is_bf(w) == bf && w.size(1) == x.size(1),
              "causal_conv: x [T, C], w [taps, C] of one dtype");
  const int64_t T = x.size(0), C = x.size(1), taps = w.size(0), S = seq_lens.numel();
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && out.dim() == 2 && out.size(0) == T && out.size(1) == C &&
              is_bf(out) == bf, "out: contiguous [T, C]");
  float* sp = f32(state, "state");
  TORCH_CHECK(state.dim() == 2 && off >= 0 && off + (taps - 1) * C <= state.size(1), "state slot too small for this filter");
  mxs::launch_causal_conv(out.data_ptr(), mat(x, bf, T, C, "x"), x.stride(0), w.data_ptr(), vec(bias, bf, C, "bias"), sp,
                          state.stride(0), i32(state_rows, S, "state_rows"), off, i32(qsl, S + 1, "qsl"),
                          i32(seq_lens, S, "seq_lens"), static_cast<int>(S), static_cast<int>(T), static_cast<int>(C),
                          static_cast<int>(taps), silu ? 1 : 0, max_q == 1 && T == S, bf, stream());
}

void gated_norm(at::Tensor out, at::Tensor o, at::Tensor gate, at::Tensor w, double eps, int64_t groups, bool silu,
                bool gate_first, double scale) {
  const float* opn = f32(o, "o");
  TORCH_CHECK(o.dim() == 2, "o: [T, N]");
  const int64_t T = o.size(0), N = o.size(1), wn = w.numel();
  const bool bf = is_bf(out);
  TORCH_CHECK(groups >= 1 && N % groups == 0 && wn >= 1 && N % wn == 0, "groups and the weight's length must divide N");
  mxs::launch_gated_norm(const_cast<void*>(mat(out, bf, T, N, "out")), out.stride(0), opn, mat(gate, bf, T, N, "gate"),
                         gate.stride(0), vec(OptT(w), bf, wn, "w"), static_cast<int>(wn), static_cast<int>(T),
                         static_cast<int>(N), static_cast<int>(groups), static_cast<float>(eps), silu ? 1 : 0,
                         gate_first ? 1 : 0, static_cast<float>(scale), bf, stream());
}

void column_scan(int kind, at::Tensor out, at::Tensor q, at::Tensor k, at::Tensor v, OptT beta, OptT a,
                 OptT dt_bias, OptT A_log, OptT D, at::Tensor state, at::Tensor state_rows, int64_t off,
                 at::Tensor qsl, at::Tensor seq_lens, int64_t H, int64_t G, int64_t dk, int64_t dv, double q_scale,
                 double unit_eps, int64_t piece = 1, int64_t npieces = 1, OptT sc_local = OptT(), OptT sc_start = OptT(),
                 OptT sc_decay = OptT(), int64_t mode = 0, int64_t max_q = 0, OptT work = OptT()) {
  const bool bf = is_bf(q), delta = kind == mxs::kDeltaRule, gla = kind == mxs::kGatedLinear;
  const int64_t T = q.size(0), S = seq_lens.numel();
  TORCH_CHECK(G >= 1 && H % G == 0, "heads must divide over the q/k heads (groups)");
  mxs::ScanArgs p{};
  p.out = f32(out, "out");
  TORCH_CHECK(out.dim() == 2 && out.size(0) == T && out.size(1) == H * dv, "out: fp32 [T, H*dv]");
  p.q = mat(q, bf, T, G * dk, "q");
  p.q_stride = q.stride(0);
  p.k = mat(k, bf, T, G * dk, "k");
  p.k_stride = k.stride(0);
  p.v = mat(v, bf, T, H * dv, "v");
  p.v_stride = v.stride(0);
  if (gla) {
    TORCH_CHECK(a.has_value() && G == H, "gated linear attention: log decays, one q/k head per head");
    p.a = mat(*a, false, T, H * dk, "log decays (fp32)");
    p.a_stride = a->stride(0);
  } else {
    TORCH_CHECK(beta.has_value() && dt_bias.has_value() && A_log.has_value(), "column scan: beta, dt_bias and A_log");
    p.beta = mat(*beta, bf, T, H, "beta");
    p.beta_stride = beta->stride(0);
    if (delta) {
      TORCH_CHECK(a.has_value(), "the delta rule needs its decay pre-activations");
      p.a = mat(*a, bf, T, H * dk, "a");
      p.a_stride = a->stride(0);
    } else {
      TORCH_CHECK(D.has_value(), "the state-space scan needs D");
    }
    p.dt_bias = f32n(dt_bias, delta ? H * dk : H, "dt_bias");
    p.A_log = f32n(A_log, H, "A_log");
    p.D = f32n(D, H, "D");
  }
  p.state = f32(state, "state");
  TORCH_CHECK(state.dim() == 2 && off >= 0 && off + H * dk * dv <= state.size(1), "state slot too small for this layer");
  p.state_stride = state.stride(0);
  p.state_rows = i32(state_rows, S, "state_rows");
  p.off = off;
  p.qsl = i32(qsl, S + 1, "qsl");
  p.seq_lens = i32(seq_lens, S, "seq_lens");
  p.n_rows = static_cast<int>(T);
  p.H = static_cast<int>(H);
  p.G = static_cast<int>(G);
  p.dk = static_cast<int>(dk);
  p.dv = static_cast<int>(dv);
  p.q_scale = static_cast<float>(q_scale);
  p.unit_eps = static_cast<float>(unit_eps);
  p.piece = 1;
  p.npieces = 1;
  p.max_q = max_q > 1 ? static_cast<int>(std::max<int64_t>(2, std::min(max_q, T))) : max_q == 1 && T == S ? 1 : 0;  // 1: every sequence brings one row
  if (npieces > 1) {  // pieces side by side: scratch [S, npieces, state] twice and the pieces' decays
    TORCH_CHECK(piece >= 16 && sc_local.has_value() && sc_start.has_value() && (delta || sc_decay.has_value()),
                "a split scan needs its scratch pools");
    TORCH_CHECK(sc_local->numel() >= S * npieces * H * dk * (delta ? dv + dk : dv) &&
                sc_start->numel() >= S * npieces * H * dk * dv &&
                (delta || sc_decay->numel() >= S * npieces * H * (gla ? dk : 1)),
                "scratch pools smaller than [S, npieces, state]");
    TORCH_CHECK(!delta || mode == 1 || mode == 2, "a split delta-rule scan is launched pass by pass");
    p.piece = static_cast<int>(piece);
    p.npieces = static_cast<int>(npieces);
    p.mode = static_cast<int>(mode);
    p.sc_local = f32(*sc_local, "sc_local");
    p.sc_start = f32(*sc_start, "sc_start");
    p.sc_decay = delta ? nullptr : f32(*sc_decay, "sc_decay");
  }
  if (work.has_value()) {
    const int64_t floats = mxs::delta_chunk_floats(p.dk, p.dv);
    TORCH_CHECK(delta && bf && floats > 0 && work->numel() >= (T / 32 + S) * H * floats, "delta rule in chunks: bf16, its sizes, its scratch");
    if (S == 0 || T == 0 || mxs::launch_delta_chunk(p, static_cast<int>(S), f32(*work, "work"), stream())) return;
  }
  TORCH_CHECK(mxs::launch_column_scan(p, static_cast<int>(S), kind, bf, stream()), "column scan: key / state size beyond 256");
}

void ssd_scan(at::Tensor out, at::Tensor x, at::Tensor B, at::Tensor C, at::Tensor dt, at::Tensor dt_bias, at::Tensor A_log,
              at::Tensor D, at::Tensor state, at::Tensor state_rows, int64_t off, at::Tensor qsl, at::Tensor seq_lens,
              int64_t H, int64_t G, int64_t N, int64_t P, int64_t piece, int64_t npieces, OptT sc_local, OptT sc_start,
              OptT sc_decay, int64_t max_q) {
  column_scan(mxs::kStateSpace, out, C, B, x, OptT(dt), OptT(), OptT(dt_bias), OptT(A_log), OptT(D), state, state_rows, off, qsl, seq_lens, H, G, N, P,
              1.0, 0.0, piece, npieces, sc_local, sc_start, sc_decay, 0, max_q);
}

void delta_scan(at::Tensor out, at::Tensor q, at::Tensor k, at::Tensor v, at::Tensor beta, at::Tensor a, at::Tensor dt_bias,
                at::Tensor A_log, at::Tensor state, at::Tensor state_rows, int64_t off, at::Tensor qsl, at::Tensor seq_lens,
                int64_t H, int64_t G, int64_t dk, int64_t dv, double q_scale, double unit_eps, int64_t mode, int64_t piece,
                int64_t npieces, OptT sc_local, OptT sc_start, int64_t max_q, OptT work) {
  column_scan(mxs::kDeltaRule, out, q, k, v, OptT(beta), OptT(a), OptT(dt_bias), OptT(A_log), OptT(), state, state_rows, off, qsl, seq_lens, H, G, dk, dv,
              q_scale, unit_eps, piece, npieces, sc_local, sc_start, OptT(), mode, max_q, work);
}

void gla_scan(at::Tensor out, at::Tensor q, at::Tensor k, at::Tensor v, at::Tensor loga, at::Tensor state,
              at::Tensor state_rows, int64_t off, at::Tensor qsl, at::Tensor seq_lens, int64_t H, int64_t dk, int64_t dv,
              double q_scale, int64_t piece, int64_t npieces, OptT sc_local, OptT sc_start, OptT sc_decay, int64_t max_q) {
  column_scan(mxs::kGatedLinear, out, q, k, v, OptT(), OptT(loga), OptT(), OptT(), OptT(), state, state_rows, off, qsl, seq_lens,
              H, H, dk, dv, q_scale, 0.0, piece, npieces, sc_local, sc_start, sc_decay, 0, max_q);
}

void decay_lowrank(at::Tensor out, at::Tensor x, at::Tensor w, at::Tensor bias, double tau) {
  const bool bf = is_bf(x);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && w.is_cuda() && w.is_contiguous() && is_bf(w) == bf && w.size(1) == x.size(1),
              "decay_lowrank: x [T, R], w [N, R] of one dtype");
  const int64_t T = x.size(0), N = w.size(0), R = w.size(1);
  float* op = f32(out, "out");
  TORCH_CHECK(out.dim() == 2 && out.size(0) == T && out.size(1) == N && tau != 0.0, "out: fp32 [T, N]; tau");
  TORCH_CHECK(mxs::launch_decay_lowrank(op, mat(x, bf, T, R, "x"), x.stride(0), w.data_ptr(), vec(OptT(bias), bf, N, "bias"),
                                        static_cast<int>(T), static_cast<int>(N), static_cast<int>(R), static_cast<float>(tau),
                                        bf, stream()), "decay_lowrank: inner size beyond what the kernel holds");
}

// ---- several residual streams, activations (streams.hip)
void streams_start(at::Tensor X, at::Tensor h, at::Tensor ids, at::Tensor table, at::Tensor w_in, at::Tensor norm_w, double eps,
                   double w_offset) {
  float* xp = f32(X, "X");
  const bool bf = is_bf(table);
  TORCH_CHECK(X.dim() == 3 && table.is_cuda() && table.dim() == 2 && table.is_contiguous() && table.size(1) == X.size(2),
              "X [T, n, W], table [V, W]");
  const int64_t T = X.size(0), n = X.size(1), W = X.size(2);
  TORCH_CHECK(ids.is_cuda() && ids.scalar_type() == at::kLong && ids.is_contiguous() && ids.numel() == T, "ids: int64 [T]");
  TORCH_CHECK(h.is_cuda() && h.is_contiguous() && h.dim() == 2 && h.size(0) == T && h.size(1) == W && is_bf(h) == bf, "h: [T, W]");
  TORCH_CHECK(w_in.numel() == n, "w_in: [n]");
  TORCH_CHECK(mxs::launch_streams(xp, static_cast<int>(n), table.data_ptr(), W, ids.data_ptr<int64_t>(), table.size(0), nullptr,
                                  nullptr, f32(w_in, "w_in"), vec(OptT(norm_w), bf, W, "norm_w"), h.data_ptr(),
                                  static_cast<int>(T), static_cast<int>(W), static_cast<float>(eps),
                                  static_cast<float>(w_offset), bf, stream()), "more streams than the kernel holds (32)");
}

void streams_update(at::Tensor X, at::Tensor y, OptT bias, OptT scale, at::Tensor coeffs, at::Tensor norm_w, at::Tensor h,
                    double eps, double w_offset) {
  float* xp = f32(X, "X");
  const bool bf = is_bf(y);
  TORCH_CHECK(X.dim() == 3, "X [T, n, W]");
  const int64_t T = X.size(0), n = X.size(1), W = X.size(2);
  TORCH_CHECK(h.is_cuda() && h.is_contiguous() && h.dim() == 2 && h.size(0) == T && h.size(1) == W && is_bf(h) == bf, "h: [T, W]");
  TORCH_CHECK(coeffs.numel() == n * n + 2 * n, "coeffs: [n * n + 2 n]");
  TORCH_CHECK(mxs::launch_streams(xp, static_cast<int>(n), mat(y, bf, T, W, "y"), y.stride(0), nullptr, 0,
                                  vec(bias, bf, W, "bias"), vec(scale, bf, W, "scale"), f32(coeffs, "coeffs"),
                                  vec(OptT(norm_w), bf, W, "norm_w"), h.data_ptr(), static_cast<int>(T), static_cast<int>(W),
                                  static_cast<float>(eps), static_cast<float>(w_offset), bf, stream()),
              "more streams than the kernel holds (32)");
}

void act_any(at::Tensor out, at::Tensor x, int64_t kind, bool gated) {
  const bool bf = is_bf(x);
  TORCH_CHECK(kind >= 0 && kind <= 2, "unknown activation");
  TORCH_CHECK(x.dim() == 2 && out.is_cuda() && out.is_contiguous() && out.dim() == 2 && out.size(0) == x.size(0) &&
              out.size(1) * (gated ? 2 : 1) == x.size(1) && is_bf(out) == bf, "x [R, F] (gated: [R, 2F]), out [R, F]");
  mxs::launch_act(out.data_ptr(), mat(x, bf, x.size(0), x.size(1), "x"), x.stride(0), static_cast<int>(x.size(0)),
                  static_cast<int>(out.size(1)), static_cast<int>(kind), gated, bf, stream());
}
void unary_act(at::Tensor out, at::Tensor x, int64_t kind) { act_any(out, x, kind, false); }
void act_mul(at::Tensor out, at::Tensor x, int64_t kind) { act_any(out, x, kind, true); }

// ---- latent attention, routed experts (latent_experts.hip)
// ---- convolved q/k/v and attention in two maps (rotary_conv.hip, differential_attention.hip)
void conv_qkv_cache(at::Tensor q, at::Tensor x, at::Tensor w, OptT bias, at::Tensor state, at::Tensor state_rows, int64_t off,
                    at::Tensor qsl, at::Tensor seq_lens, at::Tensor positions, at::Tensor slots, at::Tensor cache, int64_t koff,
                    int64_t voff, int64_t G, int64_t dk, int64_t dv, int64_t bs, double temp_coef, double temp_every,
                    int64_t max_q) {
  const bool bf = is_bf(x);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && w.is_cuda() && w.is_contiguous() && is_bf(w) == bf && w.size(1) == x.size(1),
              "conv_qkv_cache: x [T, C], w [taps, C] of one dtype");
  const int64_t T = x.size(0), C = x.size(1), taps = w.size(0), S = seq_lens.numel(), QC = C - G * (dk + dv);
  TORCH_CHECK(taps >= 1 && QC >= 1 && q.is_cuda() && q.is_contiguous() && q.dim() == 2 && q.size(0) == T && q.size(1) == QC &&
              is_bf(q) == bf, "q: contiguous [T, C - G (dk + dv)]");
  TORCH_CHECK(temp_every != 0.0, "temp_every must not be zero");
  check_cache(cache, bf, koff, voff, G, dk, dv, bs);
  float* sp = f32(state, "state");
  TORCH_CHECK(state.dim() == 2 && off >= 0 && off + (taps - 1) * C <= state.size(1), "state slot too small for this filter");
  mxs::launch_conv_qkv_cache(q.data_ptr(), mat(x, bf, T, C, "x"), x.stride(0), w.data_ptr(), vec(bias, bf, C, "bias"), sp,
                             state.stride(0), i32(state_rows, S, "state_rows"), off, i32(qsl, S + 1, "qsl"),
                             i32(seq_lens, S, "seq_lens"), static_cast<int>(S), static_cast<int>(T),
                             i64(positions, T, "positions"), i64(slots, T, "slot_mapping"), cache.data_ptr(),
                             cache.stride(0), static_cast<int>(koff), static_cast<int>(voff), static_cast<int>(QC),
                             static_cast<int>(G), static_cast<int>(dk), static_cast<int>(dv), static_cast<int>(bs),
                             static_cast<int>(taps), static_cast<float>(temp_coef), static_cast<float>(temp_every),
                             max_q == 1 && T == S, bf, stream());
}

int64_t differential_tiles(int64_t max_q, int64_t rep) {
  return mxs::differential_tiles(static_cast<int>(max_q), static_cast<int>(rep));
}

void differential_attention(at::Tensor out, at::Tensor q, at::Tensor cache, at::Tensor block_tables, at::Tensor qsl,
                            at::Tensor seq_lens, int64_t koff, int64_t voff, int64_t H, int64_t G, int64_t dk, int64_t dv,
                            int64_t bs, double scale, double softcap, double lam, double out_scale, double eps, OptT gate,
                            int64_t max_q, int64_t nsplit, OptT part) {
  const bool bf = is_bf(q);
  const int64_t T = q.size(0), S = seq_lens.numel();
  check_cache(cache, bf, koff, voff, G, 2 * dk, dv, bs);
  TORCH_CHECK(G >= 1 && H % G == 0 && dk >= 1 && dv >= 1, "query heads must divide over kv heads");
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && out.dim() == 2 && out.size(0) == T && out.size(1) == H * dv &&
              is_bf(out) == bf, "out: [T, H*dv]");
  TORCH_CHECK(block_tables.is_cuda() && block_tables.scalar_type() == at::kInt && block_tables.dim() == 2 &&
              block_tables.size(0) >= S && block_tables.size(1) >= 1 && block_tables.stride(1) == 1 &&
              block_tables.stride(0) >= block_tables.size(1), "block_tables: int32 [S, max_blocks]");
  mxs::DiffArgs a{};
  a.out = out.data_ptr();
  a.q = mat(q, bf, T, H * 2 * dk, "q");
  a.q_stride = q.stride(0);
  a.cache = cache.data_ptr();
  a.block_stride = cache.stride(0);
  a.block_tables = block_tables.data_ptr<int>();
  a.bt_stride = static_cast<int>(block_tables.stride(0));
  a.qsl = i32(qsl, S + 1, "qsl");
  a.seq_lens = i32(seq_lens, S, "seq_lens");
  a.n_rows = static_cast<int>(T);
  a.koff = static_cast<int>(koff);
  a.voff = static_cast<int>(voff);
  a.H = static_cast<int>(H);
  a.G = static_cast<int>(G);
  a.dk = static_cast<int>(dk);
  a.dv = static_cast<int>(dv);
  a.max_q = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(max_q, T)));
  a.scale = static_cast<float>(scale);
  a.softcap = static_cast<float>(softcap);
  a.lam = static_cast<float>(lam);
  a.out_scale = static_cast<float>(out_scale);
  a.eps = static_cast<float>(eps);
  if (gate.has_value()) {
    a.gate = mat(*gate, bf, T, H * dv, "gate");
    a.gate_stride = gate->stride(0);
  }
  a.nsplit = 1;
  if (nsplit > 1 && part.has_value()) {
    TORCH_CHECK(part->numel() >= T * H * 2 * nsplit * (dv + 4), "part: fp32 [T, H, 2, nsplit, dv + 4]");
    a.part = f32(*part, "part");
    a.nsplit = static_cast<int>(nsplit);
  }
  TORCH_CHECK(mxs::launch_differential_attention(a, static_cast<int>(S), static_cast<int>(bs), bf, stream()),
              "differential_attention: sizes beyond what the kernels hold (dv <= 512)");
}

void route_grouped(at::Tensor w, at::Tensor ids, at::Tensor logits, OptT correction, int64_t groups, int64_t keep, double scale,
                   bool renorm, bool softmax) {
  const float* lp = f32(logits, "logits");
  TORCH_CHECK(logits.dim() == 2 && w.dim() == 2 && ids.dim() == 2, "logits [T, E], w / ids [T, k]");
  const int64_t T = logits.size(0), E = logits.size(1), k = w.size(1);
  TORCH_CHECK(groups >= 1 && E % groups == 0 && keep >= 1 && keep <= groups && k >= 1 && k <= keep * (E / groups) &&
              w.size(0) == T && ids.size(0) == T && ids.size(1) == k, "k of E experts in the best groups; w, ids [T, k]");
  TORCH_CHECK(ids.is_cuda() && ids.scalar_type() == at::kInt && ids.is_contiguous(), "ids: contiguous int32");
  TORCH_CHECK(mxs::launch_route_grouped(f32(w, "w"), ids.data_ptr<int>(), lp, f32n(correction, E, "correction"),
                                        static_cast<int>(T), static_cast<int>(E), static_cast<int>(k), static_cast<int>(groups),
                                        static_cast<int>(keep), static_cast<float>(scale), renorm, softmax, stream()),
              "route_grouped: more experts than the kernel holds");
}

void latent_prep(at::Tensor cq, at::Tensor dq, at::Tensor dkv, at::Tensor positions, at::Tensor slots, at::Tensor cache,
                 int64_t koff, int64_t rank, int64_t bs, at::Tensor freqs, at::Tensor q_norm, at::Tensor kv_norm,
                 double eps, bool split_pairs, double mag) {
  const bool bf = is_bf(dq);
  const int64_t T = dq.size(0), qr = dq.size(1), nf = freqs.numel(), dk = rank + 2 * nf;
  TORCH_CHECK(rank >= 1 && bs >= 1, "rank and block size must be positive");
  check_cache(cache, bf, koff, koff, 1, dk, 0, bs);
  TORCH_CHECK(cq.is_cuda() && cq.is_contiguous() && cq.dim() == 2 && cq.size(0) == T && cq.size(1) == qr && is_bf(cq) == bf,
              "cq: contiguous [T, q_rank]");
  mxs::launch_latent_prep(cq.data_ptr(), mat(dq, bf, T, qr, "dq"), dq.stride(0), mat(dkv, bf, T, dk, "dkv"), dkv.stride(0),
                          i64(positions, T, "positions"), i64(slots, T, "slot_mapping"), cache.data_ptr(), cache.stride(0),
                          static_cast<int>(T), static_cast<int>(koff), static_cast<int>(qr), static_cast<int>(rank),
                          static_cast<int>(nf), static_cast<int>(bs), f32(freqs, "freqs"),
                          vec(OptT(q_norm), bf, qr, "q_norm"), vec(OptT(kv_norm), bf, rank, "kv_norm"),
                          static_cast<float>(eps), split_pairs, static_cast<float>(mag), bf, stream());
}

// The matrix-core latent attention (bf16).  Returns false when the sizes are not the kernel's: nothing
// was launched and the caller runs window_attention with strided value rows instead.
bool latent_attention(at::Tensor out, at::Tensor q, at::Tensor cache, at::Tensor block_tables, at::Tensor qsl,
                      at::Tensor seq_lens, int64_t koff, int64_t H, int64_t dk, int64_t rank, int64_t bs, double scale,
                      int64_t max_query_len, OptT sink, int64_t nsplit, OptT part, bool pair, int64_t window) {
  if (!is_bf(q)) return false;
  TORCH_CHECK(window >= 0 && window < (1LL << 30), "window out of range");
  const float* sinkp = nullptr;
  if (sink.has_value()) {
    sinkp = f32(*sink, "sink");
    TORCH_CHECK(sink->numel() == H, "sink: fp32 [H]");
  }
  const int64_t T = q.size(0), S = seq_lens.numel();
  TORCH_CHECK(rank >= 1 && rank <= dk && H >= 1, "1 <= rank <= dk");
  check_cache(cache, true, koff, koff, 1, dk, 0, bs);
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && out.dim() == 2 && out.size(0) == T && out.size(1) == H * rank &&
              is_bf(out), "out: bf16 [T, H*rank]");
  TORCH_CHECK(block_tables.is_cuda() && block_tables.scalar_type() == at::kInt && block_tables.dim() == 2 &&
              block_tables.size(0) >= S && block_tables.stride(1) == 1, "block_tables: int32 [S, max_blocks]");
  float* pp = nullptr;
  if (nsplit > 1) {
    TORCH_CHECK(part.has_value() && part->numel() >= T * H * nsplit * (rank + 4), "part: fp32 [T*H, nsplit, rank + 4]");
    pp = f32(*part, "part");
  }
  return mxs::launch_latent_attention(
      out.data_ptr(), pp, mat(q, true, T, H * dk, "q"), q.stride(0), cache.data_ptr(), cache.stride(0),
      block_tables.data_ptr<int>(), static_cast<int>(block_tables.stride(0)), i32(qsl, S + 1, "qsl"),
      i32(seq_lens, S, "seq_lens"), static_cast<int>(S), static_cast<int>(T), static_cast<int>(koff), static_cast<int>(H),
      static_cast<int>(dk), static_cast<int>(rank), static_cast<int>(bs), static_cast<float>(scale),
      static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(max_query_len, T))), sinkp, static_cast<int>(nsplit), pair,
      static_cast<int>(window), stream());
}

void latent_plan(at::Tensor base, at::Tensor offs, at::Tensor qsl, at::Tensor seq_lens, int64_t window) {
  const int64_t S = seq_lens.numel();
  TORCH_CHECK(window >= 0 && window < (1LL << 30), "window out of range");
  mxs::launch_latent_plan(const_cast<int*>(i32(base, S, "base")), const_cast<int*>(i32(offs, S + 1, "offs")), i32(qsl, S + 1, "qsl"),
                          i32(seq_lens, S, "seq_lens"), static_cast<int>(S), static_cast<int>(window), stream());
}

void latent_rows(at::Tensor out, at::Tensor cache, at::Tensor block_tables, at::Tensor base, at::Tensor offs, int64_t koff,
                 int64_t bs) {
  const int64_t n = out.size(0), dk = out.size(1), S = base.numel();
  check_cache(cache, true, koff, koff, 1, dk, 0, bs);
  TORCH_CHECK(bs == 16 && dk % 8 == 0 && koff % 8 == 0 && cache.stride(0) % 8 == 0 &&
                  reinterpret_cast<uintptr_t>(cache.data_ptr()) % 16 == 0, "latent rows: whole 16-byte pieces in pages of 16");
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && is_bf(out), "out: contiguous bf16 [n, dk]");
  TORCH_CHECK(block_tables.is_cuda() && block_tables.scalar_type() == at::kInt && block_tables.dim() == 2 &&
                  block_tables.size(0) >= S && block_tables.stride(1) == 1, "block_tables: int32 [S, max_blocks]");
  mxs::launch_latent_rows((mxs::bf16_t*)out.data_ptr(), (const mxs::bf16_t*)cache.data_ptr(), cache.stride(0),
                          block_tables.data_ptr<int>(), static_cast<int>(block_tables.stride(0)), i32(base, S, "base"),
                          i32(offs, S + 1, "offs"), static_cast<int>(S), static_cast<int>(n), static_cast<int>(koff),
                          static_cast<int>(dk), stream());
}

bool expanded_attention(at::Tensor out, at::Tensor q, at::Tensor kv, at::Tensor rows, at::Tensor base, at::Tensor qsl,
                        at::Tensor seq_lens, int64_t H, int64_t dn, int64_t dr, int64_t dv, int64_t rank, double scale,
                        int64_t max_query_len, OptT sink, int64_t window, int64_t max_seq_len) {
  const int64_t T = q.size(0), S = seq_lens.numel(), n = kv.size(0);
  TORCH_CHECK(window >= 0 && window < (1LL << 30) && H >= 1 && dn >= 8 && dr >= 8 && dv >= 16, "head sizes out of range");
  mxs::ChunkArgs a{};
  a.q = (const mxs::bf16_t*)mat(q, true, T, H * (dn + dr), "q");
  a.q_stride = q.stride(0);
  a.kx = (const mxs::bf16_t*)mat(kv, true, n, H * (dn + dv), "kv");
  a.x_stride = kv.stride(0);
  a.vx = a.kx + H * dn;
  a.kr = (const mxs::bf16_t*)mat(rows, true, n, rank + dr, "rows") + rank;
  a.r_stride = rows.stride(0);
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && out.dim() == 2 && out.size(0) == T && out.size(1) == H * dv && is_bf(out),
              "out: contiguous bf16 [T, H*dv]");
  if (T == 0 || S == 0 || n == 0) return T == 0;
  if (dn % 8 || dr % 8 || rank % 8 || a.x_stride % 8 || a.r_stride % 8 || a.q_stride % 4 || a.x_stride >= (1LL << 26) ||
      reinterpret_cast<uintptr_t>(a.kx) % 16 || reinterpret_cast<uintptr_t>(a.kr) % 16 || reinterpret_cast<uintptr_t>(a.q) % 8 ||
      (H * dn) % 8)
    return false;
  a.out = (mxs::bf16_t*)out.data_ptr();
  a.qsl = i32(qsl, S + 1, "qsl");
  a.seq_lens = i32(seq_lens, S, "seq_lens");
  a.base = i32(base, S, "base");
  a.S = static_cast<int>(S);
  a.H = a.G = static_cast<int>(H);
  a.dk = static_cast<int>(dn + dr);
  a.dn = static_cast<int>(dn);
  a.dv = static_cast<int>(dv);
  a.nrows = static_cast<int>(n);
  a.scale = static_cast<float>(scale);
  a.window = static_cast<int>(window);
  a.sink = f32n(sink, H, "sink");
  a.rows = static_cast<int>(T);
  a.nsplit = mxs::chunk_attention_splits(T, a.S, a.H, a.G, a.dk, a.dv, window > 0 ? std::min(max_seq_len, window) : max_seq_len);
  at::Tensor part;
  if (a.nsplit > 1) {
    part = at::empty({T * H * a.nsplit * (dv + 4)}, out.options().dtype(at::kFloat));
    a.part = part.data_ptr<float>();
  }
  return mxs::launch_chunk_attention(a, static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(max_query_len, T))), stream());
}

void rope_half_into(at::Tensor out, at::Tensor x, at::Tensor positions, int64_t heads, int64_t x_dim, int64_t x_col,
                    int64_t out_dim, int64_t out_col, at::Tensor freqs, bool split_pairs, double mag) {
  const bool bf = is_bf(x);
  const int64_t T = x.size(0), nf = freqs.numel();
  TORCH_CHECK(x_col >= 0 && out_col >= 0 && x_col + 2 * nf <= x_dim && out_col + 2 * nf <= out_dim,
              "the rotated columns lie outside a head");
  mxs::launch_rope_half_into(const_cast<void*>(mat(out, bf, T, heads * out_dim, "out")), out.stride(0),
                             mat(x, bf, T, heads * x_dim, "x"), x.stride(0), i64(positions, T, "positions"),
                             static_cast<int>(T), static_cast<int>(heads), static_cast<int>(x_dim), static_cast<int>(x_col),
                             static_cast<int>(out_dim), static_cast<int>(out_col), f32(freqs, "freqs"), static_cast<int>(nf),
                             split_pairs, static_cast<float>(mag), bf, stream());
}

void route_topk(at::Tensor w, at::Tensor ids, at::Tensor logits, bool renorm, bool softmax) {
  const float* lp = f32(logits, "logits");
  TORCH_CHECK(logits.dim() == 2 && w.dim() == 2 && ids.dim() == 2, "logits [T, E], w / ids [T, k]");
  const int64_t T = logits.size(0), E = logits.size(1), k = w.size(1);
  TORCH_CHECK(k >= 1 && k <= E && w.size(0) == T && ids.size(0) == T && ids.size(1) == k, "1 <= k <= E; w, ids [T, k]");
  TORCH_CHECK(ids.is_cuda() && ids.scalar_type() == at::kInt && ids.is_contiguous(), "ids: contiguous int32");
  mxs::launch_route_topk(f32(w, "w"), ids.data_ptr<int>(), lp, static_cast<int>(T), static_cast<int>(E),
                         static_cast<int>(k), renorm, softmax, stream());
}

void capped_glu(at::Tensor out, at::Tensor gu, double limit, double alpha) {
  const bool bf = is_bf(gu);
  TORCH_CHECK(gu.is_cuda() && gu.dim() == 2 && gu.size(1) % 2 == 0 && (gu.size(1) == 1 || gu.stride(1) == 1), "gu: [R, 2F]");
  const int64_t R = gu.size(0), F = gu.size(1) / 2;
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && out.dim() == 2 && out.size(0) == R && out.size(1) == F &&
              is_bf(out) == bf, "out: contiguous [R, F]");
  mxs::launch_capped_glu(out.data_ptr(), gu.data_ptr(), gu.stride(0), static_cast<int>(R), static_cast<int>(F),
                         static_cast<float>(limit), static_cast<float>(alpha), bf, stream());
}

void expert_align(at::Tensor offs, at::Tensor inv, at::Tensor ids, int64_t E) {
  const int64_t n = ids.numel();
  TORCH_CHECK(ids.is_cuda() && ids.scalar_type() == at::kInt && ids.is_contiguous(), "ids: contiguous int32");
  TORCH_CHECK(E >= 1 && n < (1LL << 30), "expert count / pair count out of range");
  int* op = const_cast<int*>(i32(offs, E + 1, "offs"));
  int* ip = const_cast<int*>(i32(inv, n, "inv"));
  TORCH_CHECK(mxs::launch_expert_align(op, ip, ids.data_ptr<int>(), static_cast<int>(n), static_cast<int>(E), stream()),
              "expert_align: more experts than the kernel's counters hold");
}

void gather_scaled(at::Tensor xs, at::Tensor h, OptT w, at::Tensor inv, int64_t k) {
  const bool bf = is_bf(h);
  TORCH_CHECK(h.dim() == 2 && k >= 1, "h [T, W], k >= 1");
  const int64_t T = h.size(0), W = h.size(1);
  const float* wp = nullptr;
  if (w.has_value()) {
    TORCH_CHECK(w->dim() == 2 && w->size(0) == T && w->size(1) == k, "w [T, k]");
    wp = f32(*w, "w");
  }
  TORCH_CHECK(xs.is_cuda() && xs.is_contiguous() && xs.dim() == 2 && xs.size(0) == T * k && xs.size(1) == W &&
              is_bf(xs) == bf, "xs: contiguous [T*k, W]");
  // inv comes from expert_align over the same pairs: a permutation of 0 .. T*k-1
  mxs::launch_gather_scaled(xs.data_ptr(), mat(h, bf, T, W, "h"), h.stride(0), wp, i32(inv, T * k, "inv"),
                            static_cast<int>(T * k), static_cast<int>(k), static_cast<int>(W), nullptr, nullptr, 0, 0, nullptr, bf,
                            stream());
}

void gather_slabs(at::Tensor xs, at::Tensor index, at::Tensor h, OptT w, at::Tensor ids, at::Tensor offs, at::Tensor inv) {
  const bool bf = is_bf(h);
  TORCH_CHECK(h.dim() == 2 && ids.dim() == 2 && ids.size(0) == h.size(0) && xs.dim() == 3, "h [T, W], ids [T, k], xs [E, cap, W]");
  const int64_t T = h.size(0), W = h.size(1), k = ids.size(1), E = xs.size(0), cap = xs.size(1);
  const float* wp = nullptr;
  if (w.has_value()) {
    TORCH_CHECK(w->dim() == 2 && w->size(0) == T && w->size(1) == k, "w [T, k]");
    wp = f32(*w, "w");
  }
  TORCH_CHECK(xs.is_cuda() && xs.is_contiguous() && xs.size(2) == W && is_bf(xs) == bf, "xs: contiguous [E, cap, W]");
  TORCH_CHECK(E * cap <= std::numeric_limits<int>::max(), "more rows than an int32 index holds");
  TORCH_CHECK(index.is_cuda() && index.is_contiguous() && index.scalar_type() == at::kInt && index.numel() == T * k, "index int32 [T*k]");
  mxs::launch_gather_scaled(xs.data_ptr(), mat(h, bf, T, W, "h"), h.stride(0), wp, i32(inv, T * k, "inv"),
                            static_cast<int>(T * k), static_cast<int>(k), static_cast<int>(W), i32(ids, T * k, "ids"),
                            i32(offs, E + 1, "offs"), static_cast<int>(E), static_cast<int>(cap), index.data_ptr<int>(), bf, stream());
}

void spread_scaled(at::Tensor xs, at::Tensor h, OptT w, at::Tensor ids) {
  const bool bf = is_bf(h);
  TORCH_CHECK(ids.dim() == 2 && h.dim() == 2 && ids.size(0) == h.size(0) && xs.dim() == 3, "h [T, W], ids [T, k], xs [E, T, W]");
  const int64_t T = h.size(0), W = h.size(1), k = ids.size(1), E = xs.size(0);
  const float* wp = nullptr;
  if (w.has_value()) {
    TORCH_CHECK(w->dim() == 2 && w->size(0) == T && w->size(1) == k, "w [T, k]");
    wp = f32(*w, "w");
  }
  TORCH_CHECK(xs.is_cuda() && xs.is_contiguous() && xs.size(1) == T && xs.size(2) == W && is_bf(xs) == bf,
              "xs: contiguous [E, T, W]");
  TORCH_CHECK(E <= 65535, "more experts than a grid dimension holds");
  mxs::launch_spread_scaled(xs.data_ptr(), mat(h, bf, T, W, "h"), h.stride(0), wp, i32(ids, T * k, "ids"),
                            static_cast<int>(T), static_cast<int>(E), static_cast<int>(k), static_cast<int>(W), bf,
                            stream());
}

void expert_combine(at::Tensor out, at::Tensor ys, OptT index, int64_t k, OptT extra, int64_t row_stride, OptT weights,
                    bool by_expert) {
  const bool bf = is_bf(ys);
  TORCH_CHECK(ys.is_cuda() && ys.is_contiguous() && ys.dim() == 2 && out.is_cuda() && out.is_contiguous() &&
              out.dim() == 2 && out.size(1) == ys.size(1) && is_bf(out) == bf, "ys [R, W], out [T, W]");
  const int64_t T = out.size(0), W = out.size(1), R = ys.size(0);
  const int* ip = nullptr;
  if (index.has_value()) {
    ip = i32(*index, T * k, "index");  // entries are rows of ys: expert_align's places (< T*k), or expert * T + t (< R)
    TORCH_CHECK(T * k <= R, "index reaches past ys");
    // by_expert: entries are experts (route_topk's ids, < R / row_stride) of an [E, row_stride, W] stack
    TORCH_CHECK(!by_expert || (row_stride >= T && R % row_stride == 0), "by_expert: ys is [E, row_stride, W]");
  } else {
    TORCH_CHECK(k >= 1 && row_stride >= T && (k - 1) * row_stride + T <= R, "the k slabs reach past ys");
  }
  const void* ep = extra.has_value() ? mat(*extra, bf, T, W, "extra") : nullptr;
  const float* wp = nullptr;
  if (weights.has_value()) {
    TORCH_CHECK(weights->numel() == T * k, "weights: fp32 [T, k]");
    wp = f32(*weights, "weights");
  }
  mxs::launch_expert_combine(out.data_ptr(), ys.data_ptr(), ip, static_cast<int>(T), static_cast<int>(k), row_stride, ep,
                             extra.has_value() ? extra->stride(0) : 0, static_cast<int>(W), wp, by_expert && index.has_value(), bf,
                             stream());
}

void embed_normed(at::Tensor out, OptT copy, OptT h, at::Tensor ids, at::Tensor table, at::Tensor w, double eps,
                  double w_offset) {
  float* op = f32(out, "out");
  float* cp = nullptr;
  if (copy.has_value()) {
    cp = f32(*copy, "copy");
    TORCH_CHECK(copy->sizes() == out.sizes(), "copy: fp32 [T, W] like out");
  }
  TORCH_CHECK(table.is_cuda() && table.dim() == 2 && table.is_contiguous(), "table: contiguous [vocab, W]");
  const bool bf = is_bf(table);
  const int64_t T = ids.numel(), W = table.size(1);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == T && out.size(1) == W, "out: fp32 [T, W]");
  void* hp = nullptr;
  if (h.has_value()) {
    TORCH_CHECK(h->is_cuda() && h->is_contiguous() && h->dim() == 2 && h->size(0) == T && h->size(1) == W && is_bf(*h) == bf,
                "h: contiguous [T, W] of the table's dtype");
    hp = h->data_ptr();
  }
  mxs::launch_embed_normed(op, cp, hp, i64(ids, T, "ids"), table.data_ptr(), vec(OptT(w), bf, W, "w"), static_cast<int>(T),
                           static_cast<int>(W), table.size(0), static_cast<float>(eps), static_cast<float>(w_offset), bf,
                           stream());
}

void depth_mix(at::Tensor hist, int64_t n, at::Tensor coeffs, OptT h) {
  float* hp = f32(hist, "hist");
  TORCH_CHECK(hist.dim() == 3 && n >= 1 && n < hist.size(0), "hist: fp32 [L, T, W], 1 <= n < L");
  const int64_t T = hist.size(1), W = hist.size(2);
  const float* cp = f32(coeffs, "coeffs");
  TORCH_CHECK(coeffs.numel() == n, "coeffs: fp32 [n]");
  void* op = nullptr;
  bool bf = false;
  if (h.has_value()) {
    TORCH_CHECK(h->is_cuda() && h->is_contiguous() && h->dim() == 2 && h->size(0) == T && h->size(1) == W, "h: contiguous [T, W]");
    bf = is_bf(*h);
    op = h->data_ptr();
  }
  TORCH_CHECK(mxs::launch_depth_mix(hp, T * W, static_cast<int>(n), cp, op, static_cast<int>(T), static_cast<int>(W), bf,
                                    stream()), "depth_mix: more slabs than the kernel's coefficient table holds");
}

void xielu(at::Tensor out, at::Tensor x, at::Tensor ab) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && out.is_cuda() && out.is_contiguous() && out.numel() == x.numel() &&
              out.scalar_type() == x.scalar_type(), "xielu: contiguous tensors of one dtype");
  const float* ap = f32(ab, "ab");
  TORCH_CHECK(ab.numel() == 2, "ab: fp32 [2]");
  mxs::launch_xielu(out.data_ptr(), x.data_ptr(), x.numel(), ap, is_bf(x), stream());
}

// Biases, q / k norms (norm_whole: one over all of a row's heads), rotary turn, q in place, k and v into the pages.
void qkv_prep_cache(at::Tensor q, OptT k, OptT v, at::Tensor positions, at::Tensor slots, at::Tensor cache, int64_t koff,
                    int64_t voff, int64_t H, int64_t G, int64_t dk, int64_t dv, int64_t bs, at::Tensor freqs, double mag,
                    bool split_pairs, OptT bq, OptT bk, OptT bv, OptT q_norm, OptT k_norm, double eps, bool norm_whole) {
  const bool bf = is_bf(q);
  const int64_t T = q.size(0);
  TORCH_CHECK(k.has_value() == v.has_value(), "k and v go together");
  TORCH_CHECK(H >= 1 && G >= 1 && H <= 4096 && G <= 4096 && dk >= 1 && bs >= 1, "head counts / sizes out of range");
  const void *kp = nullptr, *vp = nullptr;
  if (k.has_value()) {
    check_cache(cache, bf, koff, voff, G, dk, dv, bs);
    kp = mat(*k, bf, T, G * dk, "k");
    vp = mat(*v, bf, T, G * dv, "v");
  }
  const int64_t nf = freqs.numel();
  TORCH_CHECK(2 * nf <= dk, "more rotary pairs than the head has dimensions");
  const int64_t nq = norm_whole ? H * dk : dk, nk = norm_whole ? G * dk : dk;
  mxs::launch_qkv_prep_cache(const_cast<void*>(mat(q, bf, T, H * dk, "q")), q.stride(0), kp, k.has_value() ? k->stride(0) : 0,
                             vp, v.has_value() ? v->stride(0) : 0, i64(positions, T, "positions"),
                             i64(slots, T, "slot_mapping"), cache.data_ptr(), cache.stride(0), static_cast<int>(T),
                             static_cast<int>(koff), static_cast<int>(voff), static_cast<int>(H), static_cast<int>(G),
                             static_cast<int>(dk), static_cast<int>(dv), static_cast<int>(bs), f32(freqs, "freqs"),
                             static_cast<int>(nf), static_cast<float>(mag), split_pairs, vec(bq, bf, H * dk, "bias_q"),
                             vec(bk, bf, G * dk, "bias_k"), vec(bv, bf, G * dv, "bias_v"), vec(q_norm, bf, nq, "q_norm"),
                             vec(k_norm, bf, nk, "k_norm"), static_cast<float>(eps), norm_whole ? 2 : 1, bf, stream());
}

void talking_attention(at::Tensor out, at::Tensor q, at::Tensor cache, at::Tensor block_tables, at::Tensor qsl,
                       at::Tensor seq_lens, int64_t koff, int64_t voff, int64_t H, int64_t G, int64_t dk, int64_t dv,
                       int64_t bs, double scale, int64_t window, int64_t keep, int64_t max_query_len, OptT sink,
                       at::Tensor talk, int64_t nsplit, OptT part) {
  const bool bf = is_bf(q);
  const float* sinkp = nullptr;
  if (sink.has_value()) {
    sinkp = f32(*sink, "sink");
    TORCH_CHECK(sink->numel() == H, "sink: fp32 [H]");
  }
  const float* tp = f32(talk, "talk");
  TORCH_CHECK(talk.numel() == H * H, "talk: fp32 [H, H]");
  const int64_t T = q.size(0), S = seq_lens.numel();
  check_cache(cache, bf, koff, voff, G, dk, dv, bs);
  TORCH_CHECK(G >= 1 && H % G == 0, "query heads must divide over kv heads");
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && out.dim() == 2 && out.size(0) == T && out.size(1) == H * dv &&
              is_bf(out) == bf, "out: [T, H*dv]");
  TORCH_CHECK(block_tables.is_cuda() && block_tables.scalar_type() == at::kInt && block_tables.dim() == 2 &&
              block_tables.size(0) >= S && block_tables.stride(1) == 1, "block_tables: int32 [S, max_blocks]");
  float* pp = nullptr;
  TORCH_CHECK(nsplit >= 1 && nsplit <= 64, "1 <= nsplit <= 64");
  if (nsplit > 1) {
    TORCH_CHECK(part.has_value() && part->numel() >= T * H * nsplit * (dv + 4), "part: fp32 [T*H, nsplit, dv + 4]");
    pp = f32(*part, "part");
  }
  const bool ok = mxs::launch_talking_attention(
      out.data_ptr(), mat(q, bf, T, H * dk, "q"), q.stride(0), cache.data_ptr(), cache.stride(0),
      block_tables.data_ptr<int>(), static_cast<int>(block_tables.stride(0)), i32(qsl, S + 1, "qsl"),
      i32(seq_lens, S, "seq_lens"), static_cast<int>(S), static_cast<int>(T), static_cast<int>(koff),
      static_cast<int>(voff), static_cast<int>(H), static_cast<int>(G), static_cast<int>(dk), static_cast<int>(dv),
      static_cast<int>(bs), static_cast<float>(scale), static_cast<int>(window), static_cast<int>(keep),
      static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(max_query_len, T))), sinkp, tp, pp, static_cast<int>(nsplit), bf,
      stream());
  TORCH_CHECK(ok, "talking_attention: more heads or wider heads than the kernel's LDS tables hold, or a split the sizes do not take");
}

}  // namespace

void bind_streams_and_scans(pybind11::module_& m);  // bindings_streams.cpp

PYBIND11_MODULE(_M, m) {
  m.def("resid_update", &resid_update);
  m.def("cast_into", &cast_into);
  m.def("relu_sq", &relu_sq);
  m.def("softcap", &softcap);
  m.def("gated_rms_norm", &gated_rms_norm);
  m.def("gate_linear", &gate_linear);
  m.def("kv_write", &kv_write);
  m.def("window_attention", &window_attention);
  m.def("latent_plan", &latent_plan);
  m.def("latent_rows", &latent_rows);
  m.def("expanded_attention", &expanded_attention);
  m.def("decay_scan", &decay_scan);
  m.def("mlstm_scan", &mlstm_scan);
  m.def("embed_scaled", &embed_scaled);
  m.def("rope_qkv_cache", &rope_qkv_cache);
  m.def("rope_rows", &rope_rows);
  m.def("causal_conv", &causal_conv);
  m.def("gated_norm", &gated_norm);
  m.def("ssd_scan", &ssd_scan);
  m.def("delta_scan", &delta_scan);
  m.def("delta_chunk_floats", [](int64_t dk, int64_t dv) { return mxs::delta_chunk_floats(static_cast<int>(dk), static_cast<int>(dv)); });
  m.def("latent_prep", &latent_prep);
  m.def("rope_half_into", &rope_half_into);
  m.def("latent_attention", &latent_attention);
  m.def("route_topk", &route_topk);
  m.def("capped_glu", &capped_glu);
  m.def("expert_align", &expert_align);
  m.def("gather_scaled", &gather_scaled);
  m.def("gather_slabs", &gather_slabs);
  m.def("spread_scaled", &spread_scaled);
  m.def("expert_combine", &expert_combine);
  m.def("embed_normed", &embed_normed);
  m.def("depth_mix", &depth_mix);
  m.def("xielu", &xielu);
  m.def("qkv_prep_cache", &qkv_prep_cache);
  m.def("talking_attention", &talking_attention);
  m.def("streams_start", &streams_start);
  m.def("streams_update", &streams_update);
  m.def("unary_act", &unary_act);
  m.def("act_mul", &act_mul);
  m.def("conv_qkv_cache", &conv_qkv_cache);
  m.def("differential_tiles", &differential_tiles);
  m.def("differential_attention", &differential_attention);
  m.def("decay_lowrank", &decay_lowrank);
  m.def("gla_scan", &gla_scan);
  m.def("route_grouped", &route_grouped);
  bind_streams_and_scans(m);
}
