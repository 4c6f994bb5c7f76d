"""Sequence-mixer ops beyond rotary softmax attention: a 32-bit residual stream with fused norms,
paged attention with a sliding window and kept first tokens, attention in two subtracted maps, decayed and
gated linear attention, retention, selective scans, the mLSTM matrix memory, several residual streams, gated
output norms, squared ReLU and logit soft-capping.

Like mxserve.ops: GPU tensors run the gfx950 kernels of the in-tree extension `mxserve/_M*.so`
(csrc/mixers/*.hip, activations bf16 or fp32; built by `python setup_ext.py --only M` or on first
use), CPU tensors the PyTorch forms below.  Everything the recurrences touch is fp32: the state
pools, decays, gates, scores and the residual stream.

Batch layout (shared with the attention ops): sequence s owns rows qsl[s]:qsl[s+1] of a step's
flattened tokens; they are the LAST rows of its seq_lens[s] tokens.  A sequence whose first row is
position 0 starts from a zero state, whatever its slot held before.

Paged cache of one attention layer inside the block-major pool `cache` [num_blocks, block_elems]:
K at `koff` as [Hkv, BS, dk], V at `voff` as [Hkv, BS, dv], both token-major.
Recurrent state of one layer inside the slot pool `state` [slots, state_floats] (fp32): decayed
linear attention S [H, dk, dv] at `off`; mLSTM S [H, dk, dv], then n [H, dk], then m [H]; the
column scans (state-space duality, gated delta rule, gated linear attention) and retention S transposed [H, dv, dk], so
that the rows a lane owns are contiguous; the selective scan S transposed [state, channels] (a lane owns a channel); a short causal convolution its last taps - 1 inputs [taps - 1, channels].
"""
from __future__ import annotations

import importlib
import os
import threading
from dataclasses import dataclass
from typing import Optional, Union

import torch
import torch.nn.functional as F

_EXT = None
_LOCK = threading.Lock()


def ext():
    """The mixer kernels' extension; built in-tree on first use when it is missing (hipcc)."""
    global _EXT
    if _EXT is None:
        with _LOCK:
            if _EXT is None:
                try:
                    _EXT = importlib.import_module("mxserve._M")
                except ImportError:
                    import sys
                    root = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
                    if root not in sys.path:
                        sys.path.insert(0, root)
                    import setup_ext
                    setup_ext.build_M()
                    importlib.invalidate_caches()
                    _EXT = importlib.import_module("mxserve._M")
    return _EXT


def _gpu(t: torch.Tensor) -> bool:
    return t.is_cuda and os.environ.get("MXS_FORCE_REFERENCE_OPS", "0") != "1"


def _rms(x: torch.Tensor, eps: float) -> torch.Tensor:
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


# ----------------------------------------------------------------------------- residual stream
def resid_update(x: torch.Tensor, a: Optional[torch.Tensor], eps: float, *, wa: Optional[torch.Tensor] = None,
                 b: Optional[torch.Tensor] = None, wb: Optional[torch.Tensor] = None,
                 bias: Optional[torch.Tensor] = None, assign: bool = False,
                 norm_w: Optional[torch.Tensor] = None, out_dtype: Optional[torch.dtype] = None,
                 a_scale: float = 1.0, w_offset: float = 0.0, wa_offset: float = 0.0,
                 cast_dtype: Optional[torch.dtype] = None):
    """One pass over the fp32 residual stream x [T, W], in place:
        d = a * a_scale            (wa: RMSNorm(a) * (wa_offset + wa))
        d = (d + RMSNorm(b) * wb) / 2      when b is given (two branches, each normed over the width)
        d += bias                  (a [W] vector)
        x = d if assign else x + d
    and, when norm_w is given, returns RMSNorm(x) * (w_offset + norm_w) in out_dtype (the next
    sublayer's input; w_offset = 1 for weights stored as their difference from one, added in fp32).
    Without norm_w, cast_dtype asks for the updated x itself in that dtype (a next sublayer that
    reads the stream un-normed).  a = None leaves x as it is.  All sums and norms in fp32."""
    if _gpu(x):
        h = None
        if norm_w is not None:
            h = torch.empty(x.shape, dtype=out_dtype or norm_w.dtype, device=x.device)
        elif cast_dtype is not None:
            h = torch.empty(x.shape, dtype=cast_dtype, device=x.device)
        ext().resid_update(x, a, wa, b, wb, bias, bool(assign), norm_w, h, float(eps), float(a_scale), float(w_offset),
                           float(wa_offset))
        return h
    if a is not None:
        d = a.float() * a_scale if a_scale != 1.0 else a.float()
        if wa is not None:
            d = _rms(d, eps) * (wa.float() + wa_offset if wa_offset else wa.float())
        if b is not None:
            d = 0.5 * (d + _rms(b.float(), eps) * wb.float())
        if bias is not None:
            d = d + bias.float()
        if assign:
            x.copy_(d)
        else:
            x.add_(d)
    if norm_w is None:
        return None if cast_dtype is None else x.to(cast_dtype, copy=True)
    return (_rms(x, eps) * (norm_w.float() + w_offset if w_offset else norm_w.float())).to(out_dtype or norm_w.dtype)


def embed_normed(ids: torch.Tensor, table: torch.Tensor, w: torch.Tensor, eps: float, w_offset: float,
                 out: torch.Tensor, cast_dtype: Optional[torch.dtype] = None, copy: Optional[torch.Tensor] = None):
    """out (fp32 [T, W], may be one slab of a larger buffer) = RMSNorm(table[ids]) * (w_offset + w): an
    embedding that is normed before it becomes the stream; `copy` receives the same (a second slab that a
    layer then updates in place).  Returns out in cast_dtype when asked."""
    if _gpu(table):
        h = torch.empty(out.shape, dtype=cast_dtype, device=out.device) if cast_dtype is not None else None
        ext().embed_normed(out, copy, h, ids, table, w, float(eps), float(w_offset))
        return h
    out.copy_(_rms(F.embedding(ids, table).float(), eps) * (w.float() + w_offset))
    if copy is not None:
        copy.copy_(out)
    return None if cast_dtype is None else out.to(cast_dtype, copy=True)


def depth_mix(hist: torch.Tensor, n: int, coeffs: torch.Tensor, cast_dtype: Optional[torch.dtype] = None):
    """hist fp32 [L, T, W]: slab n <- sum over j < n of coeffs[j] * slab j (coeffs fp32 [n]): a stream
    that goes on as a weighted sum of everything earlier layers produced.  Returns the new slab in
    cast_dtype when asked.  fp32 products and sums, in the order of j."""
    if not 0 < n < hist.shape[0] or coeffs.numel() != n:
        raise ValueError(f"depth_mix: slab {n} of {hist.shape[0]} with {coeffs.numel()} coefficients")
    if _gpu(hist):
        h = torch.empty(hist.shape[1:], dtype=cast_dtype, device=hist.device) if cast_dtype is not None else None
        ext().depth_mix(hist, int(n), coeffs, h)
        return h
    acc = hist[0] * coeffs[0]
    for j in range(1, n):
        acc = acc + hist[j] * coeffs[j]
    hist[n].copy_(acc)
    return None if cast_dtype is None else hist[n].to(cast_dtype, copy=True)


def cast_into(dst: torch.Tensor, x: torch.Tensor) -> None:
    """dst[:, :W] = x (fp32 -> dst's dtype); dst may be a wider row-strided buffer."""
    if _gpu(x):
        ext().cast_into(dst, x)
    else:
        dst[:, :x.shape[1]].copy_(x)


@dataclass
class ExpertRows:
    """A routed feed-forward's result before its sum: out[t] = sum_j weights[t, j] ys[row(t, j)] (+ gate[t] extra[t])
    with row(t, j) as in expert_combine.  A layer's stream update takes the sum on its way into the stream."""
    ys: torch.Tensor
    index: Optional[torch.Tensor]
    k: int
    T: int
    extra: Optional[torch.Tensor] = None
    row_stride: int = 0
    weights: Optional[torch.Tensor] = None
    by_expert: bool = False
    gate: Optional[torch.Tensor] = None  # fp32 [T], what extra is multiplied by

    def sum32(self) -> torch.Tensor:
        """The sum as fp32 (PyTorch form)."""
        y2, k, T = self.ys.reshape(-1, self.ys.shape[-1]), self.k, self.T
        if self.index is None:
            idx = (torch.arange(k).view(1, k) * self.row_stride + torch.arange(T).view(T, 1)).reshape(-1)
        elif self.by_expert:
            idx = (self.index.long().view(T, k) * self.row_stride + torch.arange(T).view(T, 1)).reshape(-1)
        else:
            idx = self.index.long()
        rows = y2[idx].float().view(T, k, -1)
        if self.weights is not None:
            rows = rows * self.weights.float().view(T, k, 1)
        acc = rows.sum(1)
        if self.extra is not None:
            acc = acc + (self.extra.float() if self.gate is None else self.extra.float() * self.gate.view(T, 1))
        return acc


def _norm_rows(x: torch.Tensor, w: torch.Tensor, b: Optional[torch.Tensor], eps: float, center: bool) -> torch.Tensor:
    if center:
        x = x - x.mean(-1, keepdim=True)
    y = _rms(x, eps) * w.float()
    return y if b is None else y + b.float()


def stream_update(x: torch.Tensor, y: Union[torch.Tensor, ExpertRows, None], eps: float, *,
                  scale: Optional[torch.Tensor] = None, mult: float = 1.0, add: Optional[torch.Tensor] = None,
                  norm_w: Optional[torch.Tensor] = None, norm_b: Optional[torch.Tensor] = None, center: bool = True,
                  out_dtype: Optional[torch.dtype] = None) -> Optional[torch.Tensor]:
    """One pass over the fp32 stream x [T, W], in place:
        x <- x + mult * (y * scale) + add      (scale [W]: a layer scale; add fp32 [T, W]: an earlier stream that comes in
                                                once more; y an ExpertRows: its weighted sum; each may be absent)
    and, when norm_w is given, the next sublayer's input in out_dtype: layer norm of x (center: mean taken off, divided
    by the root of the mean squared deviation + eps) or RMS norm, times norm_w, plus norm_b.  All sums in fp32."""
    rows = isinstance(y, ExpertRows)
    if _gpu(x):
        h = None
        if norm_w is not None:
            h = torch.empty(x.shape, dtype=out_dtype or norm_w.dtype, device=x.device)
        if rows:
            ext().stream_update_experts(x, y.ys.view(-1, y.ys.shape[-1]), y.index, y.k, y.extra, y.gate, int(y.row_stride), y.weights,
                                        bool(y.by_expert), scale, add, norm_w, norm_b, h, float(mult), float(eps), bool(center))
        else:
            ext().stream_update(x, y, scale, add, norm_w, norm_b, h, float(mult), float(eps), bool(center))
        return h
    if y is not None:
        d = y.sum32() if rows else y.float()
        x.add_((d if scale is None else d * scale.float()) * mult)
    if add is not None:
        x.add_(add)
    return None if norm_w is None else _norm_rows(x, norm_w, norm_b, eps, center).to(out_dtype or norm_w.dtype)


def bigram_embed(ids: torch.Tensor, table: torch.Tensor, pairs: Optional[torch.Tensor], mul_prev: int, mul_cur: int,
                 state: Optional[torch.Tensor], state_rows: torch.Tensor, off: int, qsl: torch.Tensor,
                 seq_lens: torch.Tensor, norm_w: torch.Tensor, norm_b: Optional[torch.Tensor], eps: float,
                 out_dtype: torch.dtype, center: bool = True, keep: bool = False) -> tuple:
    """The stream's start and the first sublayer's input: x[t] = table[id] + pairs[(prev * mul_prev + id * mul_cur) mod n],
    n = rows of pairs - 1, prev the sequence's token before; row n for a sequence's first token.  The token before a
    chunk's first one is in the sequence's slot at `off` (int32 bits), and the chunk's last token is left there.
    pairs None: x[t] = table[id].  -> (x fp32 [T, W], a copy of x when `keep`, norm of x in out_dtype)."""
    T, W = ids.shape[0], table.shape[1]
    if _gpu(table):
        x = torch.empty(T, W, dtype=torch.float32, device=table.device)
        x0 = torch.empty_like(x) if keep else None
        h = torch.empty(T, W, dtype=out_dtype, device=table.device)
        ext().bigram_embed(x, x0, h, ids, table, pairs, int(mul_prev), int(mul_cur), state, state_rows, int(off), qsl, seq_lens,
                           norm_w, norm_b, float(eps), bool(center))
        return x, x0, h
    x = F.embedding(ids, table).float()
    if pairs is not None:
        n = pairs.shape[0] - 1
        row = torch.empty(T, dtype=torch.long)
        ql, sl, rows = qsl.tolist(), seq_lens.tolist(), state_rows.tolist()
        for s in range(len(sl)):
            a, e = ql[s], ql[s + 1]
            if e <= a:
                continue
            kept = state[rows[s], off:off + 1].view(torch.int32)
            cur = ids[a:e].long()
            prev = torch.cat([kept.long(), cur[:-1]])
            row[a:e] = (prev * int(mul_prev) + cur * int(mul_cur)) % n
            if sl[s] - (e - a) <= 0:
                row[a] = n
            kept.fill_(int(cur[-1]))
        x = x + F.embedding(row, pairs).float()
    return x, (x.clone() if keep else None), _norm_rows(x, norm_w, norm_b, eps, center).to(out_dtype)


# ----------------------------------------------------------------------------- several residual streams
def streams_start(ids: torch.Tensor, table: torch.Tensor, streams: int, w_in: torch.Tensor, norm_w: torch.Tensor,
                  eps: float, w_offset: float, out_dtype: torch.dtype) -> tuple:
    """n = `streams` residual streams that all begin as the embedding.  w_in fp32 [n]: what the first sublayer
    reads is u = sum_s w_in[s] x_s.  -> (X fp32 [T, n, W], RMSNorm(u) * (w_offset + norm_w) in out_dtype)."""
    T, W = ids.shape[0], table.shape[1]
    if _gpu(table):
        X = torch.empty(T, streams, W, dtype=torch.float32, device=table.device)
        h = torch.empty(T, W, dtype=out_dtype, device=table.device)
        ext().streams_start(X, h, ids, table, w_in, norm_w, float(eps), float(w_offset))
        return X, h
    e = F.embedding(ids, table).float()
    X = e.unsqueeze(1).expand(T, streams, W).contiguous()
    u = torch.einsum("s,tsw->tw", w_in, X)
    return X, (_rms(u, eps) * (norm_w.float() + w_offset)).to(out_dtype)


def streams_update(X: torch.Tensor, y: torch.Tensor, coeffs: torch.Tensor, eps: float, norm_w: torch.Tensor,
                   out_dtype: torch.dtype, *, bias: Optional[torch.Tensor] = None,
                   scale: Optional[torch.Tensor] = None, w_offset: float = 0.0) -> torch.Tensor:
    """One pass over n fp32 residual streams X [T, n, W], in place, all streams at once from the old ones:
        d = (y + bias) * scale          (bias, scale [W]; either may be absent)
        x_t <- sum_s mix[s, t] x_s + w_out[t] d
    and the next sublayer's input, RMSNorm(sum_s w_in[s] x_s) * (w_offset + norm_w) of the new streams, in
    out_dtype.  coeffs fp32 [n * n + 2 n] = mix ([from, to], row-major) | w_out | w_in.  All sums in fp32."""
    n = X.shape[1]
    if coeffs.numel() != n * n + 2 * n:
        raise ValueError(f"streams_update: {coeffs.numel()} coefficients for {n} streams")
    if _gpu(X):
        h = torch.empty(X.shape[0], X.shape[2], dtype=out_dtype, device=X.device)
        ext().streams_update(X, y, bias, scale, coeffs, norm_w, h, float(eps), float(w_offset))
        return h
    d = y.float()
    if bias is not None:
        d = d + bias.float()
    if scale is not None:
        d = d * scale.float()
    mix, w_out, w_in = coeffs[:n * n].view(n, n), coeffs[n * n:n * n + n], coeffs[n * n + n:]
    X.copy_(torch.einsum("st,bsw->btw", mix, X) + w_out.view(1, n, 1) * d.unsqueeze(1))
    u = torch.einsum("s,tsw->tw", w_in, X)
    return (_rms(u, eps) * (norm_w.float() + w_offset)).to(out_dtype)


def relu_sq(x: torch.Tensor) -> torch.Tensor:
    """max(x, 0)^2, computed in fp32."""
    if _gpu(x):
        out = torch.empty_like(x)
        ext().relu_sq(out, x)
        return out
    return F.relu(x.float()).square().to(x.dtype)


def xielu(x: torch.Tensor, ab: torch.Tensor) -> torch.Tensor:
    """ab fp32 [2] = (a, b), both positive:  z > 0: a z^2 + z / 2;  z <= 0: b (e^z - 1 - z) + z / 2.
    Computed in fp32."""
    if _gpu(x):
        out = torch.empty_like(x)
        ext().xielu(out, x, ab)
        return out
    z = x.float()
    zn = z.clamp(max=0.0)
    return torch.where(z > 0, ab[0] * z * z + 0.5 * z, ab[1] * (torch.expm1(zn) - zn) + 0.5 * z).to(x.dtype)


ACTS = {"silu": 0, "gelu_erf": 1, "gelu_tanh": 2}


def _act(z: torch.Tensor, kind: str) -> torch.Tensor:
    if kind == "silu":
        return F.silu(z)
    return F.gelu(z, approximate="tanh" if kind == "gelu_tanh" else "none")


def unary_act(x: torch.Tensor, kind: str) -> torch.Tensor:
    """act(x) with kind in silu | gelu_erf (the exact form) | gelu_tanh; computed in fp32."""
    if _gpu(x):
        out = torch.empty_like(x)
        ext().unary_act(out, x, ACTS[kind])
        return out
    return _act(x.float(), kind).to(x.dtype)


def act_mul(gu: torch.Tensor, kind: str) -> torch.Tensor:
    """act(gu[:, :F]) * gu[:, F:] of a fused gate/up projection [T, 2F]; fp32 inside."""
    Fh = gu.shape[1] // 2
    if _gpu(gu):
        out = torch.empty(gu.shape[0], Fh, dtype=gu.dtype, device=gu.device)
        ext().act_mul(out, gu, ACTS[kind])
        return out
    return (_act(gu[:, :Fh].float(), kind) * gu[:, Fh:].float()).to(gu.dtype)


def softcap(x: torch.Tensor, cap: float) -> torch.Tensor:
    """cap * tanh(x / cap) as fp32 (cap <= 0: a plain fp32 copy)."""
    if _gpu(x):
        out = torch.empty(x.shape, dtype=torch.float32, device=x.device)
        ext().softcap(out, x, float(cap))
        return out
    xf = x.float()
    return cap * torch.tanh(xf / cap) if cap > 0 else xf


def gated_rms_norm(o: torch.Tensor, gate: torch.Tensor, w: torch.Tensor, eps: float, groups: int,
                   out_dtype: torch.dtype) -> torch.Tensor:
    """RMSNorm(o) * w * sigmoid(gate).  o fp32 [T, N]; the norm runs over each of `groups` equal
    slices of a row (1: the whole row; H: per head).  gate [T, N] may be a row-strided view."""
    if _gpu(o):
        out = torch.empty(o.shape, dtype=out_dtype, device=o.device)
        ext().gated_rms_norm(out, o, gate, w, float(eps), int(groups))
        return out
    T, N = o.shape
    y = _rms(o.view(T, groups, N // groups), eps).reshape(T, N)
    return (y * w.float() * torch.sigmoid(gate.float())).to(out_dtype)


def gate_linear(h: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
    """fp32 h @ w.T + bias for a handful of output columns (recurrence gates): inputs of any float
    dtype, products and sums in fp32, fp32 out."""
    if _gpu(h):
        out = torch.empty(h.shape[0], w.shape[0], dtype=torch.float32, device=h.device)
        ext().gate_linear(out, h, w, bias)
        return out
    return F.linear(h.float(), w.float(), None if bias is None else bias.float())


# ----------------------------------------------------------------------------- windowed attention
TALK_TARGET_GROUPS = 512  # workgroups (all heads of 16 rows each) that fill the 256 CUs two deep: steps of few rows split their keys up to this


def kv_write(cache: torch.Tensor, k: torch.Tensor, v: torch.Tensor, slot_mapping: torch.Tensor, koff: int,
             voff: int, num_kv_heads: int, dk: int, dv: int, block_size: int) -> None:
    """k [T, Hkv*dk], v [T, Hkv*dv] (row-strided views) into the paged cache; slot -1 writes nothing."""
    if _gpu(k):
        ext().kv_write(cache, k, v, slot_mapping, int(koff), int(voff), num_kv_heads, dk, dv, block_size)
        return
    ok = slot_mapping >= 0
    slots = slot_mapping[ok]
    blk, off = slots // block_size, slots % block_size
    T = int(slots.numel())
    kc = cache[:, koff:koff + num_kv_heads * block_size * dk].view(-1, num_kv_heads, block_size, dk)
    vc = cache[:, voff:voff + num_kv_heads * block_size * dv].view(-1, num_kv_heads, block_size, dv)
    kc[blk, :, off] = k[ok].reshape(T, num_kv_heads, dk).to(cache.dtype)
    vc[blk, :, off] = v[ok].reshape(T, num_kv_heads, dv).to(cache.dtype)


def window_attention(q: torch.Tensor, cache: torch.Tensor, block_tables: torch.Tensor, qsl: torch.Tensor,
                     seq_lens: torch.Tensor, koff: int, voff: int, num_heads: int, num_kv_heads: int, dk: int,
                     dv: int, block_size: int, scale: float, window: int, keep_first: int,
                     max_query_len: int = 0, sink: Optional[torch.Tensor] = None, v_stride: int = 0,
                     talk: Optional[torch.Tensor] = None, max_seq_len: int = 0) -> torch.Tensor:
    """Softmax attention over the paged cache (this step's keys already written).  The query at
    position i sees key j <= i when i - j < window or j < keep_first (window <= 0: every j <= i).
    q [T, H*dk] (row-strided view) -> [T, H*dv] in q's dtype; scores and weights in fp32.
    Query head h reads kv head h // (H / Hkv).  sink (fp32 [H]): the softmax denominator of head h also
    holds exp(sink[h]), a key without a value whose score is not scaled.  v_stride (elements, 0: dv): the
    distance between two tokens' value rows, for values that are a slice of a wider cached row (then
    num_kv_heads is 1 and voff points at the slice inside the first row).  max_query_len: the longest chunk of the step (host
    int); from 16 rows a bf16 step with head sizes that are multiples of 16 runs the MFMA kernel.  max_seq_len (host int,
    0: not known): a bound of the keys, by which long walks of few chunks are split over workgroups.
    talk (fp32 [H, H]): the heads' scaled scores of a (query, key) pair are mixed before the softmax,
    score_h <- sum_g talk[h, g] score_g (the mask and the sink act on the mixed scores); a workgroup then
    serves all heads of its rows, and a bf16 step of few rows splits every row's keys over several
    workgroups (max_seq_len, a host int, bounds how many are worth it) whose stretches are merged."""
    T = q.shape[0]
    if _gpu(q) and talk is not None:
        if v_stride and v_stride != dv:
            raise ValueError("mixed heads read value rows back to back")
        out = torch.empty(T, num_heads * dv, dtype=q.dtype, device=q.device)
        nsplit, part = 1, None
        if q.dtype == torch.bfloat16 and T and block_size == 16 and dk % 16 == 0 and dv % 16 == 0 and dk <= 128 and dv <= 128:
            mq = max(1, min(int(max_query_len) or T, T))
            tiles = seq_lens.numel() * (-(-mq // 16))
            span = int(max_seq_len) or 16
            if window > 0:
                span = min(span, int(window) + int(keep_first) + 15)
            nsplit = max(1, min(16, TALK_TARGET_GROUPS // max(tiles, 1), -(-span // 16) // 2))
            if nsplit > 1:
                part = torch.empty(T * num_heads * nsplit * (dv + 4), dtype=torch.float32, device=q.device)
        ext().talking_attention(out, q, cache, block_tables, qsl, seq_lens, int(koff), int(voff), num_heads, num_kv_heads,
                                dk, dv, block_size, float(scale), int(window), int(keep_first), int(max_query_len), sink,
                                talk, nsplit, part)
        return out
    if _gpu(q):
        out = torch.empty(T, num_heads * dv, dtype=q.dtype, device=q.device)
        ext().window_attention(out, q, cache, block_tables, qsl, seq_lens, int(koff), int(voff), num_heads,
                               num_kv_heads, dk, dv, block_size, float(scale), int(window), int(keep_first),
                               int(max_query_len), sink, int(v_stride), int(max_seq_len))
        return out
    out = torch.zeros(T, num_heads, dv, dtype=torch.float32)
    kc = cache[:, koff:koff + num_kv_heads * block_size * dk].view(-1, num_kv_heads, block_size, dk)
    if v_stride and v_stride != dv:
        if num_kv_heads != 1:
            raise ValueError("strided value rows need a single kv head")
        vc = torch.as_strided(cache, (cache.shape[0], 1, block_size, dv), (cache.stride(0), 0, v_stride, 1),
                              cache.storage_offset() + voff)
    else:
        vc = cache[:, voff:voff + num_kv_heads * block_size * dv].view(-1, num_kv_heads, block_size, dv)
    g = num_heads // num_kv_heads
    ql, sl = qsl.tolist(), seq_lens.tolist()
    for s in range(len(sl)):
        a, e = ql[s], ql[s + 1]
        n = sl[s]
        if e <= a:
            continue
        nb = -(-n // block_size)
        blocks = block_tables[s, :nb].long()
        K = kc[blocks].permute(0, 2, 1, 3).reshape(nb * block_size, num_kv_heads, dk)[:n].float()
        V = vc[blocks].permute(0, 2, 1, 3).reshape(nb * block_size, num_kv_heads, dv)[:n].float()
        qs = q[a:e].reshape(e - a, num_heads, dk).float()
        sc = torch.einsum("mhd,nhd->hmn", qs, K.repeat_interleave(g, dim=1)) * scale
        if talk is not None:
            sc = torch.einsum("hg,gmn->hmn", talk.float(), sc)
        i = torch.arange(n - (e - a), n).unsqueeze(1)
        j = torch.arange(n).unsqueeze(0)
        seen = j <= i
        if window > 0:
            seen = seen & ((i - j < window) | (j < keep_first))
        sc = sc.masked_fill(~seen.unsqueeze(0), float("-inf"))
        if sink is not None:  # one more column, dropped after the softmax: it has no value
            sc = torch.cat([sc, sink.float().view(-1, 1, 1).expand(-1, sc.shape[1], 1)], dim=-1)
        p = torch.softmax(sc, dim=-1)[..., :n]
        out[a:e] = torch.einsum("hmn,nhd->mhd", p, V.repeat_interleave(g, dim=1))
    return out.reshape(T, num_heads * dv).to(q.dtype)


# ----------------------------------------------------------------------------- recurrences
SCAN_PIECE = int(os.environ.get("MXS_SCAN_PIECE", "0"))  # tokens per piece of a time-split scan; 0: by the launch's size
SCAN_SCRATCH_BYTES = 512 << 20
SCAN_TARGET_BLOCKS = 1024  # workgroups that fill the 256 CUs four deep


def _scan_split(S: int, T: int, max_query_len: int, floats: int, heads: int, dv: int, device, spare: bool = False) -> tuple:
    """(piece, npieces, scratch pool, scratch pool) of a scan launch: chunks of 2 pieces or more are cut
    into pieces that run side by side (two passes and a chaining step, csrc/mixers/scan.hip).  Pieces
    are 64 to 256 tokens, as short as it takes to reach SCAN_TARGET_BLOCKS workgroups over the long
    chunks of the step, and grow until both scratch pools [S, npieces, state] fit SCAN_SCRATCH_BYTES.
    spare: with several sequences, an empty piece more where the count is a multiple of 8.  Single tokens beside
    a chunk use their first piece only; at strides of 8 states those meet in few channels of the memory (state
    space, 8 heads of 64 x 128, a chunk of 512 beside 64 single tokens: 130 -> 62 us; 500 more tokens: 144 -> 76)."""
    piece, n = _scan_pieces(S, T, max_query_len, floats, heads, dv, spare)
    if n == 1:
        return 1, 1, None, None
    pool = torch.empty(2, S * n * floats, dtype=torch.float32, device=device)
    return piece, n, pool[0], pool[1]


def _scan_pieces(S: int, T: int, max_query_len: int, floats: int, heads: int, dv: int, spare: bool = False) -> tuple:
    """(piece, npieces) of _scan_split; npieces 1: not cut."""
    max_query_len = min(max_query_len, T)
    if max_query_len < 128:
        return 1, 1
    piece = SCAN_PIECE
    if piece <= 0:
        per_piece = heads * -(-dv // 64) * max(1, T // max_query_len)  # workgroups one piece index adds
        want = -(-SCAN_TARGET_BLOCKS // per_piece)
        piece = 256
        while piece > 64 and -(-max_query_len // piece) < want:
            piece //= 2
    while max_query_len >= 2 * piece:
        n = -(-max_query_len // piece)
        if spare and S > 1 and n % 8 == 0 and 2 * S * (n + 1) * floats * 4 <= SCAN_SCRATCH_BYTES:
            n += 1
        if 2 * S * n * floats * 4 <= SCAN_SCRATCH_BYTES:
            return piece, n
        piece *= 2
    return 1, 1


def decay_scan(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, decay: torch.Tensor, state: torch.Tensor,
               state_rows: torch.Tensor, off: int, qsl: torch.Tensor, seq_lens: torch.Tensor, num_heads: int,
               dk: int, dv: int, silu: bool = True, max_query_len: int = 0) -> torch.Tensor:
    """Decayed linear attention, token by token per head: S = decay_h S + k v^T, o = S^T q, with q, k, v
    passed through SiLU first when `silu`.  q, k [T, H*dk], v [T, H*dv] (row-strided views); decay
    fp32 [H]; returns o fp32 [T, H*dv] and leaves each sequence's S in its slot.  max_query_len: the
    step's longest chunk (host int); long chunks are cut into pieces that run side by side."""
    T = q.shape[0]
    if _gpu(q):
        out = torch.empty(T, num_heads * dv, dtype=torch.float32, device=q.device)
        plan = _scan_split(seq_lens.numel(), T, max_query_len, num_heads * dk * dv, num_heads, dv, q.device)
        ext().decay_scan(out, q, k, v, decay, state, state_rows, int(off), qsl, seq_lens, num_heads, dk, dv,
                         bool(silu), *plan)
        return out
    out = torch.zeros(T, num_heads, dv, dtype=torch.float32)
    qf, kf, vf = (t.float().reshape(T, num_heads, -1) for t in (q, k, v))
    if silu:
        qf, kf, vf = F.silu(qf), F.silu(kf), F.silu(vf)
    ql, sl, rows = qsl.tolist(), seq_lens.tolist(), state_rows.tolist()
    n = num_heads * dk * dv
    for s in range(len(sl)):
        a, e = ql[s], ql[s + 1]
        if e <= a:
            continue
        S = state[rows[s], off:off + n].view(num_heads, dk, dv)
        if sl[s] - (e - a) == 0:
            S.zero_()
        for t in range(a, e):
            S.mul_(decay.view(-1, 1, 1)).add_(kf[t].unsqueeze(2) * vf[t].unsqueeze(1))
            out[t] = torch.einsum("hdv,hd->hv", S, qf[t])
    return out.reshape(T, num_heads * dv)


def mlstm_state_floats(num_heads: int, dk: int, dv: int) -> int:
    return num_heads * (dk * dv + dk + 1)


def mlstm_scan(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, gates: torch.Tensor, state: torch.Tensor,
               state_rows: torch.Tensor, off: int, qsl: torch.Tensor, seq_lens: torch.Tensor, num_heads: int,
               dk: int, dv: int, gate_cap: float, q_scale: float, max_query_len: int = 0) -> torch.Tensor:
    """mLSTM matrix memory, token by token per head.  gates fp32 [T, 2H]: the input gates' then the
    forget gates' pre-activations.  With i = cap tanh(pre_i / cap), f = logsigmoid(cap tanh(pre_f / cap))
    and a running maximum m (0 at the start):
        m' = max(f + m, i);  S = e^(f + m - m') S + e^(i - m') k v^T;  n likewise with k;
        o = S^T q~ / (max(|n . q~|, e^(-m')) + 1e-6),   q~ = q_scale q.
    Returns o fp32 [T, H*dv] (before any norm)."""
    T = q.shape[0]
    if _gpu(q):
        out = torch.empty(T, num_heads * dv, dtype=torch.float32, device=q.device)
        plan = _scan_split(seq_lens.numel(), T, max_query_len, mlstm_state_floats(num_heads, dk, dv) + num_heads,
                           num_heads, dv, q.device)
        ext().mlstm_scan(out, q, k, v, gates, state, state_rows, int(off), qsl, seq_lens, num_heads, dk, dv,
                         float(gate_cap), float(q_scale), *plan)
        return out
    H = num_heads
    out = torch.zeros(T, H, dv, dtype=torch.float32)
    qf = q.float().reshape(T, H, dk) * q_scale
    kf, vf = k.float().reshape(T, H, dk), v.float().reshape(T, H, dv)
    ig = gate_cap * torch.tanh(gates[:, :H] / gate_cap)
    fg = F.logsigmoid(gate_cap * torch.tanh(gates[:, H:] / gate_cap))
    ql, sl, rows = qsl.tolist(), seq_lens.tolist(), state_rows.tolist()
    nS, nn = H * dk * dv, H * dk
    for s in range(len(sl)):
        a, e = ql[s], ql[s + 1]
        if e <= a:
            continue
        st = state[rows[s]]
        S = st[off:off + nS].view(H, dk, dv)
        n = st[off + nS:off + nS + nn].view(H, dk)
        m = st[off + nS + nn:off + nS + nn + H]
        if sl[s] - (e - a) == 0:
            S.zero_(), n.zero_(), m.zero_()
        for t in range(a, e):
            m_new = torch.maximum(fg[t] + m, ig[t])
            fa, ia = torch.exp(fg[t] + m - m_new), torch.exp(ig[t] - m_new)
            S.mul_(fa.view(H, 1, 1)).add_(ia.view(H, 1, 1) * kf[t].unsqueeze(2) * vf[t].unsqueeze(1))
            n.mul_(fa.view(H, 1)).add_(ia.view(H, 1) * kf[t])
            m.copy_(m_new)
            den = torch.maximum((n * qf[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6
            out[t] = torch.einsum("hdv,hd->hv", S, qf[t]) / den.unsqueeze(1)
    return out.reshape(T, H * dv)


# ----------------------------------------------------------------------------- embedding, feed-forward
def embed_scaled(ids: torch.Tensor, table: torch.Tensor, scale: float) -> torch.Tensor:
    """table[ids] * scale as the fp32 residual stream [T, W]."""
    if _gpu(table):
        out = torch.empty(ids.shape[0], table.shape[1], dtype=torch.float32, device=table.device)
        ext().embed_scaled(out, ids, table, float(scale))
        return out
    return F.embedding(ids, table).float() * scale


def silu_mul(gu: torch.Tensor) -> torch.Tensor:
    """SiLU(gu[:, :F]) * gu[:, F:] of a fused gate/up projection [T, 2F]; fp32 inside."""
    Fh = gu.shape[1] // 2
    if _gpu(gu):
        out = torch.empty(gu.shape[0], Fh, dtype=gu.dtype, device=gu.device)
        ext().act_mul(out, gu, ACTS["silu"])
        return out
    return (F.silu(gu[:, :Fh].float()) * gu[:, Fh:].float()).to(gu.dtype)


# ----------------------------------------------------------------------------- rotary positions
def _rotate(x: torch.Tensor, pos: torch.Tensor, freqs: torch.Tensor, sign: float, mag: float = 1.0) -> torch.Tensor:
    """x fp32 [T, heads, dim]: pair (2i, 2i+1) turned by sign * pos * freqs[i]; the rest passes."""
    n = freqs.numel()
    ang = pos.to(torch.float32).view(-1, 1, 1) * freqs.float().view(1, 1, n) * sign
    c, s = torch.cos(ang) * mag, torch.sin(ang) * mag
    u, v = x[..., 0:2 * n:2], x[..., 1:2 * n:2]
    y = x.clone()
    y[..., 0:2 * n:2] = u * c - v * s
    y[..., 1:2 * n:2] = v * c + u * s
    return y


def rope_qkv_cache(q: torch.Tensor, k: Optional[torch.Tensor], v: Optional[torch.Tensor], positions: torch.Tensor,
                   slot_mapping: torch.Tensor, cache: torch.Tensor, koff: int, voff: int, num_heads: int,
                   num_kv_heads: int, dk: int, dv: int, block_size: int, freqs: torch.Tensor,
                   q_norm: Optional[torch.Tensor] = None, k_norm: Optional[torch.Tensor] = None, eps: float = 1e-5,
                   v_freqs: Optional[torch.Tensor] = None, *, bias_q: Optional[torch.Tensor] = None,
                   bias_k: Optional[torch.Tensor] = None, bias_v: Optional[torch.Tensor] = None,
                   norm_whole: bool = False, split_pairs: bool = False, mag: float = 1.0) -> None:
    """Queries, keys and values of a step from the fused projection to what attention reads, in one
    launch.  Per head: optional RMS norm over the head (weight [dk], plain), then interleaved rotary
    pairs (2i, 2i+1) on the first 2 * len(freqs) dimensions by position * freqs[i]; values are
    turned over 2 * len(v_freqs) dimensions when v_freqs is given.  q [T, H*dk] is rewritten in place;
    k [T, G*dk] and v [T, G*dv] go into the paged cache (slot -1: not written).  k = v = None: a layer
    that reads another layer's pages.  Angles, norms and rotations in fp32, one rounding at the end.
    The keyword forms (one launch of a workgroup per token): bias_q / bias_k / bias_v are added first;
    norm_whole: ONE RMS norm over all of q's columns and one over all of k's (weights [H*dk], [G*dk]);
    split_pairs: coordinate i pairs with i + len(freqs) instead of its neighbour; mag multiplies cos and sin."""
    general = bias_q is not None or bias_k is not None or bias_v is not None or norm_whole or split_pairs or mag != 1.0
    if _gpu(q) and general:
        if v_freqs is not None:
            raise ValueError("turned values come with the per-head form only")
        ext().qkv_prep_cache(q, k, v, positions, slot_mapping, cache, int(koff), int(voff), num_heads, num_kv_heads, dk, dv,
                             block_size, freqs, float(mag), bool(split_pairs), bias_q, bias_k, bias_v, q_norm, k_norm,
                             float(eps), bool(norm_whole))
        return
    if _gpu(q):
        ext().rope_qkv_cache(q, k, v, positions, slot_mapping, cache, int(koff), int(voff), num_heads, num_kv_heads,
                             dk, dv, block_size, freqs, q_norm, k_norm, float(eps), v_freqs)
        return
    T = q.shape[0]

    def prep(x, heads, dim, norm_w, fr, bias):
        y = x.float()
        if bias is not None:
            y = y + bias.float()
        if norm_w is not None and norm_whole:
            y = _rms(y, eps) * norm_w.float()
        y = y.reshape(T, heads, dim)
        if norm_w is not None and not norm_whole:
            y = _rms(y, eps) * norm_w.float()
        if fr is None:
            return y
        if split_pairs:
            n = fr.numel()
            return torch.cat([_rotate_half(y[..., :2 * n], positions, fr, mag), y[..., 2 * n:]], dim=-1)
        return _rotate(y, positions, fr, 1.0, mag)

    q.copy_(prep(q, num_heads, dk, q_norm, freqs, bias_q).reshape(T, -1).to(q.dtype))
    if k is None:
        return
    kk = prep(k, num_kv_heads, dk, k_norm, freqs, bias_k).reshape(T, -1).to(k.dtype)
    vv = prep(v, num_kv_heads, dv, None, v_freqs, bias_v).reshape(T, -1).to(v.dtype)
    kv_write(cache, kk, vv, slot_mapping, koff, voff, num_kv_heads, dk, dv, block_size)


def rope_rows(x: torch.Tensor, positions: torch.Tensor, heads: int, dim: int, freqs: torch.Tensor, sign: float,
              out_scale: float, out: torch.Tensor) -> None:
    """out = out_scale * (x with every head's pairs (2i, 2i+1) turned by sign * position * freqs[i]).
    x [T, heads*dim]; out may be a row-strided view of the same shape (a slice of a wider buffer)."""
    if _gpu(x):
        ext().rope_rows(out, x, positions, heads, dim, freqs, float(sign), float(out_scale))
        return
    T = x.shape[0]
    out.copy_((_rotate(x.float().reshape(T, heads, dim), positions, freqs, sign) * out_scale).reshape(T, -1).to(out.dtype))


# ----------------------------------------------------------------------------- short causal convolution
def causal_conv(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], state: torch.Tensor,
                state_rows: torch.Tensor, off: int, qsl: torch.Tensor, seq_lens: torch.Tensor,
                silu: bool = True, max_query_len: int = 0) -> torch.Tensor:
    """Per-channel causal filter over time: y[t, c] = bias[c] + sum_j w[j, c] x[t - (taps-1) + j, c], the
    last row of w weighing the current token, inputs before a sequence's start being zero; then
    SiLU.  x [T, C] (row-strided view), w tap-major [taps, C] (a checkpoint's [C, taps] transposed, so
    that neighbouring channels' weights are neighbours).  The sequence's last taps - 1 inputs live in
    its state slot at `off` as fp32 [taps - 1, C], oldest first, and are replaced by this step's.
    max_query_len (host int) 1: every sequence brings one row, one launch does both."""
    T, C = x.shape
    taps = w.shape[0]
    if _gpu(x):
        out = torch.empty(T, C, dtype=x.dtype, device=x.device)
        ext().causal_conv(out, x, w, bias, state, state_rows, int(off), qsl, seq_lens, bool(silu), int(max_query_len))
        return out
    out = torch.zeros(T, C, dtype=torch.float32)
    ql, sl, rows = qsl.tolist(), seq_lens.tolist(), state_rows.tolist()
    wf = w.float()
    for s in range(len(sl)):
        a, e = ql[s], ql[s + 1]
        if e <= a:
            continue
        n = e - a
        st = state[rows[s], off:off + (taps - 1) * C].view(taps - 1, C)
        prev = torch.zeros(taps - 1, C) if sl[s] - n == 0 else st.clone()
        full = torch.cat([prev, x[a:e].float()])
        y = torch.zeros(n, C) if bias is None else bias.float().expand(n, C).clone()
        for j in range(taps):
            y += wf[j] * full[j:j + n]
        out[a:e] = y
        if taps > 1:
            st.copy_(full[n:])
    return (F.silu(out) if silu else out).to(x.dtype)


def conv_qkv_cache(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], state: torch.Tensor,
                   state_rows: torch.Tensor, off: int, qsl: torch.Tensor, seq_lens: torch.Tensor,
                   positions: torch.Tensor, slot_mapping: torch.Tensor, cache: torch.Tensor, koff: int, voff: int,
                   q_cols: int, num_kv_heads: int, dk: int, dv: int, block_size: int, temp_coef: float = 0.0,
                   temp_every: float = 1.0, max_query_len: int = 0) -> torch.Tensor:
    """Queries, keys and values of a step from the fused projection to what attention reads, for a mixer whose
    q, k, v pass a short causal filter: u = x + bias (x [T, q_cols + G*dk + G*dv], a row-strided view),
    y[t, c] = sum_j w[j, c] u[t - (taps-1) + j, c] as in causal_conv (no bias after it, no activation; the carried
    inputs are u).  Query columns are multiplied by 1 + temp_coef * ln(floor((p + 1) / temp_every) + 1) at position
    p and returned [T, q_cols]; keys and values go into the paged cache (slot -1: not written).  fp32 inside, one
    rounding at the end."""
    T, C = x.shape
    if C != q_cols + num_kv_heads * (dk + dv):
        raise ValueError(f"conv_qkv_cache: {C} columns for {q_cols} query, {num_kv_heads} x ({dk} + {dv}) key / value")
    if _gpu(x):
        q = torch.empty(T, q_cols, dtype=x.dtype, device=x.device)
        ext().conv_qkv_cache(q, x, w, bias, state, state_rows, int(off), qsl, seq_lens, positions, slot_mapping, cache,
                             int(koff), int(voff), num_kv_heads, dk, dv, block_size, float(temp_coef), float(temp_every),
                             int(max_query_len))
        return q
    u = x.float() if bias is None else x.float() + bias.float()
    y = causal_conv(u, w.float(), None, state, state_rows, off, qsl, seq_lens, silu=False)
    q = y[:, :q_cols]
    if temp_coef != 0.0:
        q = q * (1.0 + temp_coef * torch.log(torch.floor((positions.float() + 1.0) / temp_every) + 1.0)).unsqueeze(1)
    nk = num_kv_heads * dk
    kv_write(cache, y[:, q_cols:q_cols + nk], y[:, q_cols + nk:], slot_mapping, koff, voff, num_kv_heads, dk, dv, block_size)
    return q.to(x.dtype)


# ----------------------------------------------------------------------------- attention in two maps
DIFF_TARGET_GROUPS = 512  # workgroups that fill the 256 CUs two deep: steps of few rows split their keys up to this


def differential_attention(q: torch.Tensor, cache: torch.Tensor, block_tables: torch.Tensor, qsl: torch.Tensor,
                           seq_lens: torch.Tensor, koff: int, voff: int, num_heads: int, num_kv_heads: int, dk: int,
                           dv: int, block_size: int, scale: float, softcap: float, lam: float, out_scale: float,
                           eps: float, gate: Optional[torch.Tensor] = None, max_query_len: int = 0,
                           max_seq_len: int = 0, num_singles: int = 0) -> torch.Tensor:
    """Softmax attention in two maps over the same values, causal, through the paged cache (this step's keys
    already written).  Query head h has two queries q [T, H, 2, dk]; a cached key row holds the two keys of a kv
    head (K at `koff` as [G, BS, 2, dk], V at `voff` as [G, BS, dv]); head h reads kv head h // (H / G).
        a_m = softmax over j <= i of cap(scale q_m . k_m,j), times the values        (m = 1, 2)
        o = a_1 - lam a_2;   o <- o / sqrt(mean(o^2) + eps) * out_scale   over dv;   o <- o * sigmoid(gate)
    with cap(s) = softcap tanh(s / softcap) (softcap <= 0: s itself) and gate [T, H*dv] (a row-strided view, optional).
    Scores, weights, both maps' sums and the norm in fp32; returns [T, H*dv] in q's dtype.
    num_singles: so many of the step's leading sequences have one row each (they run a form of their own when the
    step also holds longer chunks); max_query_len / max_seq_len: host bounds on the chunks and contexts."""
    T = q.shape[0]
    if _gpu(q):
        out = torch.empty(T, num_heads * dv, dtype=q.dtype, device=q.device)
        S = seq_lens.numel()
        bf = q.dtype == torch.bfloat16
        mq = max(1, min(int(max_query_len) or T, T))
        span = max(int(max_seq_len) or 16, 16)
        # (first sequence, last sequence, its longest chunk): single tokens apart from chunks in a mixed step
        spans = [(0, S, mq)] if mq == 1 or not 0 < num_singles < S or not bf else [(0, num_singles, 1), (num_singles, S, mq)]
        for s0, s1, m in spans:
            nsplit, part = 1, None
            if bf:
                tiles = (s1 - s0) * num_kv_heads * ext().differential_tiles(m, num_heads // num_kv_heads)
                nsplit = max(1, min(32, DIFF_TARGET_GROUPS // max(tiles, 1), span // 128))
                if nsplit > 1:
                    part = torch.empty(T * num_heads * 2 * nsplit * (dv + 4), dtype=torch.float32, device=q.device)
            ext().differential_attention(out, q, cache, block_tables[s0:s1], qsl[s0:s1 + 1], seq_lens[s0:s1], int(koff),
                                         int(voff), num_heads, num_kv_heads, dk, dv, block_size, float(scale),
                                         float(softcap), float(lam), float(out_scale), float(eps), gate, m, nsplit, part)
        return out
    out = torch.zeros(T, num_heads, dv, dtype=torch.float32)
    G = num_kv_heads
    kc = cache[:, koff:koff + G * block_size * 2 * dk].view(-1, G, block_size, 2, dk)
    vc = cache[:, voff:voff + G * block_size * dv].view(-1, G, block_size, dv)
    rep = num_heads // G
    ql, sl = qsl.tolist(), seq_lens.tolist()
    for s in range(len(sl)):
        a, e = ql[s], ql[s + 1]
        n = sl[s]
        if e <= a:
            continue
        nb = -(-n // block_size)
        blocks = block_tables[s, :nb].long()
        K = kc[blocks].permute(0, 2, 1, 3, 4).reshape(nb * block_size, G, 2, dk)[:n].float().repeat_interleave(rep, dim=1)
        V = vc[blocks].permute(0, 2, 1, 3).reshape(nb * block_size, G, dv)[:n].float().repeat_interleave(rep, dim=1)
        sc = torch.einsum("ihmd,jhmd->hmij", q[a:e].reshape(e - a, num_heads, 2, dk).float(), K) * scale
        if softcap > 0:
            sc = softcap * torch.tanh(sc / softcap)
        i = torch.arange(n - (e - a), n).unsqueeze(1)
        sc = sc.masked_fill(torch.arange(n).unsqueeze(0) > i, float("-inf"))
        am = torch.einsum("hmij,jhd->mihd", torch.softmax(sc, dim=-1), V)
        out[a:e] = am[0] - lam * am[1]
    y = (_rms(out, eps) * out_scale).reshape(T, num_heads * dv)
    if gate is not None:
        y = y * torch.sigmoid(gate.float())
    return y.to(q.dtype)


# ----------------------------------------------------------------------------- column scans
def decay_lowrank(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor, tau: float) -> torch.Tensor:
    """Logarithms of decays from a low-rank pair's inner values: log(sigmoid(w x + bias)) / tau, fp32 [T, N].
    x [T, R] (row-strided view), w [N, R], bias [N]; products and sums in fp32."""
    if _gpu(x):
        out = torch.empty(x.shape[0], w.shape[0], dtype=torch.float32, device=x.device)
        ext().decay_lowrank(out, x, w, bias, float(tau))
        return out
    return F.logsigmoid(F.linear(x.float(), w.float(), bias.float())) / tau


def gla_scan(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, loga: torch.Tensor, state: torch.Tensor,
             state_rows: torch.Tensor, off: int, qsl: torch.Tensor, seq_lens: torch.Tensor, num_heads: int, dk: int,
             dv: int, q_scale: float, max_query_len: int = 0) -> torch.Tensor:
    """Gated linear attention with one decay per head and key channel:
        S <- diag(exp(loga_t)) S + k_t v_t^T,   o_t = S^T (q_scale q_t)
    so the read-out sees the token's own write.  q, k [T, H*dk], v [T, H*dv] (row-strided views), loga fp32
    [T, H*dk] (<= 0).  Returns o fp32 [T, H*dv]; S (fp32, stored [H, dv, dk]) stays in the sequence's slot.
    max_query_len: the step's longest chunk (host int); the step is a diagonal map of the state, so long chunks
    are cut into pieces that run side by side (end states from an empty start, chained by the pieces' summed
    logarithms, then the outputs)."""
    T, H = q.shape[0], num_heads
    if _gpu(q):
        out = torch.empty(T, H * dv, dtype=torch.float32, device=q.device)
        piece, npieces, loc, start = _scan_split(seq_lens.numel(), T, max_query_len, H * dv * dk, H, 4 * dv, q.device)
        dec = torch.empty(seq_lens.numel() * npieces * H * dk, dtype=torch.float32, device=q.device) if npieces > 1 else None
        ext().gla_scan(out, q, k, v, loga, state, state_rows, int(off), qsl, seq_lens, H, dk, dv, float(q_scale), piece,
                       npieces, loc, start, dec, int(max_query_len))
        return out
    out = torch.zeros(T, H, dv, dtype=torch.float32)
    qf, kf, vf = (q.float() * q_scale).reshape(T, H, dk), k.float().reshape(T, H, dk), v.float().reshape(T, H, dv)
    a = torch.exp(loga).reshape(T, H, dk)
    ql, sl, rows = qsl.tolist(), seq_lens.tolist(), state_rows.tolist()
    for s in range(len(sl)):
        b, e = ql[s], ql[s + 1]
        if e <= b:
            continue
        S = state[rows[s], off:off + H * dv * dk].view(H, dv, dk)
        if sl[s] - (e - b) == 0:
            S.zero_()
        for t in range(b, e):
            S.mul_(a[t].unsqueeze(1)).add_(vf[t].unsqueeze(2) * kf[t].unsqueeze(1))
            out[t] = (S * qf[t].unsqueeze(1)).sum(-1)
    return out.reshape(T, H * dv)


def rotary_table(positions: torch.Tensor, freqs: torch.Tensor, mag: float = 1.0) -> torch.Tensor:
    """cos and sin of position * freqs[i], times mag: fp32 [T, len(freqs), 2].  One table serves every layer of a step
    that turns by the same frequencies."""
    T, n = positions.shape[0], freqs.numel()
    if _gpu(positions):
        out = torch.empty(T, n, 2, dtype=torch.float32, device=positions.device)
        ext().rotary_table(out, positions, freqs, float(mag))
        return out
    ang = positions.to(torch.float32).view(-1, 1) * freqs.float().view(1, n)
    return torch.stack([torch.cos(ang) * mag, torch.sin(ang) * mag], dim=-1)


def _turn_by(x: torch.Tensor, table: torch.Tensor) -> torch.Tensor:
    """x fp32 [T, heads, dim]: coordinate i pairs with i + n for the table's n pairs; the rest passes."""
    n = table.shape[1]
    c, s = table[:, :, 0].unsqueeze(1), table[:, :, 1].unsqueeze(1)
    u, v = x[..., :n], x[..., n:2 * n]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * n:]], dim=-1)


RETENTION_CHUNK = 64  # tokens of a tile of the chunked form
RETENTION_MAX_V = 256  # value size up to which the norm and the gate are taken where the head's outputs meet


def retention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, gate: torch.Tensor, table: torch.Tensor,
              decay: torch.Tensor, state: torch.Tensor, state_rows: torch.Tensor, off: int, qsl: torch.Tensor,
              seq_lens: torch.Tensor, num_heads: int, dk: int, dv: int, k_scale: float, eps: float,
              max_query_len: int = 0) -> torch.Tensor:
    """Retention: q, k turned by `table` (rotary_table; half-split pairs on the head's first coordinates), k times k_scale;
        S <- decay_h S + k_t v_t^T,   o_t = S^T q_t,   y = o / sqrt(mean(o^2) + eps) over the head, times SiLU(gate).
    q, k [T, H*dk], v, gate [T, H*dv] (row-strided views), decay fp32 [H].  Returns y [T, H*dv] in q's dtype; S (fp32,
    stored [H, dv, dk]) stays in the sequence's slot.  Everything between the projections and y is fp32.  Single-token
    steps (max_query_len 1, a host int) update the state in place; chunks run in tiles of RETENTION_CHUNK tokens: every
    tile's own contribution to the state, the states at the tiles' starts chained from those, then all outputs, as
    fp32 matrix products."""
    T, H = q.shape[0], num_heads
    if _gpu(q):
        S = seq_lens.numel()
        fused = dv <= RETENTION_MAX_V
        out = torch.empty(T, H * dv, dtype=q.dtype if fused else torch.float32, device=q.device)
        mq = max(1, min(int(max_query_len) or T, T))
        ntiles = -(-mq // RETENTION_CHUNK)
        pool = torch.empty(S * ntiles * H * dv * dk, dtype=torch.float32, device=q.device) if ntiles > 1 else None
        ext().retention(out, q, k, v, gate, table, decay, state, state_rows, int(off), qsl, seq_lens, H, dk, dv, float(k_scale),
                        float(eps), mq, pool)
        if fused:
            return out
        return gated_norm(out, gate, torch.ones(1, dtype=q.dtype, device=q.device), eps, H, "silu", False, q.dtype)
    qf, kf = _turn_by(q.float().reshape(T, H, dk), table), _turn_by(k.float().reshape(T, H, dk), table) * k_scale
    vf = v.float().reshape(T, H, dv)
    out = torch.zeros(T, H, dv, dtype=torch.float32)
    ql, sl, rows = qsl.tolist(), seq_lens.tolist(), state_rows.tolist()
    for s in range(len(sl)):
        b, e = ql[s], ql[s + 1]
        if e <= b:
            continue
        St = state[rows[s], off:off + H * dv * dk].view(H, dv, dk)
        if sl[s] - (e - b) <= 0:
            St.zero_()
        for t in range(b, e):
            St.mul_(decay.view(H, 1, 1)).add_(vf[t].unsqueeze(2) * kf[t].unsqueeze(1))
            out[t] = (St * qf[t].unsqueeze(1)).sum(-1)
    return (_rms(out, eps).reshape(T, H * dv) * F.silu(gate.float())).to(q.dtype)


SELECTIVE_MAX_STATE = 512


def selective_scan(u: torch.Tensor, dt: torch.Tensor, B: torch.Tensor, C: torch.Tensor, z: torch.Tensor, A: torch.Tensor,
                   dt_bias: torch.Tensor, D: torch.Tensor, state: torch.Tensor, state_rows: torch.Tensor, off: int,
                   qsl: torch.Tensor, seq_lens: torch.Tensor, max_query_len: int = 0) -> torch.Tensor:
    """Selective scan with a decay per channel and state: with d = softplus(dt + dt_bias) per channel,
        S[n, c] <- exp(d_c A[n, c]) S[n, c] + d_c u_c B_n,   y_c = (sum_n S[n, c] C_n + D_c u_c) * SiLU(z_c).
    u, dt, z [T, I], B, C [T, N] (row-strided views); A fp32 [N, I] (negative), dt_bias, D fp32 [I].  Returns y [T, I] in
    u's dtype; S (fp32, stored [N, I]) stays in the sequence's slot.  max_query_len: the step's longest chunk (host
    int); the step is a diagonal map of the state, so long chunks are cut into pieces that run side by side (end
    states from an empty start, chained by the pieces' summed d, then the outputs)."""
    T, I = u.shape
    N = B.shape[1]
    if _gpu(u):
        out = torch.empty(T, I, dtype=u.dtype, device=u.device)
        S = seq_lens.numel()
        lanes = ext().selective_lanes(N)
        piece, npieces, loc, start = _scan_split(S, T, max_query_len, N * I, 1, -(-I * lanes // 4), u.device)
        dsum = torch.empty(S * npieces * I, dtype=torch.float32, device=u.device) if npieces > 1 else None
        ext().selective_scan(out, u, dt, B, C, z, A, dt_bias, D, state, state_rows, int(off), qsl, seq_lens, piece, npieces, loc, start,
                             dsum)
        return out
    d = F.softplus(dt.float() + dt_bias, threshold=1e9)
    uf, Bf, Cf = u.float(), B.float(), C.float()
    out = torch.zeros(T, I, dtype=torch.float32)
    ql, sl, rows = qsl.tolist(), seq_lens.tolist(), state_rows.tolist()
    for s in range(len(sl)):
        b, e = ql[s], ql[s + 1]
        if e <= b:
            continue
        St = state[rows[s], off:off + N * I].view(N, I)
        if sl[s] - (e - b) <= 0:
            St.zero_()
        for t in range(b, e):
            St.mul_(torch.exp(d[t] * A)).add_((d[t] * uf[t]) * Bf[t].unsqueeze(1))
            out[t] = (St * Cf[t].unsqueeze(1)).sum(0) + D * uf[t]
    return (out * F.silu(z.float())).to(u.dtype)


def ssd_scan(x: torch.Tensor, B: torch.Tensor, C: torch.Tensor, dt: torch.Tensor, dt_bias: torch.Tensor,
             A_log: torch.Tensor, D: torch.Tensor, state: torch.Tensor, state_rows: torch.Tensor, off: int,
             qsl: torch.Tensor, seq_lens: torch.Tensor, num_heads: int, groups: int, N: int, P: int,
             max_query_len: int = 0) -> torch.Tensor:
    """Selective state-space recurrence with a scalar decay per head and token (state-space duality):
        d = softplus(dt + dt_bias_h);  S = exp(-exp(A_log_h) d) S + d B_g x_h^T;  y_h = S^T C_g + D_h x_h
    with S [N, P] per head and head h reading group h // (H / G).  x [T, H*P], B, C [T, G*N], dt [T, H]
    (row-strided views of any float dtype); dt_bias, A_log, D fp32 [H].  Returns y fp32 [T, H*P]; the
    state (fp32, stored [H, P, N]) stays in the sequence's slot.  max_query_len: the step's longest
    chunk (host int); the step is a diagonal map of the state, so long chunks are cut into pieces
    that run side by side (a piece's end state from an empty state, the true state at every piece's
    start chained from those and the pieces' decays, then the outputs)."""
    T = x.shape[0]
    H = num_heads
    if _gpu(x):
        out = torch.empty(T, H * P, dtype=torch.float32, device=x.device)
        piece, npieces, loc, start = _scan_split(seq_lens.numel(), T, max_query_len, H * N * P, H, 4 * P, x.device, spare=True)
        dec = torch.empty(seq_lens.numel() * npieces * H, dtype=torch.float32, device=x.device) if npieces > 1 else None
        ext().ssd_scan(out, x, B, C, dt, dt_bias, A_log, D, state, state_rows, int(off), qsl, seq_lens, H, groups, N, P,
                       piece, npieces, loc, start, dec, int(max_query_len))
        return out
    out = torch.zeros(T, H, P, dtype=torch.float32)
    xf = x.float().reshape(T, H, P)
    rep = H // groups
    Bf = B.float().reshape(T, groups, N).repeat_interleave(rep, dim=1)
    Cf = C.float().reshape(T, groups, N).repeat_interleave(rep, dim=1)
    d = F.softplus(dt.float() + dt_bias.float(), threshold=1e9)
    a = torch.exp(-torch.exp(A_log.float()) * d)
    ql, sl, rows = qsl.tolist(), seq_lens.tolist(), state_rows.tolist()
    for s in range(len(sl)):
        b, e = ql[s], ql[s + 1]
        if e <= b:
            continue
        S = state[rows[s], off:off + H * P * N].view(H, P, N)
        if sl[s] - (e - b) == 0:
            S.zero_()
        for t in range(b, e):
            S.mul_(a[t].view(H, 1, 1)).add_((d[t].view(H, 1) * xf[t]).unsqueeze(2) * Bf[t].unsqueeze(1))
            out[t] = (S * Cf[t].unsqueeze(1)).sum(-1) + D.float().view(H, 1) * xf[t]
    return out.reshape(T, H * P)


# A bf16 step of the delta rule runs in chunks when token by token it would be cut into pieces, and otherwise from
# DELTA_CHUNK_TOKENS tokens in its longest chunk on, or 32 fewer and so many for each sequence, since a single token costs its
# heads as much as 32: DELTA_CHUNK_TOKENS_PER_SEQ, or more beside shorter ones where the heads fill the chip (one for each 70,000
# entries of a sequence's state).  Token by token / in chunks, us, 16 heads of 128: a chunk of 70 39 / 45, 96 49 / 45, 256
# 177 / 55, 4,096 1,360 / 425; 16 chunks of 100 189 / 172; beside 32 single tokens 128 109 / 129, 257 174 / 142, 400 241 / 149,
# beside 64 300 242 / 219.  64 heads of 128: beside 32 300 361 / 472, 400 426 / 491, 600 567 / 560.  64 heads of 64: beside 64
# 300 211 / 239, 512 294 / 276; 16 chunks of 160 294 / 310, as with 16 heads of 128 x 64 148 / 164: such many small heads want
# some tokens more.
DELTA_CHUNK_TOKENS, DELTA_CHUNK_TOKENS_PER_SEQ = 96, 5.5
DELTA_MIN_PIECES = 4  # a split delta-rule scan does three times the work: fewer pieces do not pay


def delta_in_chunks(S: int, T: int, max_query_len: int, heads: int, dk: int, dv: int) -> bool:
    if _scan_pieces(S, T, max_query_len, heads * (dv + dk) * dk, heads, 4 * (dv + dk))[1] >= DELTA_MIN_PIECES:
        return True
    each, state = DELTA_CHUNK_TOKENS_PER_SEQ, heads * dk * dv
    if 2 * T < S * max_query_len:  # mostly shorter ones
        each = max(each, state / 70000)
    some = 16 if dk * dv < 128 * 128 <= state / 8 and S > 4 else 0
    return min(max_query_len, T) >= DELTA_CHUNK_TOKENS + max(0, each * S + some - 32)


def delta_scan(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, beta: torch.Tensor, a: torch.Tensor,
               dt_bias: torch.Tensor, A_log: torch.Tensor, state: torch.Tensor, state_rows: torch.Tensor, off: int,
               qsl: torch.Tensor, seq_lens: torch.Tensor, num_heads: int, qk_heads: int, dk: int, dv: int,
               q_scale: float, unit_eps: float = 1e-6, max_query_len: int = 0) -> torch.Tensor:
    """Gated delta rule with one decay per head and key channel.  q, k [T, G*dk] are made unit vectors
    per head (x / sqrt(sum x^2 + unit_eps)), q also times q_scale; head h reads q/k head h // (H / G).
        g = exp(-exp(A_log_h) softplus(a + dt_bias))   [H, dk]      b = sigmoid(beta)   [H]
        S = diag(g) S;   u = b (v - S^T k);   S = S + k u^T;   o = S^T q
    so the read-out sees the token's own write.  v [T, H*dv], beta [T, H], a [T, H*dk] (row-strided
    views); dt_bias fp32 [H*dk], A_log fp32 [H].  Returns o fp32 [T, H*dv]; S (fp32, stored [H, dv, dk])
    stays in the sequence's slot.
    max_query_len: the step's longest chunk (host int).  A token maps the state as S -> A_t S + b_t with
    A_t = (I - b k k^T) diag(g), so a piece of tokens maps it as S -> P S + L: long chunks are cut into
    pieces that run side by side, pass 1 giving every piece's L (end state from an empty start) and P
    (dk more state columns started as the identity and fed no values), the states at the pieces'
    starts following by one fp32 matrix product per piece, pass 2 writing the outputs.  Three times
    the multiply-adds, but DELTA_MIN_PIECES or more pieces at once instead of one serial walk.
    bf16 steps with a long chunk run in chunks of 32 tokens on the matrix cores instead (csrc/mixers/delta_chunk.hip)."""
    T = q.shape[0]
    H, G = num_heads, qk_heads
    if _gpu(q):
        out = torch.empty(T, H * dv, dtype=torch.float32, device=q.device)
        S = seq_lens.numel()
        args = (out, q, k, v, beta, a, dt_bias, A_log, state, state_rows, int(off), qsl, seq_lens, H, G, dk, dv,
                float(q_scale), float(unit_eps))
        if q.dtype == torch.bfloat16 and delta_in_chunks(S, T, max_query_len, H, dk, dv):
            floats = ext().delta_chunk_floats(dk, dv) * (T // 32 + S) * H
            if 0 < 4 * floats <= SCAN_SCRATCH_BYTES and state.data_ptr() % 16 == 0 and state.stride(0) % 4 == 0 and off % 4 == 0:
                work = torch.empty(floats, dtype=torch.float32, device=q.device)
                ext().delta_scan(*args, 0, 1, 1, None, None, int(max_query_len), work)
                return out
        piece, npieces, _, _ = _scan_split(S, T, max_query_len, H * (dv + dk) * dk, H, 4 * (dv + dk), q.device)
        if npieces < DELTA_MIN_PIECES:
            ext().delta_scan(*args, 0, 1, 1, None, None, int(max_query_len), None)
            return out
        n = H * dv * dk
        loc = torch.empty(S, npieces, H, dv + dk, dk, dtype=torch.float32, device=q.device)
        start = torch.empty(S, npieces, H * dv, dk, dtype=torch.float32, device=q.device)
        ext().delta_scan(*args, 1, piece, npieces, loc, start, int(max_query_len), None)
        first = (seq_lens - (qsl[1:] - qsl[:-1]) <= 0).view(S, 1, 1)
        slot = state.index_select(0, state_rows.long())[:, off:off + n].view(S, H * dv, dk)
        start[:, 0] = torch.where(first, torch.zeros((), dtype=torch.float32, device=q.device), slot)
        for p in range(npieces - 1):  # St' = St Pt + Lt in the transposed storage, batched over sequences and heads
            start[:, p + 1] = torch.baddbmm(loc[:, p, :, :dv].reshape(S * H, dv, dk), start[:, p].reshape(S * H, dv, dk),
                                            loc[:, p, :, dv:].reshape(S * H, dk, dk)).view(S, H * dv, dk)
        ext().delta_scan(*args, 2, piece, npieces, loc, start, int(max_query_len), None)
        return out
    out = torch.zeros(T, H, dv, dtype=torch.float32)
    rep = H // G

    def unit(t):
        t = t.float().reshape(T, G, dk)
        return (t * torch.rsqrt(t.pow(2).sum(-1, keepdim=True) + unit_eps)).repeat_interleave(rep, dim=1)

    qf, kf = unit(q) * q_scale, unit(k)
    vf = v.float().reshape(T, H, dv)
    b = torch.sigmoid(beta.float())
    g = torch.exp(-torch.exp(A_log.float()).view(1, H, 1) *
                  F.softplus(a.float() + dt_bias.float(), threshold=1e9).reshape(T, H, dk))
    ql, sl, rows = qsl.tolist(), seq_lens.tolist(), state_rows.tolist()
    for s in range(len(sl)):
        c, e = ql[s], ql[s + 1]
        if e <= c:
            continue
        S = state[rows[s], off:off + H * dv * dk].view(H, dv, dk)
        if sl[s] - (e - c) == 0:
            S.zero_()
        for t in range(c, e):
            S.mul_(g[t].unsqueeze(1))
            u = b[t].view(H, 1) * (vf[t] - (S * kf[t].unsqueeze(1)).sum(-1))
            S.add_(u.unsqueeze(2) * kf[t].unsqueeze(1))
            out[t] = (S * qf[t].unsqueeze(1)).sum(-1)
    return out.reshape(T, H * dv)


def gated_norm(o: torch.Tensor, gate: torch.Tensor, w: torch.Tensor, eps: float, groups: int, act: str,
               gate_first: bool, out_dtype: torch.dtype, out_scale: float = 1.0,
               out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """A mixer's output norm with its gate.  o fp32 [T, N]; the RMS norm runs over each of `groups`
    equal slices of a row; w has N entries or a divisor of N (then it repeats, e.g. one weight per
    head size shared by the heads); act(gate) with act in silu | sigmoid multiplies before the norm
    (gate_first) or after it.  The result, times out_scale, goes to `out` (may be a row-strided view
    of a wider buffer) or a new [T, N] tensor of out_dtype."""
    T, N = o.shape
    if out is None:
        out = torch.empty(T, N, dtype=out_dtype, device=o.device)
    if _gpu(o):
        ext().gated_norm(out, o, gate, w, float(eps), int(groups), act == "silu", bool(gate_first), float(out_scale))
        return out
    gf = F.silu(gate.float()) if act == "silu" else torch.sigmoid(gate.float())
    wf = w.float().repeat(N // w.numel())
    y = o * gf if gate_first else o
    y = _rms(y.view(T, groups, N // groups), eps).reshape(T, N) * wf
    if not gate_first:
        y = y * gf
    out.copy_((y * out_scale).to(out.dtype))
    return out


# ----------------------------------------------------------------------------- latent attention
def _rotate_half(x: torch.Tensor, pos: torch.Tensor, freqs: torch.Tensor, mag: float = 1.0) -> torch.Tensor:
    """x fp32 [T, heads, 2n]: coordinate i pairs with i + n and the pair turns by pos * freqs[i]."""
    n = freqs.numel()
    ang = pos.to(torch.float32).view(-1, 1, 1) * freqs.float().view(1, 1, n)
    c, s = torch.cos(ang) * mag, torch.sin(ang) * mag
    u, v = x[..., :n], x[..., n:]
    return torch.cat([u * c - v * s, v * c + u * s], dim=-1)


def latent_prep(dq: torch.Tensor, dkv: torch.Tensor, positions: torch.Tensor, slot_mapping: torch.Tensor,
                cache: torch.Tensor, koff: int, rank: int, block_size: int, freqs: torch.Tensor,
                q_norm: torch.Tensor, kv_norm: torch.Tensor, eps: float, split_pairs: bool = True,
                mag: float = 1.0) -> torch.Tensor:
    """The two down-projections of a latent attention, from the fused projection to what the next
    steps read, in one launch.  dq [T, q_rank] (row-strided view): returns RMSNorm(dq) * q_norm as a
    new [T, q_rank].  dkv [T, rank + 2n]: the first `rank` columns RMS-normed times kv_norm, the last
    2n (n = len(freqs)) turned in the half-split layout (i pairs with i + n; split_pairs False: 2i with
    2i + 1) by position * freqs[i], cos and sin times mag; the row [latent | turned part] goes into the paged cache at
    `koff` as [BS, rank + 2n] (one shared kv head; slot -1: not written).  Norms, angles and turns in fp32, one rounding at the end."""
    T, qr = dq.shape
    n = freqs.numel()
    dk = rank + 2 * n
    if _gpu(dq):
        cq = torch.empty(T, qr, dtype=dq.dtype, device=dq.device)
        ext().latent_prep(cq, dq, dkv, positions, slot_mapping, cache, int(koff), int(rank), int(block_size), freqs,
                          q_norm, kv_norm, float(eps), bool(split_pairs), float(mag))
        return cq
    cq = (_rms(dq.float(), eps) * q_norm.float()).to(dq.dtype)
    d = dkv.float()
    c = _rms(d[:, :rank], eps) * kv_norm.float()
    part = d[:, rank:].unsqueeze(1)
    kr = (_rotate_half(part, positions, freqs, mag) if split_pairs else _rotate(part, positions, freqs, 1.0, mag)).squeeze(1)
    row = torch.cat([c, kr], dim=-1).to(cache.dtype)
    ok = slot_mapping >= 0
    slots = slot_mapping[ok]
    kc = cache[:, koff:koff + block_size * dk].view(-1, block_size, dk)
    kc[slots // block_size, slots % block_size] = row[ok]
    return cq


def rope_half_into(out: torch.Tensor, x: torch.Tensor, positions: torch.Tensor, heads: int, x_dim: int, x_col: int,
                   out_dim: int, out_col: int, freqs: torch.Tensor, split_pairs: bool = True, mag: float = 1.0) -> None:
    """Per token and head: the 2n columns of x's head (x [T, heads*x_dim], from column x_col of the head)
    turned in the half-split layout (split_pairs False: as neighbouring pairs) by position * freqs[i] (cos and sin
    times mag), written to columns out_col.. of the same head in out [T, heads*out_dim].  out may be x with the same
    columns (turned in place).  fp32 inside."""
    n = freqs.numel()
    if _gpu(x):
        ext().rope_half_into(out, x, positions, int(heads), int(x_dim), int(x_col), int(out_dim), int(out_col), freqs,
                             bool(split_pairs), float(mag))
        return
    T = x.shape[0]
    part = x.reshape(T, heads, x_dim)[:, :, x_col:x_col + 2 * n].float()
    turned = _rotate_half(part, positions, freqs, mag) if split_pairs else _rotate(part, positions, freqs, 1.0, mag)
    out.view(T, heads, out_dim)[:, :, out_col:out_col + 2 * n] = turned.to(out.dtype)


LATENT_TARGET_WAVES = 1024  # waves that fill the 256 CUs one deep: single-token steps split their keys up to this
# the widest rows (over 320 entries): "pair" = two waves per 16-row tile, each half of the row; "single" = one wave
# per tile with its queries in LDS; "auto" = pair
LATENT_WIDE_FORM = os.environ.get("MXS_LATENT_WIDE_FORM", "auto")


def latent_attention(q: torch.Tensor, cache: torch.Tensor, block_tables: torch.Tensor, qsl: torch.Tensor,
                     seq_lens: torch.Tensor, koff: int, num_heads: int, dk: int, rank: int, block_size: int, scale: float,
                     max_query_len: int = 0, max_seq_len: int = 0, sink: Optional[torch.Tensor] = None,
                     window: int = 0) -> torch.Tensor:
    """Softmax attention of every head over the same cached rows [latent | rotated part] (dk entries a
    row at `koff`, written by latent_prep), causal, within the last `window` positions when window > 0;
    the values are the rows' first `rank` entries.
    q [T, H*dk] (the folded queries) -> the weighted latents [T, H*rank]; scores and weights fp32; sink as
    in window_attention.  bf16 on the GPU with dk a multiple of 8 up to 576 and rank a multiple of 16 up
    to 512 runs the matrix-core kernel; a step of few rows splits each row's keys over several waves
    (max_seq_len bounds how many are worth it) and merges the stretches.  Everything else runs
    window_attention with one kv head and value rows dk apart."""
    T = q.shape[0]
    if _gpu(q) and q.dtype == torch.bfloat16 and T:
        S = seq_lens.numel()
        mq = max(1, min(int(max_query_len) or T, T))
        tiles = S * (-(-mq * num_heads // 16))
        span = min(int(max_seq_len) or 16, int(window) + 15) if window > 0 else (int(max_seq_len) or 16)
        blocks = max(1, -(-span // 16))
        nsplit = max(1, min(16, LATENT_TARGET_WAVES // max(tiles, 1), blocks // 2))
        out = torch.empty(T, num_heads * rank, dtype=q.dtype, device=q.device)
        part = (torch.empty(T * num_heads * nsplit * (rank + 4), dtype=torch.float32, device=q.device)
                if nsplit > 1 else None)
        if ext().latent_attention(out, q, cache, block_tables, qsl, seq_lens, int(koff), num_heads, dk, rank, block_size,
                                  float(scale), mq, sink, nsplit, part,
                                  LATENT_WIDE_FORM != "single", int(window)):
            return out
    return window_attention(q, cache, block_tables, qsl, seq_lens, koff, koff, num_heads, 1, dk, rank, block_size, scale,
                            int(window), 0, max_query_len, sink=sink, v_stride=dk)


def latent_plan(qsl: torch.Tensor, seq_lens: torch.Tensor, window: int = 0) -> tuple:
    """Where the cached rows that a step's chunks see lie when they are gathered back to back (latent_rows): (base int32 [S],
    the row of a sequence's key position 0, and offs int32 [S + 1], its first row).  With window > 0 a sequence's rows begin
    at the page of its first query's oldest visible key."""
    S = seq_lens.numel()
    base = torch.empty(S, dtype=torch.int32, device=seq_lens.device)
    offs = torch.empty(S + 1, dtype=torch.int32, device=seq_lens.device)
    if _gpu(seq_lens):
        ext().latent_plan(base, offs, qsl, seq_lens, int(window))
        return base, offs
    qlen = qsl[1:S + 1] - qsl[:S]
    past = (seq_lens - qlen).clamp(min=0)
    first = (past - window + 1).clamp(min=0) // 16 * 16 if window > 0 else torch.zeros_like(past)
    offs[0] = 0
    offs[1:] = torch.where(qlen > 0, past + qlen - first, torch.zeros_like(past)).cumsum(0)
    base.copy_(offs[:S] - first)
    return base, offs


def latent_rows(cache: torch.Tensor, block_tables: torch.Tensor, base: torch.Tensor, offs: torch.Tensor, n: int, koff: int,
                dk: int, block_size: int) -> torch.Tensor:
    """The cached rows [n, dk] of latent_plan's places; n = offs[S], known to the host."""
    out = torch.empty(n, dk, dtype=cache.dtype, device=cache.device)
    if _gpu(cache):
        ext().latent_rows(out, cache, block_tables, base, offs, int(koff), int(block_size))
        return out
    kc = cache[:, koff:koff + block_size * dk].view(-1, block_size, dk)
    for s in range(base.numel()):
        a, e = int(offs[s]), int(offs[s + 1])
        key = torch.arange(a, e) - int(base[s])
        out[a:e] = kc[block_tables[s].long()[key // block_size], key % block_size]
    return out


def expanded_attention(q: torch.Tensor, kv: torch.Tensor, rows: torch.Tensor, base: torch.Tensor, qsl: torch.Tensor,
                       seq_lens: torch.Tensor, num_heads: int, dn: int, dr: int, dv: int, scale: float, max_query_len: int,
                       sink: Optional[torch.Tensor] = None, window: int = 0, out: Optional[torch.Tensor] = None,
                       max_seq_len: int = 0) -> Optional[torch.Tensor]:
    """Causal softmax attention of chunks over keys and values that every head expanded from gathered latent rows.
    q [T, H*(dn + dr)], kv [n, H*dn + H*dv]: the heads' plain key parts, then their values; the last dr entries of `rows`
    [n, rank + dr] are the key part that all heads share.  Row of key position j of sequence s: base[s] + j.  sink, window
    as in latent_attention, max_seq_len as in window_attention.  -> [T, H*dv] (in `out` if given); None: head sizes that the
    kernel does not hold."""
    T, H, rank = q.shape[0], num_heads, rows.shape[1] - dr
    if out is None:
        out = torch.empty(T, H * dv, dtype=q.dtype, device=q.device)
    if _gpu(q):
        ok = q.dtype == torch.bfloat16 and ext().expanded_attention(out, q, kv, rows, base, qsl, seq_lens, H, dn, dr, dv, rank,
                                                                    float(scale), int(max_query_len), sink, int(window),
                                                                    int(max_seq_len))
        return out if ok else None
    ql, sl, bl = qsl.tolist(), seq_lens.tolist(), base.tolist()
    for s in range(len(sl)):
        a, e = ql[s], ql[s + 1]
        if e <= a:
            continue
        lo = max(0, -bl[s])
        r = torch.arange(lo, sl[s]) + bl[s]
        K = torch.cat([kv[r, :H * dn].view(-1, H, dn), rows[r, rank:].unsqueeze(1).expand(-1, H, -1)], -1).float()
        sc = torch.einsum("mhd,nhd->hmn", q[a:e].reshape(e - a, H, dn + dr).float(), K) * scale
        i, j = torch.arange(sl[s] - (e - a), sl[s]).unsqueeze(1), torch.arange(lo, sl[s]).unsqueeze(0)
        seen = (j <= i) & (i - j < window) if window > 0 else j <= i
        sc = sc.masked_fill(~seen.unsqueeze(0), float("-inf"))
        if sink is not None:
            sc = torch.cat([sc, sink.float().view(-1, 1, 1).expand(-1, sc.shape[1], 1)], dim=-1)
        p = torch.softmax(sc, dim=-1)[..., :r.numel()]
        out[a:e] = torch.einsum("hmn,nhd->mhd", p, kv[r, H * dn:].view(-1, H, dv).float()).reshape(e - a, -1).to(out.dtype)
    return out


# ----------------------------------------------------------------------------- routed experts
def route_topk(logits: torch.Tensor, k: int, renorm: bool = False, softmax: bool = False, *,
               correction: Optional[torch.Tensor] = None, groups: int = 1, keep: int = 1, scale: float = 1.0) -> tuple:
    """Router: scores = sigmoid(logits), or softmax over all experts (fp32 [T, E]); the k largest per
    token (ties: the lower index first), their scores as weights (renorm: divided by their sum).
    The keyword forms: correction (fp32 [E]) is added to the scores for the choice only; with groups > 1 the experts
    form that many equal runs of neighbours, a group's score is the sum of its two largest choice scores, and only
    experts of the `keep` best groups can be chosen; weights are multiplied by scale.
    -> (weights fp32 [T, k], ids int32 [T, k])."""
    T, E = logits.shape
    if E % groups or not 1 <= keep <= groups or k > keep * (E // groups):
        raise ValueError(f"route_topk: {k} of {E} experts in {keep} of {groups} groups")
    grouped = correction is not None or groups > 1 or scale != 1.0
    if _gpu(logits):
        w = torch.empty(T, k, dtype=torch.float32, device=logits.device)
        ids = torch.empty(T, k, dtype=torch.int32, device=logits.device)
        if grouped:
            ext().route_grouped(w, ids, logits, correction, int(groups), int(keep), float(scale), bool(renorm), bool(softmax))
        else:
            ext().route_topk(w, ids, logits, bool(renorm), bool(softmax))
        return w, ids
    s = torch.softmax(logits.float(), dim=-1) if softmax else torch.sigmoid(logits.float())
    c = s if correction is None else s + correction.float()
    if groups > 1:
        per = c.view(T, groups, E // groups)
        gs = per.topk(min(2, E // groups), dim=-1)[0].sum(-1)
        best = torch.argsort(gs, dim=-1, descending=True, stable=True)[:, :keep]
        seen = torch.zeros(T, groups, dtype=torch.bool).scatter_(1, best, True)
        c = per.masked_fill(~seen.unsqueeze(-1), float("-inf")).reshape(T, E)
    order = torch.argsort(c, dim=-1, descending=True, stable=True)[:, :k]
    w = torch.gather(s, 1, order)
    if renorm:
        w = w / (w.sum(-1, keepdim=True) + 1e-20)
    return w * scale if scale != 1.0 else w, order.to(torch.int32)


def route_linear(h: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], experts: int, k: int) -> tuple:
    """Router projection and choice in one launch: z = h w^T + bias (fp32 products and sums; w [experts + gates, W], bias
    its rows' or None).  The k largest of the first `experts` logits are chosen (ties: the lower index first), their
    weights are the softmax over the chosen logits alone; the rows behind them are gates, sigmoid(z).
    -> (weights fp32 [T, k], ids int32 [T, k], gates fp32 [T, rows - experts])."""
    T, n = h.shape[0], w.shape[0]
    if not 1 <= k <= experts <= n:
        raise ValueError(f"route_linear: {k} of {experts} experts in {n} rows")
    if _gpu(h):
        wt = torch.empty(T, k, dtype=torch.float32, device=h.device)
        ids = torch.empty(T, k, dtype=torch.int32, device=h.device)
        gates = torch.empty(T, n - experts, dtype=torch.float32, device=h.device)
        ext().route_linear(wt, ids, gates, h, w, bias, int(experts))
        return wt, ids, gates
    z = F.linear(h.float(), w.float(), None if bias is None else bias.float())
    order = torch.argsort(z[:, :experts], dim=-1, descending=True, stable=True)[:, :k]
    return torch.softmax(torch.gather(z, 1, order), dim=-1), order.to(torch.int32), torch.sigmoid(z[:, experts:])


def capped_glu(gu: torch.Tensor, limit: float, alpha: float = 1.702) -> torch.Tensor:
    """A fused [gate | up] projection [R, 2F] -> [R, F]:  g = min(gate, limit), u = clamp(up, -limit, limit),
    g * sigmoid(alpha * g) * (u + 1); fp32 inside."""
    Fh = gu.shape[1] // 2
    if _gpu(gu):
        out = torch.empty(gu.shape[0], Fh, dtype=gu.dtype, device=gu.device)
        ext().capped_glu(out, gu, float(limit), float(alpha))
        return out
    g = gu[:, :Fh].float().clamp(max=limit)
    u = gu[:, Fh:].float().clamp(-limit, limit)
    return (g * torch.sigmoid(alpha * g) * (u + 1.0)).to(gu.dtype)


def expert_align(ids: torch.Tensor, num_experts: int) -> tuple:
    """Counting sort of the (token, slot) pairs by expert.  ids int32 [T, k] -> (offs int32 [E + 1]:
    expert e owns the sorted rows offs[e]:offs[e+1]; inv int32 [T*k]: the sorted row of pair p = t*k + j;
    the order of one expert's rows is free)."""
    T, k = ids.shape
    if _gpu(ids):
        offs = torch.empty(num_experts + 1, dtype=torch.int32, device=ids.device)
        inv = torch.empty(T * k, dtype=torch.int32, device=ids.device)
        ext().expert_align(offs, inv, ids, int(num_experts))
        return offs, inv
    flat = ids.reshape(-1).long()
    order = torch.argsort(flat, stable=True)
    inv = torch.empty_like(order)
    inv[order] = torch.arange(order.numel())
    counts = torch.bincount(flat, minlength=num_experts)
    offs = torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)])
    return offs.to(torch.int32), inv.to(torch.int32)


def gather_scaled(h: torch.Tensor, weights: Optional[torch.Tensor], inv: torch.Tensor, k: int = 0) -> torch.Tensor:
    """xs[inv[p]] = weights[p] * h[p // k] for every pair p (weights fp32 [T, k]): the experts' inputs,
    sorted by expert, each already times its routing weight (product in fp32, rounded once).
    weights None (then k says how many pairs a token has): the rows themselves."""
    T = h.shape[0]
    k = int(k) if weights is None else weights.shape[1]
    xs = torch.empty(T * k, h.shape[1], dtype=h.dtype, device=h.device)
    if _gpu(h):
        ext().gather_scaled(xs, h, weights, inv, k)
        return xs
    if weights is None:
        rows = h.unsqueeze(1).expand(T, k, h.shape[1]).reshape(T * k, -1)
    else:
        rows = (h.float().unsqueeze(1) * weights.float().unsqueeze(2)).reshape(T * k, -1).to(h.dtype)
    xs[inv.long()] = rows
    return xs


def gather_slabs(h: torch.Tensor, weights: Optional[torch.Tensor], ids: torch.Tensor, offs: torch.Tensor, inv: torch.Tensor,
                 cap: int) -> tuple:
    """(xs [E, cap, W], index int32 [T*k]): gather_scaled's rows with expert e's from row e * cap on, for a batched product
    over all experts; index[p] is pair p's row of the [E * cap, W] stack.  offs, inv from expert_align over ids; cap is at
    least every expert's count.  Rows behind an expert's last one are not written."""
    (T, k), E = ids.shape, offs.numel() - 1
    if _gpu(h):
        xs = torch.empty(E, int(cap), h.shape[1], dtype=h.dtype, device=h.device)
        index = torch.empty(T * k, dtype=torch.int32, device=h.device)
        ext().gather_slabs(xs, index, h, weights, ids, offs, inv)
        return xs, index
    rows = gather_scaled(h, weights, inv, k)
    flat = ids.reshape(-1).long()
    index = flat * int(cap) + inv.long() - offs.long()[flat]
    xs = torch.zeros(E * int(cap), h.shape[1], dtype=h.dtype)
    xs[index] = rows[inv.long()]
    return xs.view(E, int(cap), -1), index.to(torch.int32)


def spread_scaled(h: torch.Tensor, weights: Optional[torch.Tensor], ids: torch.Tensor, num_experts: int) -> torch.Tensor:
    """[E, T, W]: row (e, t) = weights[t, j] * h[t] where ids[t, j] = e, zeros for the experts a token
    did not choose (the experts' inputs for a batched product over all experts, no sorting).
    weights None: the chosen rows are h[t] itself."""
    T, k = ids.shape
    if _gpu(h):
        xs = torch.empty(num_experts, T, h.shape[1], dtype=h.dtype, device=h.device)
        ext().spread_scaled(xs, h, weights, ids)
        return xs
    cw = torch.zeros(T, num_experts, dtype=torch.float32)
    cw.scatter_(1, ids.long(), torch.ones(T, k) if weights is None else weights.float())
    return (cw.t().unsqueeze(2) * h.float().unsqueeze(0)).to(h.dtype)


def expert_combine(ys: torch.Tensor, index: Optional[torch.Tensor], k: int, T: int, extra: Optional[torch.Tensor] = None,
                   row_stride: int = 0, weights: Optional[torch.Tensor] = None, by_expert: bool = False) -> torch.Tensor:
    """out[t] = sum_j ys[index[t*k + j]] (+ extra[t]); index None: row j*row_stride + t (the k slabs
    of a [k, T, W] stack); by_expert: index holds experts and the row is index[t*k + j]*row_stride + t (a
    token's chosen slabs of an [E, T, W] stack).  weights (fp32 [T, k]): row j of token t enters times
    weights[t, j] (routing weights on the experts' outputs).  Summed in fp32, rounded once."""
    W = ys.shape[-1]
    if _gpu(ys):
        out = torch.empty(T, W, dtype=ys.dtype, device=ys.device)
        ext().expert_combine(out, ys.reshape(-1, W), index, int(k), extra, int(row_stride), weights, bool(by_expert))
        return out
    return ExpertRows(ys, index, k, T, extra, row_stride, weights, by_expert).sum32().to(ys.dtype)
