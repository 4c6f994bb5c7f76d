"""Feed-forward sublayers that a layer-list design can be built from, each with its sizes and
constants as parameters.  Like the mixers (mxserve/models/mixers.py) they name their checkpoint
tensors, re-pack them once when the weights are loaded, and compute from a step's flattened batch.

  GatedFF        W_down(act(W_gate h) * W_up h), gate and up as one projection; act = silu, or a gelu in its
                 exact or its tanh form
  CurvedFF       W_down(act(W_up h)) without a gate; act is a parabola above zero and an exponential
                 below it, with two learned numbers (`<p>act`)
  CappedExpert   one small gated unit with clipped pre-activations: g = min(W_gate x, limit),
                 u = clamp(W_up x, -limit, limit), W_down(g * sigmoid(alpha g) * (u + 1))
  RoutedExperts  a router (fp32; sigmoid scores, a softmax over all experts, or the logits themselves with a
                 softmax over the chosen ones) picks `top` of `experts`
                 small units per token (CappedExperts, or plain gated units when no limit is given, or
                 ungated W_down(act(W_up h))); the choice may add a learned correction to the scores and
                 be limited to the best groups of experts; the chosen scores (optionally renormalised and
                 scaled) weigh each expert's INPUT or its OUTPUT; an optional shared expert (a CappedExpert or a
                 GatedFF with its own size) sees every token, unweighted or times a sigmoid gate per token

The kernels are in mxserve/ops/seqmix.py (csrc/mixers/latent_experts.hip on the GPU); the matrix products go
through ops.linear and torch.bmm (hipBLASLt).
"""
from __future__ import annotations

from typing import Optional

import torch

from .. import ops
from ..ops import seqmix


class FeedForward:
    def shapes(self) -> dict:
        """Checkpoint tensor names -> shapes."""
        raise NotImplementedError

    def finish_weights(self, w: dict) -> None:
        pass

    def forward(self, h: torch.Tensor, w: dict) -> torch.Tensor:
        raise NotImplementedError


class GatedFF(FeedForward):
    def __init__(self, prefix: str, width: int, ff: int, act: str = "silu"):
        if act not in seqmix.ACTS:
            raise ValueError(f"{prefix}: unknown activation {act!r}")
        self.p, self.width, self.ff, self.act = prefix, width, int(ff), act

    def shapes(self) -> dict:
        p = self.p
        return {p + "gate": (self.ff, self.width), p + "up": (self.ff, self.width), p + "down": (self.width, self.ff)}

    def finish_weights(self, w: dict) -> None:
        p = self.p
        w[p + "_gu"] = torch.cat([w.pop(p + "gate"), w.pop(p + "up")]).contiguous()

    def forward(self, h: torch.Tensor, w: dict) -> torch.Tensor:
        p = self.p
        gu = ops.linear(h, w[p + "_gu"])
        a = seqmix.silu_mul(gu) if self.act == "silu" else seqmix.act_mul(gu, self.act)
        return ops.linear(a, w[p + "down"])


class CurvedFF(FeedForward):
    """act(z) = softplus(p) z^2 + z / 2 for z > 0, (1/2 + softplus(q)) (e^z - 1 - z) + z / 2 otherwise, with
    (p, q) = `<p>act`; the two softplus values are formed once, in fp32, when the weights are loaded."""

    def __init__(self, prefix: str, width: int, ff: int):
        self.p, self.width, self.ff = prefix, width, int(ff)

    def shapes(self) -> dict:
        p = self.p
        return {p + "up": (self.ff, self.width), p + "down": (self.width, self.ff), p + "act": (2,)}

    def finish_weights(self, w: dict) -> None:
        sp = torch.nn.functional.softplus(w.pop(self.p + "act").to(torch.float32), threshold=1e9)
        w[self.p + "_act"] = torch.stack([sp[0], 0.5 + sp[1]]).contiguous()

    def forward(self, h: torch.Tensor, w: dict) -> torch.Tensor:
        p = self.p
        return ops.linear(seqmix.xielu(ops.linear(h, w[p + "up"]), w[p + "_act"]), w[p + "down"])


class CappedExpert(FeedForward):
    def __init__(self, prefix: str, width: int, ff: int, limit: float, alpha: float = 1.702):
        self.p, self.width, self.ff = prefix, width, int(ff)
        self.limit, self.alpha = float(limit), float(alpha)

    def shapes(self) -> dict:
        p = self.p
        return {p + "gate": (self.ff, self.width), p + "up": (self.ff, self.width), p + "down": (self.width, self.ff)}

    def finish_weights(self, w: dict) -> None:
        p = self.p
        w[p + "_gu"] = torch.cat([w.pop(p + "gate"), w.pop(p + "up")]).contiguous()

    def forward(self, h: torch.Tensor, w: dict) -> torch.Tensor:
        p = self.p
        return ops.linear(seqmix.capped_glu(ops.linear(h, w[p + "_gu"]), self.limit, self.alpha), w[p + "down"])


class RoutedExperts(FeedForward):
    """Tensors: `<p>router` [E, width], `<p>e<i>.{gate,up,down}` (ungated: no gate), optionally `<p>router.b` [E],
    `<p>correction` [E], `<p>shared.{gate,up,down}` and `<p>shared.sg` [1, width].  Loaded as `<p>_in` [E, width, 2 ff] (ungated: [E, width, ff]) and `<p>_down`
    [E, ff, width], the right-hand operands of the batched products as they are (never a transposed view).

    Two ways through the experts, both exact (a token never meets an expert it did not choose with
    anything but a zero row, and a zero row gives a zero output):
      batched   every expert over all T rows of `spread_scaled` in two batched products -- no sorting
                and no host round trip, so a captured single-token step can replay it; E / top times
                the needed products, which steps of a few tokens do not feel (they stream the
                experts' weights either way)
      sorted    rows sorted by expert (expert_align; one host read of the E + 1 offsets) into slabs as long as the
                fullest expert, again two batched products; or, where the slabs would be mostly empty, one product pair per
                expert that got rows.  expert_combine gathers each token's rows
    """

    BATCHED_MAX_TOKENS = 32    # always batched up to this many tokens ...
    BATCHED_MAX_ROWS = 1024    # ... and beyond while experts x tokens stays within this many rows
    # Sorted rows: an expert's own two products take no less than about 40 us, however few its rows (and half as long again as
    # its share of a batched product when it has a thousand: they fill a third of the chip).  8 experts of 2,048 x 2,560,
    # even choices, products alone: 64 tokens 333 us one by one, 49 us in slabs; 512 tokens 332 / 80; 2,048: 353 / 141;
    # 4,096: 435 / 273.  So slabs, until their empty rows (at a large product's rate, and read and written by two products and the
    # activation at the memory's) and the weights of experts without rows cost more than 30 us for each expert that has some: 128
    # experts of 128 x 64, 4,096 tokens with one of them 102 us one by one, 240 in slabs; 8 of 256 x 512, 8,192 tokens with two
    # of them 155 / 193.  And never more than SLAB_MAX_BYTES of slabs, however the rows fall.
    SLAB_GAIN_S, SLAB_FLOPS, SLAB_BYTES = 30e-6, 1e15, 5e12
    SLAB_MAX_BYTES = 2 << 30

    def __init__(self, prefix: str, width: int, experts: int, top: int, ff: int, limit: Optional[float],
                 shared: Optional[FeedForward] = None, alpha: float = 1.702, renorm: bool = False,
                 score: str = "sigmoid", weigh: str = "input", gated: bool = True, act: str = "silu",
                 correction: bool = False, groups: int = 1, keep: int = 1, scale: float = 1.0, router_bias: bool = False,
                 shared_gate: bool = False):
        """limit None: an expert is W_down(act(W_gate x) * W_up x), or W_down act(W_up x) when not `gated`.  score:
        sigmoid | softmax (over all experts, before the choice) | softmax_top (the logits choose, the weights are the
        softmax over the chosen ones; with it come router_bias, a bias on the logits, and shared_gate, a row that gives
        the shared expert its sigmoid gate per token).  weigh: input | output (what a chosen score
        multiplies).  correction: a tensor added to the scores for the choice only.  groups, keep: the choice is
        limited to the `keep` best of so many groups of neighbours.  renorm, scale: the weights are the chosen
        scores, divided by their sum, times scale."""
        if not 1 <= top <= experts:
            raise ValueError(f"{prefix}: top {top} of {experts} experts")
        if score not in ("sigmoid", "softmax", "softmax_top") or weigh not in ("input", "output") or act not in seqmix.ACTS:
            raise ValueError(f"{prefix}: score {score!r}, weigh {weigh!r}, act {act!r}")
        if groups < 1 or experts % groups or not 1 <= keep <= groups or top > keep * (experts // groups):
            raise ValueError(f"{prefix}: top {top} of {experts} experts in {keep} of {groups} groups")
        if limit is not None and not gated:
            raise ValueError(f"{prefix}: capped experts are gated")
        self.on_logits = score == "softmax_top"
        if self.on_logits and (weigh != "output" or correction or groups != 1 or scale != 1.0):
            raise ValueError(f"{prefix}: a softmax over the chosen logits weighs outputs, without corrections, groups or scale")
        if (router_bias or shared_gate) and not self.on_logits or shared_gate and shared is None:
            raise ValueError(f"{prefix}: router_bias / shared_gate need score softmax_top, a gate needs a shared expert")
        self.router_bias, self.shared_gate = bool(router_bias), bool(shared_gate)
        self.p, self.width, self.E, self.top, self.ff = prefix, width, int(experts), int(top), int(ff)
        self.limit = None if limit is None else float(limit)
        self.alpha, self.renorm, self.shared = float(alpha), bool(renorm), shared
        self.softmax, self.on_output = score == "softmax", weigh == "output"
        self.gated, self.act_kind, self.correction = bool(gated), act, bool(correction)
        self.groups, self.keep, self.scale = int(groups), int(keep), float(scale)

    def act(self, gu: torch.Tensor) -> torch.Tensor:
        if not self.gated:
            return seqmix.unary_act(gu, self.act_kind)
        if self.limit is None:
            return seqmix.silu_mul(gu) if self.act_kind == "silu" else seqmix.act_mul(gu, self.act_kind)
        return seqmix.capped_glu(gu, self.limit, self.alpha)

    def shapes(self) -> dict:
        p, sh = self.p, {self.p + "router": (self.E, self.width)}
        if self.correction:
            sh[p + "correction"] = (self.E,)
        if self.router_bias:
            sh[p + "router.b"] = (self.E,)
        if self.shared_gate:
            sh[p + "shared.sg"] = (1, self.width)
        for e in range(self.E):
            if self.gated:
                sh[f"{p}e{e}.gate"] = (self.ff, self.width)
            sh[f"{p}e{e}.up"] = (self.ff, self.width)
            sh[f"{p}e{e}.down"] = (self.width, self.ff)
        if self.shared is not None:
            sh.update(self.shared.shapes())
        return sh

    def finish_weights(self, w: dict) -> None:
        p = self.p
        names = ("gate", "up") if self.gated else ("up",)
        w[p + "_in"] = torch.stack([torch.cat([w.pop(f"{p}e{e}.{n}") for n in names]).t() for e in range(self.E)]).contiguous()
        w[p + "_down"] = torch.stack([w.pop(f"{p}e{e}.down").t() for e in range(self.E)]).contiguous()
        if self.correction:
            w[p + "correction"] = w[p + "correction"].to(torch.float32).contiguous()
        if self.shared_gate:  # one more row of the router's projection
            w[p + "router"] = torch.cat([w[p + "router"], w.pop(p + "shared.sg")]).contiguous()
            if self.router_bias:
                w[p + "router.b"] = torch.cat([w[p + "router.b"], torch.zeros_like(w[p + "router.b"][:1])]).contiguous()
        if self.shared is not None:
            self.shared.finish_weights(w)

    def route(self, h: torch.Tensor, w: dict) -> tuple:
        """(weights fp32 [T, top], ids int32 [T, top], the shared expert's gate fp32 [T] or None)."""
        p = self.p
        if self.on_logits:
            tw, ids, gates = seqmix.route_linear(h, w[p + "router"], w.get(p + "router.b"), self.E, self.top)
            return tw, ids, gates.reshape(-1) if self.shared_gate else None
        logits = seqmix.gate_linear(h, w[p + "router"], None)  # fp32 products and sums
        return seqmix.route_topk(logits, self.top, self.renorm, self.softmax,
                                 correction=w[p + "correction"] if self.correction else None, groups=self.groups,
                                 keep=self.keep, scale=self.scale) + (None,)

    def slab_rows(self, offs: list, size: int) -> int:
        """Rows of an expert's slab for these offsets of sorted rows; 0: one product pair per expert."""
        counts = [b - a for a, b in zip(offs, offs[1:])]
        cap, used = max(counts), self.E - counts.count(0)
        up = 2 * self.ff if self.gated else self.ff
        per_row = self.width * (up + self.ff)  # multiply-adds of a row, weights of an expert
        row = 2 * self.width + up + self.ff  # what a row takes in memory; the up product's output is read once more, as is the rest
        empty = self.E * cap - offs[-1]
        cost = (2.0 * per_row * empty / self.SLAB_FLOPS
                + size * (2.0 * (row - self.width) * empty + per_row * (self.E - used)) / self.SLAB_BYTES)
        return cap if cost <= self.SLAB_GAIN_S * used and self.E * cap * row * size <= self.SLAB_MAX_BYTES else 0

    def rows(self, h: torch.Tensor, w: dict) -> seqmix.ExpertRows:
        """The experts' outputs and what sums them: for a layer whose stream update takes the sum itself."""
        p, T = self.p, h.shape[0]
        tw, ids, gate = self.route(h, w)
        w_in, w_out = (None, tw) if self.on_output else (tw, None)
        extra = self.shared.forward(h, w) if self.shared is not None else None
        up, down = w[p + "_in"], w[p + "_down"]
        capturing = h.is_cuda and torch.cuda.is_current_stream_capturing()
        if T <= self.BATCHED_MAX_TOKENS or T * self.E <= self.BATCHED_MAX_ROWS or capturing:
            xs = seqmix.spread_scaled(h, w_in, ids, self.E)  # [E, T, W]
            a = self.act(torch.bmm(xs, up).view(self.E * T, -1))
            ys = torch.bmm(a.view(self.E, T, -1), down)  # [E, T, W]
            if w_out is None:
                return seqmix.ExpertRows(ys, None, self.E, T, extra, row_stride=T, gate=gate)
            # weights on the outputs: a token's k chosen slabs, row (expert, t) of the stack
            return seqmix.ExpertRows(ys, ids.reshape(-1), self.top, T, extra, row_stride=T, weights=w_out, by_expert=True,
                                     gate=gate)
        offs, inv = seqmix.expert_align(ids, self.E)
        o = offs.tolist()  # the one host read of this path
        cap = self.slab_rows(o, up.element_size())
        if cap:
            xs, index = seqmix.gather_slabs(h, w_in, ids, offs, inv, cap)
            a = self.act(torch.bmm(xs, up).view(self.E * cap, -1))
            ys = torch.bmm(a.view(self.E, cap, -1), down)
            return seqmix.ExpertRows(ys, index, self.top, T, extra, weights=w_out, gate=gate)
        xs = seqmix.gather_scaled(h, w_in, inv, self.top)
        ys = torch.empty_like(xs)
        for e in range(self.E):
            a0, a1 = o[e], o[e + 1]
            if a1 > a0:
                torch.mm(self.act(torch.mm(xs[a0:a1], up[e])), down[e], out=ys[a0:a1])
        return seqmix.ExpertRows(ys, inv, self.top, T, extra, weights=w_out, gate=gate)

    def forward(self, h: torch.Tensor, w: dict) -> torch.Tensor:
        if self.shared_gate:
            raise ValueError(f"{self.p}: a gated shared expert's sum is taken by the stream update (rows())")
        r = self.rows(h, w)
        return seqmix.expert_combine(r.ys, r.index, r.k, r.T, r.extra, row_stride=r.row_stride, weights=r.weights,
                                     by_expert=r.by_expert)
