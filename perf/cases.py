"""The workloads that this framework's speed is measured on: engine steps of served models.

A pass is one step of the engine as the serving loop runs it: `ModelRunner.launch` on a scheduled batch (its
inputs prepared on the host, one upload, the captured graph of a batch of single tokens or the launches of a
batch with prompt chunks, the sampling of every finished row).  The models are the headline's Llama-3.2-1B and
two of the layer-list designs, which between them hold every kind of sublayer that the designs share most:
Tapasun (state space, rotary attention with a sink, gated delta rule) and Momuvik (latent attention), both with
the sizes that the design benchmark gives a width.  The routed feed-forward that four designs use is measured as
the sublayer it is: with random weights a router behind other layers sits on ties that any rounding turns over.

Every case says how many sequences bring one token (`decodes`, with contexts of ctx_lo .. ctx_hi tokens) and how
many bring a chunk (`chunks` of new_lo .. new_hi tokens behind past_lo .. past_hi tokens that are in the cache
already: a chat's earlier turns, an earlier chunk of a long prompt).  Lengths follow from the case alone, the
tokens, weights, pages and states from the seed.  Sampled tokens are not among the outputs: the weights are
random, so that the likeliest tokens lie closer together than bf16 tells apart; the logits are."""
from __future__ import annotations

import json
import math
import os
import tempfile

import torch

from mxserve.config import EngineArgs
from mxserve.engine.model_runner import ModelRunner
from mxserve.engine.request import Request, SamplingParams
from mxserve.engine.scheduler import ScheduledReq, SchedulerOutput
from mxserve.models import config as model_config
from mxserve.models.feedforward import CappedExpert, RoutedExperts
from mxserve.ops import decode_gemm

PAGE = 16  # tokens a cache block holds
F64 = torch.float64


# ------------------------------------------------------------------------------------------- the cases
def _step(name, model, width=0, decodes=0, ctx=(0, 0), chunks=0, new=(0, 0), past=(0, 0)):
    c = {"kind": "step", "model": model, "width": width, "decodes": decodes, "ctx_lo": ctx[0], "ctx_hi": ctx[1],
         "chunks": chunks, "new_lo": new[0], "new_hi": new[1], "past_lo": past[0], "past_hi": past[1]}
    return dict(c, name=name) if name else c


def _experts(name, width, tokens, replay):
    c = {"kind": "experts", "width": width, "tokens": tokens, "replay": replay}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one user in a chat: the smallest step, weights streamed for one token
        _step("llama-decode-1", "llama", decodes=1, ctx=(903, 903)),
        # the headline's running set: 4,000-token prompts, up to 500 tokens into their answers
        _step("llama-decode-256", "llama", decodes=256, ctx=(4001, 4500)),
        # the headline's prompt in a step of its own
        _step("llama-prompt-4000", "llama", chunks=1, new=(4000, 4000)),
        # conversations: new turns behind cached earlier ones, beside running answers
        _step("llama-chat", "llama", decodes=8, ctx=(300, 1500), chunks=5, new=(24, 310), past=(0, 900)),
        # a layer-list design with recurrent layers: a batch of answers, a long prompt, uneven work of both kinds
        _step("tapasun-decode-64", "tapasun", 2048, decodes=64, ctx=(1900, 2200)),
        _step("tapasun-prompt-4096", "tapasun", 2048, chunks=1, new=(4096, 4096)),
        _step("tapasun-ragged", "tapasun", 2048, decodes=6, ctx=(150, 1700), chunks=5, new=(17, 700), past=(0, 600)),
        # a layer-list design over latent pages: the same three
        _step("momuvik-decode-64", "momuvik", 2048, decodes=64, ctx=(1900, 2200)),
        _step("momuvik-prompt-4096", "momuvik", 2048, chunks=1, new=(4096, 4096)),
        _step("momuvik-ragged", "momuvik", 2048, decodes=12, ctx=(150, 1700), chunks=4, new=(40, 610), past=(0, 1500)),
        # eight capped experts, two per token, and a shared one: a decode batch (replayed, as in a captured step), a prompt
        _experts("experts-64", 2048, 64, True),
        _experts("experts-4096", 2048, 4096, False),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def span(lo, hi):
        a, b = log(lo, hi), log(lo, hi)
        return min(a, b), max(a, b)

    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed", "experts"])
    if kind == "experts":
        tokens = log(1, 4096)
        return _experts(None, rng.choice([1024, 2048]), tokens, tokens <= 64 and rng.random() < 0.7)
    model = rng.choice(["llama", "tapasun", "momuvik"])
    width = 0 if model == "llama" else rng.choice([1024, 2048])
    if kind == "decode":
        n = log(1, 256 if model == "llama" else 64)
        return _step(None, model, width, decodes=n, ctx=span(64, 4500 if model == "llama" else 2200))
    if kind == "prompt":
        chunks = rng.choice([1, 1, 2, 3, 5])
        new = span(16, 4000 // chunks)
        past = (0, 0) if rng.random() < 0.6 else span(16, 1500)
        return _step(None, model, width, chunks=chunks, new=new, past=past)
    return _step(None, model, width, decodes=log(1, 32), ctx=span(64, 2000), chunks=rng.choice([1, 2, 4, 7]),
                 new=span(8, 400), past=span(1, 900))


# ------------------------------------------------------------------------------------------- models
LLAMA = {"layers": 16, "width": 2048, "ff": 8192, "heads": 32, "kv_heads": 8, "dim": 64, "vocab": 128256}
VOCAB = 32000  # of the designs


def _tapasun(width):
    """State space, attention, attention beside a delta rule, attention on the second layer's pages."""
    heads, ffn = width // 64, {"kind": "dense", "ff": (8 * width // 3) // 256 * 256}
    att = {"heads": heads, "kv_heads": heads // 4, "dim": 64, "vdim": 64, "scale": 0.125,
           "rot": {"dims": 64, "base": 500000.0, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
    ssm = {"heads": width // 32, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}
    pair = {"left": {"heads": heads, "kv_heads": heads // 8, "dim": 64, "vdim": 64, "scale": 0.125,
                     "rot": {"dims": 32, "base": 500000.0, "scaling": {"factor": 4.0}}},
            "right": {"heads": width // 128, "kv_heads": width // 128, "dim": 128, "vdim": 128, "conv": 4},
            "left_scale": 0.5, "right_scale": 1.0}
    return {"architecture": "Tapasun", "width": width, "vocab": VOCAB, "norm": {"eps": 1e-5}, "embedding": {"scale": 1.0},
            "layers": [{"type": "mamba2", "mlp": ffn, "mixer": ssm}, {"type": "attention", "mlp": ffn, "mixer": att},
                       {"type": "parallel", "mlp": ffn, "mixer": pair},
                       {"type": "attention", "mlp": ffn, "mixer": dict(att, kv_from=1)}]}


def _momuvik(width):
    """Four layers of latent attention with dense feed-forwards."""
    att = {"heads": width // 128, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "q_rank": max(3 * width // 8, 256),
           "scale": 192 ** -0.5, "rot": {"dims": 64, "base": 10000.0}}
    layer = {"type": "latent_attention", "mixer": att, "mlp": {"kind": "dense", "ff": (8 * width // 3) // 256 * 256}}
    return {"architecture": "Momuvik", "width": width, "vocab": VOCAB, "norm": {"eps": 1e-5}, "embedding": {"scale": 1.0},
            "residual_mult": 1.0, "layers": [layer] * 4}


DESIGNS = {"tapasun": _tapasun, "momuvik": _momuvik}
_folders: dict = {}


def _model_name(case):
    """What --model gets: the registry's name, or a folder with the design's config.json."""
    if case["model"] == "llama":
        return "meta-llama/Llama-3.2-1B-Instruct"
    key = (case["model"], case["width"])
    if key not in _folders:
        _folders[key] = tempfile.TemporaryDirectory(prefix="%s-w%d-" % key)
        with open(os.path.join(_folders[key].name, "config.json"), "w") as f:
            json.dump(DESIGNS[case["model"]](case["width"]), f)
    return _folders[key].name


# ------------------------------------------------------------------------------------------- inputs
def _spread(lo, hi, n):
    return [lo + int((hi - lo) * ((0.31 + i * 0.6180339887) % 1.0) + 0.5) for i in range(n)]


def _lengths(case):
    """[(tokens in the cache, new tokens)], the single tokens first."""
    seqs = [(c - 1, 1) for c in _spread(case["ctx_lo"], case["ctx_hi"], case["decodes"])]
    return seqs + list(zip(_spread(case["past_lo"], case["past_hi"], case["chunks"]),
                           _spread(case["new_lo"], case["new_hi"], case["chunks"])))


def _batch(case, seed):
    """(sequences as (cached tokens, new tokens' ids, cache blocks), blocks in the pool).  Blocks are scattered over the
    pool; the last ones of the single-token sequences, which the step writes into, are the pool's first."""
    g = torch.Generator().manual_seed(seed)
    lengths, d = _lengths(case), case["decodes"]
    vocab = LLAMA["vocab"] if case["model"] == "llama" else VOCAB
    counts = [-(-(p + n) // PAGE) for p, n in lengths]
    total = sum(counts)
    free = (torch.randperm(total - d, generator=g) + d).tolist()
    seqs = []
    for i, ((p, n), c) in enumerate(zip(lengths, counts)):
        own = [free.pop() for _ in range(c - 1 if i < d else c)] + ([i] if i < d else [])
        seqs.append((p, torch.randint(3, vocab, (n,), generator=g).tolist(), own))
    return seqs, total


def _fill(t, g, std):
    """Random values of a pool, some rows at a time."""
    rows = max(1, (1 << 28) // max(1, t[0].numel()))
    for a in range(0, t.shape[0], rows):
        t[a:a + rows].normal_(0.0, std, generator=g)


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(seed * 7919 + salt)


STATE_STD = 0.2
GRAPHS = (1, 2, 4, 8, 16, 24, 32, 48, 64, 96, 128, 160, 192, 224, 256)


def _slots(case):
    n = case["decodes"] + case["chunks"]
    return next(b for b in GRAPHS if b >= max(n, 8 if case["chunks"] else 1))


def prepare(case, seed):
    if case["kind"] == "experts":
        return _prepare_experts(case, seed)
    seqs, blocks = _batch(case, seed)
    slots = _slots(case)
    args = EngineArgs(model=_model_name(case), device="cuda", dtype="bfloat16", block_size=PAGE, num_gpu_blocks=blocks,
                      max_num_seqs=slots, load_format="random", seed=seed, cuda_graph_max_bs=1 if case["chunks"] else slots)
    runner = ModelRunner(args, model_config.get_model_config(args.model))
    _fill(runner.kv_cache, _gen(seed, 1), 1.0)
    if runner.state is not None:
        _fill(runner.state, _gen(seed, 2), STATE_STD)
    so = SchedulerOutput()
    for i, (past, toks, own) in enumerate(seqs):
        sp = SamplingParams(max_tokens=64, seed=i, temperature=0.7 if i % 2 else 0.0, top_p=0.95)
        req = Request("r%d" % i, [0] * past + toks, sp, block_ids=own, num_computed_tokens=past)
        (so.decodes if i < case["decodes"] else so.prefills).append(ScheduledReq(req, len(toks), True, start=past))
    # a captured step's split sums go through a workspace of the process that the next engine's start replaces: with several
    # engines in one process, as here, each one's has to be kept for as long as its graphs
    return {"runner": runner, "so": so, "n": len(seqs), "pages": case["decodes"] if not case["chunks"] else blocks,
            "workspace": (decode_gemm.TABLE.part, decode_gemm.TABLE.cnt)}


@torch.inference_mode()
def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if "ff" in state:
        return state["ff"].forward(state["h"], state["w"])
    r, n = state["runner"], state["n"]
    r.launch(state["so"])
    out = {"logits": r._logits[:n], "pages": r.kv_cache[:state["pages"]]}
    if r.state is not None:
        out["state"] = r.state[:n]
    return out


# ------------------------------------------------------------------------------------------- routed experts
EXPERTS, TOP, LIMIT = 8, 2, 7.0


def _expert_sizes(width):
    return (4 * width // 3) // 256 * 256, max(width // 3 // 128 * 128, 128)


def _expert_inputs(case, seed):
    W = case["width"]
    ff, sf = _expert_sizes(W)
    g = _gen(seed, 3)

    def rnd(rows, cols, std=1.0):
        return (torch.randn(rows, cols, generator=g, device="cuda") * (std * cols ** -0.5)).to(torch.bfloat16)

    w = {"router": rnd(EXPERTS, W, 2.0)}
    for p, f in [("e%d." % e, ff) for e in range(EXPERTS)] + [("shared.", sf)]:
        w.update({p + "gate": rnd(f, W), p + "up": rnd(f, W), p + "down": rnd(W, f)})
    return torch.randn(case["tokens"], W, generator=g, device="cuda").to(torch.bfloat16), w


def _prepare_experts(case, seed):
    W = case["width"]
    ff, sf = _expert_sizes(W)
    h, w = _expert_inputs(case, seed)
    block = RoutedExperts("", W, EXPERTS, TOP, ff, LIMIT, CappedExpert("shared.", W, sf, LIMIT))
    block.finish_weights(w)
    if not case["replay"]:
        return {"ff": block, "h": h, "w": w}
    with torch.inference_mode():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                block.forward(h, w)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = block.forward(h, w)
    return {"graph": graph, "out": out, "h": h, "w": w, "block": block}


def _exact_experts(case, seed):
    h, w = _expert_inputs(case, seed)
    h, w = h.to(F64), {k: t.to(F64) for k, t in w.items()}

    def unit(x, p):
        a = torch.clamp(x @ w[p + "gate"].t(), max=LIMIT)
        return (a * torch.sigmoid(1.702 * a) * (torch.clamp(x @ w[p + "up"].t(), -LIMIT, LIMIT) + 1.0)) @ w[p + "down"].t()

    score = torch.sigmoid(h @ w["router"].t())
    top = score.topk(TOP, dim=-1).indices
    out = unit(h, "shared.")
    for e in range(EXPERTS):
        rows = (top == e).any(-1).nonzero().flatten()
        if rows.numel():
            out[rows] += unit(h[rows] * score[rows, e:e + 1], "e%d." % e)
    return out


# ------------------------------------------------------------------------------------------- work
def _keys(lengths):
    """Query-key pairs of a step."""
    return sum(n * p + n * (n + 1) // 2 for p, n in lengths)


def work(case):
    if case["kind"] == "experts":
        T, W = case["tokens"], case["width"]
        ff, sf = _expert_sizes(W)
        used = min(EXPERTS, TOP * T)
        return {"bytes": 2 * (3 * W * (used * ff + sf) + EXPERTS * W + 2 * T * W),
                "flops": 2 * T * W * (3 * (TOP * ff + sf) + EXPERTS)}
    lengths = _lengths(case)
    T, rows, ctx = sum(n for _, n in lengths), len(lengths), sum(p for p, _ in lengths)
    pairs = _keys(lengths)
    if case["model"] == "llama":
        c = LLAMA
        H, D = c["width"], c["dim"]
        qkv, o, mlp = H * D * (c["heads"] + 2 * c["kv_heads"]), H * H, 3 * H * c["ff"]
        weights, head, token = c["layers"] * (qkv + o + mlp), c["vocab"] * H, 2 * c["kv_heads"] * D * c["layers"]
        # behind the last layer's keys only the rows that give logits go on
        flops = 2 * (T * (weights - o - mlp) + rows * (o + mlp)) + 4 * c["heads"] * D * pairs * (c["layers"] - 1)
        state = 0
    else:
        W = case["width"]
        ff, head = 3 * W * ((8 * W // 3) // 256 * 256), VOCAB * W
        if case["model"] == "momuvik":
            H, q = W // 128, max(3 * W // 8, 256)
            layer = W * (q + 576) + q * H * 192 + H * 128 * 512 * 2 + H * 128 * W + ff
            weights, token, state = 4 * layer, 4 * 576, 0
            # single tokens meet the latents themselves, chunks the keys and values that every head expands from them
            single = _keys(lengths[:case["decodes"]])
            flops = 2 * T * weights + 4 * 2 * H * ((576 + 512) * single + (192 + 128) * (pairs - single))
        else:
            hq, h1, hd = W // 64, W // 32, W // 128
            inner, gn = h1 * 64, 8 * 128
            mamba = W * (2 * inner + 2 * gn + h1) + inner * W
            att, att2 = W * 64 * (hq + hq // 2) + W * W, 2 * W * W
            left, right = W * 64 * (hq + hq // 4) + W * W, W * (3 * hd * 128 + 32 + hd) + 32 * hd * 128 + hd * 128 * W
            weights, token = mamba + att + att2 + left + right + 4 * ff, 128 * (hq // 4 + hq // 8)
            s1, s2 = h1 * 64 * 128, hd * 128 * 128
            state = rows * 4 * 2 * (s1 + s2 + 3 * (inner + 2 * gn + 3 * hd * 128))
            flops = 2 * T * weights + 3 * 4 * hq * 64 * pairs + T * (4 * s1 + 7 * s2)
        weights += 0 if case["model"] == "momuvik" else min(T, VOCAB) * W  # the embedding is a table of its own
    return {"bytes": 2 * (weights + head + token * (ctx + T)) + state + rows * (LLAMA["vocab"] * 2 if case["model"] == "llama" else VOCAB * 4),
            "flops": flops + 2 * rows * head}


def tolerance(case):
    """Rounding of bf16 activations and weights through the layers: what the path is off from 64 bits, and with it what
    another order of its sums may be off from this one."""
    if case["kind"] == "experts":
        return {"rel": 0.015}
    return {"rel": 0.03}


# ------------------------------------------------------------------------------------------- in 64 bits
def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _attend(q, k, v, past, scale, sink=None):
    """q [m, H, d] at positions past .. past + m - 1, k, v [n, G, .] of positions 0 .. n - 1; sink [H]."""
    m, H, _ = q.shape
    n, G, _ = k.shape
    out = torch.empty(m, H, v.shape[2], dtype=F64, device=q.device)
    seen = torch.arange(n, device=q.device)[None, :] <= past + torch.arange(m, device=q.device)[:, None]
    for h in range(H):
        s = (q[:, h] @ k[:, h * G // H].t()).mul_(scale).masked_fill_(~seen, -math.inf)
        top = s.max(-1, keepdim=True).values
        if sink is not None:
            top = torch.clamp(top, min=float(sink[h]))
        p = torch.exp(s - top)
        z = p.sum(-1, keepdim=True)
        if sink is not None:
            z = z + torch.exp(sink[h] - top)
        out[:, h] = (p @ v[:, h * G // H]) / z
    return out


def _bands(f, sc):
    """Frequencies slowed by wavelength: long waves by the factor, short ones not, in between a blend."""
    wave = 2 * math.pi / f
    if wave < sc["original"] / sc["high"]:
        return f
    if wave > sc["original"] / sc["low"]:
        return f / sc["factor"]
    s = (sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])
    return (1 - s) * f / sc["factor"] + s * f


def _freqs(rot):
    f = [float(rot["base"]) ** (-2.0 * i / rot["dims"]) for i in range(rot["dims"] // 2)]
    sc = rot.get("scaling")
    if sc:
        f = [_bands(x, sc) if "original" in sc else x / sc["factor"] for x in f]
    return torch.tensor(f, dtype=F64, device="cuda")


def _turn(x, pos, f, halves, sign=1.0):
    """x [m, H, d]: pairs (i, i + d / 2) or (2i, 2i + 1) of the first 2 len(f) entries turned by pos * f."""
    a = sign * pos.to(F64)[:, None, None] * f
    c, s, n, y = torch.cos(a), torch.sin(a), 2 * f.numel(), x.clone()
    i, j = (slice(0, n // 2), slice(n // 2, n)) if halves else (slice(0, n, 2), slice(1, n, 2))
    u, v = x[..., i], x[..., j]
    y[..., i], y[..., j] = u * c - v * s, v * c + u * s
    return y


class _Pages:
    """The cache in 64 bits where it is returned, and as it was before the step where it is only read."""

    def __init__(self, pool, keep, seqs):
        self.old, self.new, self.seqs = pool, pool[:keep].to(F64), seqs

    def read(self, i, view):
        """Entries [past, ...] of sequence i; view(pool) -> [blocks, PAGE, ...]."""
        past, _, own = self.seqs[i]
        b = torch.tensor(own[:-(-past // PAGE)], dtype=torch.long, device="cuda")
        return view(self.old[b]).flatten(0, 1)[:past].to(F64)

    def write(self, i, view, x):
        past, toks, own = self.seqs[i]
        p = torch.arange(past, past + len(toks))
        b = torch.tensor(own)[p // PAGE].cuda()
        view(self.new)[b, (p % PAGE).cuda()] = x


def _exact_llama(seed, seqs, pages):
    c, eps = LLAMA, 1e-5
    H, D, G, V = c["heads"], c["dim"], c["kv_heads"], c["vocab"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003)

    def weight(*shape):
        return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0.0, 0.02, generator=g)

    f = _freqs({"base": 500000.0, "dims": D, "scaling": {"factor": 32.0, "low": 1.0, "high": 4.0, "original": 8192}})
    embed = weight(V, c["width"])
    ends = torch.tensor([len(t) for _, t, _ in seqs]).cumsum(0)
    x = embed[torch.tensor([t for s in seqs for t in s[1]], device="cuda")].to(F64)
    for layer in range(c["layers"]):
        wqkv, wo = weight((H + 2 * G) * D, c["width"]).to(F64), weight(c["width"], H * D).to(F64)
        wgu, wd = weight(2 * c["ff"], c["width"]).to(F64), weight(c["width"], c["ff"]).to(F64)
        y = _rms(x, eps) @ wqkv.t()
        o = torch.empty(x.shape[0], H * D, dtype=F64, device="cuda")
        kview = lambda p: p[:, layer, 0].transpose(1, 2)  # noqa: E731  [blocks, PAGE, G, D]
        vview = lambda p: p[:, layer, 1].view(p.shape[0], G, D, PAGE).permute(0, 3, 1, 2)  # noqa: E731
        for i, (past, toks, _) in enumerate(seqs):
            e = int(ends[i])
            a, m = e - len(toks), len(toks)
            pos = torch.arange(past, past + m, device="cuda")
            q, k, v = y[a:e].view(m, H + 2 * G, D).split([H, G, G], dim=1)
            q, k = _turn(q, pos, f, True), _turn(k, pos, f, True)
            pages.write(i, kview, k)
            pages.write(i, vview, v)
            o[a:e] = _attend(q, torch.cat([pages.read(i, kview), k]), torch.cat([pages.read(i, vview), v]), past,
                             D ** -0.5).reshape(m, -1)
        x = x + o @ wo.t()
        gu = _rms(x, eps) @ wgu.t()
        x = x + (_silu(gu[:, :c["ff"]]) * gu[:, c["ff"]:]) @ wd.t()
    return _rms(x[(ends - 1).cuda()], eps) @ embed.to(F64).t()


def _design_names(d, model):
    """[(name, shape)] of a design's tensors."""
    W = d["width"]
    ff = (8 * W // 3) // 256 * 256
    names = [("embed", (VOCAB, W))]
    names += [("final.norm", ()), ("head", (VOCAB, W))] if model == "tapasun" else [("final.norm", (W,))]
    for i, layer in enumerate(d["layers"]):
        p, mx = "l%d." % i, layer["mixer"]
        m = p + "mix."
        if model == "momuvik":
            H, q, r = mx["heads"], mx["q_rank"], mx["kv_rank"]
            names += [(p + "norm1", (W,)), (m + "dq", (q, W)), (m + "dkv", (r + 64, W)), (m + "dq.norm", (q,)),
                      (m + "dkv.norm", (r,)), (m + "uq", (H * 192, q)), (m + "uk", (H * 128, r)), (m + "uv", (H * 128, r)),
                      (m + "o", (W, H * 128)), (m + "sink", (H,)), (p + "norm2", (W,))]
        else:
            names += [(p + "norm1", ()), (p + "norm1b", ())]
            if layer["type"] == "mamba2":
                H, inner, gn = mx["heads"], mx["heads"] * mx["vdim"], mx["groups"] * mx["state"]
                names += [(m + "in", (2 * inner + 2 * gn + H, W)), (m + "conv", (inner + 2 * gn, 4)),
                          (m + "conv.b", (inner + 2 * gn,)), (m + "dt_bias", (H,)), (m + "A_log", (H,)), (m + "D", (H,)),
                          (m + "norm", (inner,)), (m + "o", (W, inner))]
            else:
                l = mx.get("left", mx)
                a, hq, hk = m + ("left." if "left" in mx else ""), l["heads"] * 64, l["kv_heads"] * 64
                own = l.get("kv_from") is None
                names += [(a + "q", (hq, W))] + ([(a + "k", (hk, W)), (a + "v", (hk, W))] if own else [])
                more = [(a + "o", (W, hq))]
                if "left" in mx:
                    H, b = mx["right"]["heads"], m + "right."
                    n = H * 128
                    names += [(b + "q", (n, W)), (b + "k", (n, W)), (b + "v", (n, W)), (b + "a1", (16, W)), (b + "g1", (16, W)),
                              (b + "b", (H, W))]
                    more += [(a + "sink", (l["heads"],)), (b + "q.conv", (n, 4)), (b + "k.conv", (n, 4)), (b + "v.conv", (n, 4)),
                             (b + "a2", (n, 16)), (b + "g2", (n, 16)), (b + "dt_bias", (n,)), (b + "A_log", (H,)),
                             (b + "norm", (128,)), (b + "o", (W, n))]
                else:
                    more += [(a + "q.norm", (64,))] + ([(a + "k.norm", (64,))] if own else [])
                names += more
            names += [(p + "norm2", ()), (p + "norm2b", ())]
        names += [(p + "mlp.gate", (ff, W)), (p + "mlp.up", (ff, W)), (p + "mlp.down", (W, ff))]
    return names


def _design_weights(model, width, seed):
    """The random weights of a design by name: projections of unit gain, and numbers of their own for norms, sinks and the
    constants of the recurrences, drawn in the order of the design's tensors."""
    d = DESIGNS[model](width)
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = {}
    for name, shape in _design_names(d, model):
        t, leaf = torch.randn(shape, generator=g, device="cuda"), name.rsplit(".", 1)[-1]
        if not shape:
            t = 1.0 + 0.2 * t
        elif leaf in ("norm1", "norm2") or name == "final.norm":
            t = 0.1 * t
        elif leaf == "norm":
            t = 1.0 + 0.1 * t
        elif leaf == "A_log":
            t = -0.5 + 0.8 * t
        elif leaf == "dt_bias":
            t = -1.0 + t
        elif leaf == "b" and len(shape) == 1:
            t = 0.1 * t
        elif leaf not in ("D", "sink"):
            t = t * shape[1] ** -0.5
        w[name] = t.to(torch.bfloat16)
    return d, w


def _conv(x, carried, w, bias):
    """Causal filter of a chunk x [m, C] behind the carried inputs [taps - 1, C] (replaced), then SiLU."""
    full = torch.cat([carried, x])
    taps = w.shape[1]
    y = sum(w[:, j] * full[j:j + x.shape[0]] for j in range(taps))
    carried.copy_(full[x.shape[0]:])
    return _silu(y if bias is None else y + bias)


def _mamba2(mx, w, p, h, state, fresh):
    H, P, N, G = mx["heads"], mx["vdim"], mx["state"], mx["groups"]
    I, C = H * P, H * P + 2 * G * N
    S, carried = state[:H * P * N].view(H, P, N), state[H * P * N:H * P * N + 3 * C].view(3, C)
    if fresh:
        S.zero_(), carried.zero_()
    y = h @ w[p + "in"].t()
    z, dt = y[:, :I], torch.nn.functional.softplus(y[:, I + C:] + w[p + "dt_bias"])
    c = _conv(y[:, I:I + C], carried, w[p + "conv"], w[p + "conv.b"])
    x = c[:, :I].view(-1, H, P)
    B, R = (c[:, I + k * G * N:I + (k + 1) * G * N].view(-1, G, N).repeat_interleave(H // G, dim=1) for k in (0, 1))
    a, out = torch.exp(-torch.exp(w[p + "A_log"]) * dt), torch.empty_like(x)
    for t in range(h.shape[0]):
        S.mul_(a[t].view(H, 1, 1)).add_((dt[t].view(H, 1) * x[t]).unsqueeze(2) * B[t].unsqueeze(1))
        torch.matmul(S, R[t].unsqueeze(2), out=out[t].unsqueeze(2))
    o = (out + w[p + "D"].view(H, 1) * x).reshape(-1, I) * _silu(z)
    return (_rms(o.view(o.shape[0], mx["norm_groups"], -1), 1e-5).reshape(-1, I) * w[p + "norm"]) @ w[p + "o"].t()


def _delta(mx, w, p, h, state, fresh):
    H, D = mx["heads"], mx["dim"]
    n = H * D
    S, carried = state[:n * D].view(H, D, D), state[n * D:n * D + 9 * n].view(3, 3 * n)  # S: [head, value, key]
    if fresh:
        S.zero_(), carried.zero_()
    taps = torch.cat([w[p + k + ".conv"] for k in "qkv"])
    c = _conv(torch.cat([h @ w[p + k].t() for k in "qkv"], dim=1), carried, taps, None)
    q, k, v = (c[:, i * n:(i + 1) * n].view(-1, H, D) for i in range(3))
    q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) * D ** -0.5
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    beta = torch.sigmoid(h @ w[p + "b"].t())
    d = torch.nn.functional.softplus((h @ w[p + "a1"].t()) @ w[p + "a2"].t() + w[p + "dt_bias"]).view(-1, H, D)
    a, out = torch.exp(-torch.exp(w[p + "A_log"]).view(H, 1) * d), torch.empty_like(v)
    for t in range(h.shape[0]):
        S.mul_(a[t].unsqueeze(1))
        u = beta[t].view(H, 1) * (v[t] - (S @ k[t].unsqueeze(2)).squeeze(2))
        S.add_(u.unsqueeze(2) * k[t].unsqueeze(1))
        torch.matmul(S, q[t].unsqueeze(2), out=out[t].unsqueeze(2))
    gate = torch.sigmoid((h @ w[p + "g1"].t()) @ w[p + "g2"].t())
    return ((_rms(out, 1e-5) * w[p + "norm"]).reshape(-1, n) * gate) @ w[p + "o"].t()


def _exact_design(case, seed, seqs, pages, state):
    model, W = case["model"], case["width"]
    d, w = _design_weights(model, W, seed)
    w = {k: t.to(F64) for k, t in w.items()}
    eps, tap = 1e-5, model == "tapasun"
    spans, e = [], 0
    for past, toks, _ in seqs:
        spans.append((past, e, e + len(toks)))
        e += len(toks)
    x = w["embed"][torch.tensor([t for s in seqs for t in s[1]], device="cuda")]
    koff = soff = 0
    shared = {}
    for i, layer in enumerate(d["layers"]):
        p, mx = "l%d." % i, layer["mixer"]
        m = p + "mix."
        h = _rms(x, eps) * (w[p + "norm1"] if tap else 1.0 + w[p + "norm1"])
        y = torch.zeros_like(x)
        if layer["type"] == "mamba2":
            C = mx["heads"] * mx["vdim"] + 2 * mx["groups"] * mx["state"]
            size = mx["heads"] * mx["vdim"] * mx["state"] + 3 * C
            for s, (past, a, e) in enumerate(spans):
                y[a:e] = _mamba2(mx, w, m, h[a:e], state[s, soff:soff + size], past == 0)
            soff += size
        elif layer["type"] == "latent_attention":
            H, r, f = mx["heads"], mx["kv_rank"], _freqs(mx["rot"])
            view = lambda pool: pool[:, koff:koff + PAGE * (r + 64)].view(-1, PAGE, r + 64)  # noqa: E731
            uk, uv = w[m + "uk"].view(H, 128, r), w[m + "uv"].view(H, 128, r)
            for s, (past, a, e) in enumerate(spans):
                pos = torch.arange(past, past + e - a, device="cuda")
                q = ((_rms(h[a:e] @ w[m + "dq"].t(), eps) * w[m + "dq.norm"]) @ w[m + "uq"].t()).view(-1, H, 192)
                q = torch.cat([q[..., :128], _turn(q[..., 128:], pos, f, True)], dim=-1)
                kv = h[a:e] @ w[m + "dkv"].t()
                row = torch.cat([_rms(kv[:, :r], eps) * w[m + "dkv.norm"], _turn(kv[:, None, r:], pos, f, True)[:, 0]], dim=-1)
                pages.write(s, view, row)
                rows = torch.cat([pages.read(s, view), row])
                o = torch.empty(e - a, H * 128, dtype=F64, device="cuda")
                for j in range(H):
                    k = torch.cat([rows[:, :r] @ uk[j].t(), rows[:, r:]], dim=-1)
                    o[:, j * 128:(j + 1) * 128] = _attend(q[:, j:j + 1], k[:, None], (rows[:, :r] @ uv[j].t())[:, None], past,
                                                          mx["scale"], w[m + "sink"][j:j + 1])[:, 0]
                y[a:e] = o @ w[m + "o"].t()
            koff += PAGE * (r + 64)
        else:
            pair = "left" in mx
            l, b = (mx["left"], m + "left.") if pair else (mx, m)
            H, G, f = l["heads"], l["kv_heads"], _freqs(l["rot"])
            vf = _freqs({"base": l["rot"]["base"], "dims": 64})
            own = l.get("kv_from") is None
            if own:
                shared[i], koff = koff, koff + 2 * G * PAGE * 64
            at = shared[i if own else l["kv_from"]]
            views = [lambda pool, o=at + k * G * PAGE * 64: pool[:, o:o + G * PAGE * 64].view(-1, G, PAGE, 64).transpose(1, 2)
                     for k in (0, 1)]
            sink = w[m + "left.sink"] if pair else torch.zeros(H, dtype=F64, device="cuda")
            for s, (past, a, e) in enumerate(spans):
                pos = torch.arange(past, past + e - a, device="cuda")
                q = (h[a:e] @ w[b + "q"].t()).view(-1, H, 64)
                if not pair:
                    q = _rms(q, eps) * w[b + "q.norm"]
                if own:
                    k, v = ((h[a:e] @ w[b + n].t()).view(-1, G, 64) for n in "kv")
                    if not pair:
                        k = _rms(k, eps) * w[b + "k.norm"]
                    k, v = _turn(k, pos, f, False), _turn(v, pos, vf, False) if pair else v
                    new = [torch.cat([pages.read(s, u), t]) for u, t in zip(views, (k, v))]
                    pages.write(s, views[0], k), pages.write(s, views[1], v)
                    shared[i, s] = new
                k, v = shared[i if own else l["kv_from"], s]
                o = _attend(_turn(q, pos, f, False), k, v, past, l["scale"], sink)
                if pair:
                    o = _turn(o, pos, vf, False, -1.0)
                y[a:e] = (o.reshape(e - a, -1) @ w[b + "o"].t()) * (mx["left_scale"] if pair else 1.0)
            if pair:
                n = mx["right"]["heads"] * 128
                size = n * 128 + 9 * n
                for s, (past, a, e) in enumerate(spans):
                    y[a:e] += mx["right_scale"] * _delta(mx["right"], w, m + "right.", h[a:e], state[s, soff:soff + size], past == 0)
                soff += size
        x = x + (_rms(y, eps) * w[p + "norm1b"] if tap else y)
        h = _rms(x, eps) * (w[p + "norm2"] if tap else 1.0 + w[p + "norm2"])
        y = (_silu(h @ w[p + "mlp.gate"].t()) * (h @ w[p + "mlp.up"].t())) @ w[p + "mlp.down"].t()
        x = x + (_rms(y, eps) * w[p + "norm2b"] if tap else y)
    last = _rms(x[[e - 1 for _, _, e in spans]], eps) * (w["final.norm"] if tap else 1.0 + w["final.norm"])
    return last @ w["head" if tap else "embed"].t()


@torch.inference_mode()
def exact(case, seed):
    if case["kind"] == "experts":
        return _exact_experts(case, seed)
    seqs, blocks = _batch(case, seed)
    llama = case["model"] == "llama"
    row = {"llama": (16, 2, 8, PAGE, 64), "tapasun": (PAGE * 2 * 64 * (case["width"] // 256 + case["width"] // 512),),
           "momuvik": (4 * PAGE * 576,)}[case["model"]]
    pool = torch.empty(blocks, *row, dtype=torch.bfloat16, device="cuda")
    _fill(pool, _gen(seed, 1), 1.0)
    pages = _Pages(pool, blocks if case["chunks"] else case["decodes"], seqs)
    if llama:
        return {"logits": _exact_llama(seed, seqs, pages), "pages": pages.new}
    if case["model"] == "momuvik":
        return {"logits": _exact_design(case, seed, seqs, pages, None), "pages": pages.new}
    W = case["width"]
    floats = (W // 32) * 64 * 128 + 3 * (W // 32 * 64 + 2048) + W * 128 + 9 * W
    state = torch.empty(_slots(case) + 8, floats, dtype=torch.float32, device="cuda")
    _fill(state, _gen(seed, 2), STATE_STD)
    state = state[:len(seqs)].to(F64)
    return {"logits": _exact_design(case, seed, seqs, pages, state), "pages": pages.new, "state": state}
