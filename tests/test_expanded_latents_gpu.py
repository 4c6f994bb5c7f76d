"""Latent attention of chunks on keys and values that every head expands from the gathered rows: the kernels against 64
bits at borders of tiles and pages, and the mixer's two ways (expanded, folded) against its formulas."""
import math
import types

import pytest
import torch

from mxserve.models import mixers
from mxserve.models.mixers import LatentAttention, StepContext
from mxserve.ops import seqmix

pytestmark = pytest.mark.gpu


def softmax_mix(q, K, V, past, scale, sink, window, lo=0):
    """q [m, H, d] at positions past .., K, V [n, H, .] of positions lo .. -> [m, H, dv], all in 64 bits."""
    m, n = q.shape[0], K.shape[0]
    i, j = past + torch.arange(m)[:, None], lo + torch.arange(n)[None, :]
    seen = (j <= i) & ((i - j < window) if window > 0 else torch.tensor(True))
    s = torch.einsum("mhd,nhd->hmn", q, K) * scale
    s = s.masked_fill(~seen, -math.inf)
    if sink is not None:
        s = torch.cat([s, sink.double().view(-1, 1, 1).expand(-1, m, 1)], -1)
    return torch.einsum("hmn,nhd->mhd", torch.softmax(s, -1)[..., :n], V)


@pytest.mark.parametrize("H,dn,dr,dv,rank", [(2, 128, 64, 128, 512), (3, 8, 8, 16, 16), (4, 64, 32, 48, 64), (1, 104, 88, 112, 40)])
@pytest.mark.parametrize("chunks,window", [([(0, 64)], 0), ([(0, 31), (17, 33), (0, 1)], 0), ([(100, 129), (0, 200)], 0),
                                           ([(100, 129), (3, 40), (300, 5)], 40), ([(64, 128), (0, 32)], 17)])
def test_gathered_rows_and_their_attention(gpu, H, dn, dr, dv, rank, chunks, window):
    g = torch.Generator().manual_seed(H * 100 + dn + window)
    dk, koff = rank + dr, 24
    nb = [-(-(p + n) // 16) for p, n in chunks]
    bt = torch.zeros(len(chunks), max(nb) + 1, dtype=torch.int32)
    ids, used = torch.randperm(sum(nb), generator=g), 0
    for s, n in enumerate(nb):
        bt[s, :n] = ids[used:used + n]
        used += n
    cache = torch.randn(sum(nb), koff + 16 * dk + 8, generator=g).bfloat16()
    qsl = torch.tensor([0] + [n for _, n in chunks]).cumsum(0).int()
    lens = torch.tensor([p + n for p, n in chunks], dtype=torch.int32)
    base, offs = seqmix.latent_plan(qsl, lens, window)
    gbase, goffs = seqmix.latent_plan(qsl.to(gpu), lens.to(gpu), window)
    assert torch.equal(gbase.cpu(), base) and torch.equal(goffs.cpu(), offs)
    n = int(offs[-1])
    rows = seqmix.latent_rows(cache, bt, base, offs, n, koff, dk, 16)
    assert torch.equal(seqmix.latent_rows(cache.to(gpu), bt.to(gpu), gbase, goffs, n, koff, dk, 16).cpu(), rows)
    q = torch.randn(int(qsl[-1]), H * (dn + dr), generator=g).bfloat16()
    kv = torch.randn(n, H * (dn + dv), generator=g).bfloat16()
    sink, scale = torch.randn(H, generator=g), (dn + dr) ** -0.5
    got = seqmix.expanded_attention(q.to(gpu), kv.to(gpu), rows.to(gpu), gbase, qsl.to(gpu), lens.to(gpu), H, dn, dr, dv, scale,
                                    max(m for _, m in chunks), sink.to(gpu), window).cpu().double()
    plain = seqmix.expanded_attention(q, kv, rows, base, qsl, lens, H, dn, dr, dv, scale, 0, sink, window).double()
    for s, (p, m) in enumerate(chunks):
        a, e, r = int(qsl[s]), int(qsl[s + 1]), slice(int(offs[s]), int(offs[s + 1]))
        K = torch.cat([kv[r, :H * dn].view(-1, H, dn), rows[r, rank:].unsqueeze(1).expand(-1, H, -1)], -1).double()
        want = softmax_mix(q[a:e].double().view(-1, H, dn + dr), K, kv[r, H * dn:].view(-1, H, dv).double(), p, scale, sink, window,
                           int(offs[s] - base[s])).reshape(e - a, -1)
        for x in (got, plain):  # bf16 result (2^-9 of it), weights of 16 bits (kernel) or fp32 (plain form)
            err = (x[a:e] - want).abs() - 2.0 ** -8 * want.abs()
            assert float(err.max()) <= 2.0 ** -13 * float(kv.float().abs().max()), (s, float(err.max()))


@pytest.mark.parametrize("oldest", [0, 15, 16, 31, 32, 47, 2048, 2063])
@pytest.mark.parametrize("window,new", [(40, 130), (17, 20), (1024, 300)])
def test_windowed_rows_between_others(gpu, oldest, window, new):
    """The rows around a sequence's own are no numbers, before the first sequence and between two: a tile that begins a page
    before the first gathered row takes nothing from there."""
    H, dn, dr, dv, rank = 2, 128, 64, 128, 64
    g = torch.Generator().manual_seed(oldest + window)
    past = oldest + window - 1  # the first query's oldest key is `oldest`
    chunks = [(past, new), (0, 16), (past, new)]
    qsl = torch.tensor([0] + [n for _, n in chunks]).cumsum(0).int()
    lens = torch.tensor([p + n for p, n in chunks], dtype=torch.int32)
    base, offs = seqmix.latent_plan(qsl.to(gpu), lens.to(gpu), window)
    off = offs.tolist()
    q = torch.randn(int(qsl[-1]), H * (dn + dr), generator=g).bfloat16()
    kv, rows = (torch.full((off[-1] + 64, n), float("nan"), dtype=torch.bfloat16) for n in (H * (dn + dv), rank + dr))
    for a, e in ((off[0], off[1]), (off[2], off[3])):  # the second sequence's rows are no numbers either
        kv[32 + a:32 + e] = torch.randn(e - a, kv.shape[1], generator=g).bfloat16()
        rows[32 + a:32 + e] = torch.randn(e - a, rows.shape[1], generator=g).bfloat16()
    inner = slice(32, 32 + off[-1])
    sink, scale = torch.randn(H, generator=g), (dn + dr) ** -0.5
    got = seqmix.expanded_attention(q.to(gpu), kv.to(gpu)[inner], rows.to(gpu)[inner], base, qsl.to(gpu), lens.to(gpu), H, dn, dr, dv,
                                    scale, new, sink.to(gpu), window, max_seq_len=past + new).cpu().double()
    kv, rows = kv[inner], rows[inner]
    for s in (0, 2):
        a, e, r = int(qsl[s]), int(qsl[s + 1]), slice(off[s], off[s + 1])
        K = torch.cat([kv[r, :H * dn].view(-1, H, dn), rows[r, rank:].unsqueeze(1).expand(-1, H, -1)], -1).double()
        want = softmax_mix(q[a:e].double().view(-1, H, dn + dr), K, kv[r, H * dn:].view(-1, H, dv).double(), past, scale, sink, window,
                           off[s] - int(base[s])).reshape(e - a, -1)
        err = (got[a:e] - want).abs() - 2.0 ** -8 * want.abs()  # as above
        assert float(err.max()) <= 2.0 ** -13 * float(kv[r].float().abs().max()), (s, float(err.max()))


@pytest.mark.parametrize("window", [0, 50])
@pytest.mark.parametrize("singles", [0, 3])
def test_mixer_expands_and_folds(gpu, monkeypatch, window, singles):
    """A step of chunks (and single tokens before them): what the mixer gives with the chunks' lengths known and unknown,
    both against the formulas in 64 bits; the expanded way is no further off."""
    monkeypatch.setattr(mixers, "EXPAND_MIN_QUERIES", 16)  # chunks of this size fold when left to themselves
    monkeypatch.setattr(mixers, "EXPAND_MIN_PAIRS", 0)
    W, H, dn, dr, vd, rank, qr = 256, 4, 128, 64, 128, 128, 192
    rot = {"dims": dr, "base": 10000.0}
    m = LatentAttention("", W, H, dn, dr, vd, rank, qr, 192 ** -0.5, rot, window=window)
    g = torch.Generator().manual_seed(window + singles)
    names = m.proj_rows()
    w = {k: torch.randn(s, generator=g) * (s[-1] ** -0.5 if len(s) == 2 else 1.0) for k, s in
         {**{k: (r, W) for k, r in names}, **m.extra_shapes()}.items()}
    for k in ("dq.norm", "dkv.norm"):
        w[k] = 1.0 + 0.1 * w[k]
    w = {k: t.bfloat16() for k, t in w.items()}
    lens = [(40 + 30 * i, 1) for i in range(singles)] + [(0, 150), (200, 90), (16, 70)]
    T = sum(n for _, n in lens)
    h = torch.randn(T, W, generator=g).bfloat16()
    nb = [-(-(p + n) // 16) for p, n in lens]
    bt = torch.zeros(len(lens), max(nb), dtype=torch.int32)
    ids, used = torch.randperm(sum(nb), generator=g), 0
    for s, n in enumerate(nb):
        bt[s, :n] = ids[used:used + n]
        used += n
    cache = torch.randn(sum(nb), 16 * m.dk, generator=g).bfloat16()
    pos = torch.cat([torch.arange(p, p + n) for p, n in lens])
    slots = torch.cat([bt[s].long()[torch.arange(p, p + n) // 16] * 16 + torch.arange(p, p + n) % 16 for s, (p, n) in enumerate(lens)])
    qsl = torch.tensor([0] + [n for _, n in lens]).cumsum(0).int()
    wg = {k: t.to(gpu) for k, t in w.items()}
    w_in = torch.cat([wg.pop(k) for k, _ in names])
    m.finish_weights(wg)
    outs = {}
    for way in ("expanded", "folded"):
        c = cache.to(gpu)
        md = types.SimpleNamespace(
            positions=pos.to(gpu), slot_mapping=slots.to(gpu), block_tables=bt.to(gpu), query_start_loc=qsl.to(gpu),
            prefill_query_start_loc=(qsl[singles:] - qsl[singles]).to(gpu), max_query_len=150, max_seq_len=290, num_decodes=singles,
            seq_lens=torch.tensor([p + n for p, n in lens], dtype=torch.int32, device=gpu),
            chunks=tuple(lens[singles:]) if way == "expanded" else None)
        ctx = StepContext(md=md, cache=c, state=None, block_size=16, eps=1e-5)
        y = h.to(gpu) @ w_in.T
        outs[way] = m.forward([y[:, :qr], y[:, qr:]], h.to(gpu), wg, ctx, 0, 0, 0).cpu().double()
        assert (ctx.expansion(window, H) is not None) == (way == "expanded")
    d = {k: t.double() for k, t in w.items()}
    f = torch.tensor([10000.0 ** (-2.0 * i / dr) for i in range(dr // 2)], dtype=torch.float64)

    def turn(x, at):
        a = at.double().view(-1, *([1] * (x.dim() - 1))) * f
        u, v = x[..., :dr // 2], x[..., dr // 2:]
        return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)

    rms = lambda x: x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5)  # noqa: E731
    x = h.double()
    q = ((rms(x @ d["dq"].T) * d["dq.norm"]) @ d["uq"].T).view(T, H, dn + dr)
    q = torch.cat([q[..., :dn], turn(q[..., dn:], pos)], -1)
    kv = x @ d["dkv"].T
    new = torch.cat([rms(kv[:, :rank]) * d["dkv.norm"], turn(kv[:, rank:], pos)], -1)
    want = []
    for s, (p, n) in enumerate(lens):
        a = int(qsl[s])
        old = cache[bt[s, :nb[s]].long()].view(-1, m.dk)[:p].double()
        r = torch.cat([old, new[a:a + n]])
        K = torch.cat([(r[:, :rank] @ d["uk"].T).view(-1, H, dn), r[:, None, rank:].expand(-1, H, -1)], -1)
        want.append(softmax_mix(q[a:a + n], K, (r[:, :rank] @ d["uv"].T).view(-1, H, vd), p, 192 ** -0.5, d["sink"], window).reshape(n, -1))
    want = torch.cat(want) @ d["o"].T
    err = {k: float((o - want).norm() / want.norm()) for k, o in outs.items()}
    # the chain of bf16 roundings (projections, rows, keys, values, outputs): about six of 2^-9 each
    assert err["folded"] < 0.012 and err["expanded"] < 0.012 and err["expanded"] <= err["folded"], err


@pytest.mark.parametrize("past,new,window", [(0, 140, 0), (75, 130, 50)])
def test_a_value_reaches_only_queries_that_see_it(gpu, past, new, window):
    """A gathered row whose expanded value is no number: queries that do not see its key give what they give without it."""
    H, dn, dr, dv, rank = 2, 64, 32, 96, 64
    g = torch.Generator().manual_seed(past)
    qsl, lens = torch.tensor([0, new], dtype=torch.int32, device=gpu), torch.tensor([past + new], dtype=torch.int32, device=gpu)
    base, offs = seqmix.latent_plan(qsl, lens, window)
    n, b = int(offs[1]), int(base[0])
    q, kv, rows = (torch.randn(*s, generator=g).bfloat16().to(gpu) for s in ((new, H * (dn + dr)), (n, H * (dn + dv)), (n, rank + dr)))
    run = lambda kv: seqmix.expanded_attention(q, kv, rows, base, qsl, lens, H, dn, dr, dv, 0.1, new, None, window).cpu().float()  # noqa: E731
    clean, i = run(kv), past + torch.arange(new)
    for j in (past + 3, past + 40, past + 63, past + new - 2, max(past - 20, 0)):
        broken = kv.clone()
        broken[b + j, H * dn + dv + 5] = float("nan")  # head 1, entry 5
        y = run(broken).view(new, H, dv)
        seen = (i >= j) & ((i - j < window) if window > 0 else torch.tensor(True))
        assert not torch.isfinite(y[seen, 1, 5]).any()
        y[seen, 1, 5] = clean.view(new, H, dv)[seen, 1, 5]
        torch.testing.assert_close(y.view(new, -1), clean, rtol=2.0 ** -7, atol=2.0 ** -12)


def test_pages_off_the_16_byte_grid_fold(gpu, monkeypatch):
    """Pages that the gathering kernel does not take are served by the folded form, as before there was another."""
    monkeypatch.setattr(mixers, "EXPAND_MIN_QUERIES", 0)
    monkeypatch.setattr(mixers, "EXPAND_MIN_PAIRS", 0)
    W, H, T, rot = 128, 2, 80, {"dims": 32, "base": 10000.0}
    m = LatentAttention("", W, H, 64, 32, 64, 64, 64, 96 ** -0.5, rot)
    g = torch.Generator().manual_seed(3)
    names = m.proj_rows()
    w = {k: (torch.randn(s, generator=g) * s[-1] ** -0.5).bfloat16().to(gpu) for k, s in
         {**{k: (r, W) for k, r in names}, **m.extra_shapes()}.items()}
    h = torch.randn(T, W, generator=g).bfloat16().to(gpu)
    y = h @ torch.cat([w.pop(k) for k, _ in names]).T
    m.finish_weights(w)
    pos = torch.arange(T, device=gpu)
    ints = [torch.tensor(x, dtype=torch.int32, device=gpu) for x in ([[0, 1, 2, 3, 4]], [0, T], [T])]
    md = types.SimpleNamespace(positions=pos, slot_mapping=pos, block_tables=ints[0], query_start_loc=ints[1],
                               prefill_query_start_loc=ints[1], seq_lens=ints[2], max_query_len=T, max_seq_len=T, num_decodes=0,
                               chunks=((0, T),))
    outs = []
    for shift in (0, 4):
        cache = torch.zeros(5 * 16 * m.dk + 8, dtype=torch.bfloat16, device=gpu)[shift:shift + 5 * 16 * m.dk].view(5, -1)
        outs.append(m.forward([y[:, :64], y[:, 64:]], h, w, StepContext(md=md, cache=cache, state=None, block_size=16, eps=1e-5), 0, 0, 0))
    # both forms round queries or keys, values and outputs to bf16: some 2^-8 of the layer's scale
    assert float((outs[0] - outs[1]).float().norm() / outs[0].float().norm()) < 0.012
