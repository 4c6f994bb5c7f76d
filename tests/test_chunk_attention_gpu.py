"""Attention of prompt chunks on the matrix cores against softmax in 64 bits: head sizes that fill the registers and that
ride in zeroed columns, groups of query heads that do not divide a tile, chunks around the borders of tiles and pages,
windows with kept first tokens, sinks, and stale numbers in the pages behind every sequence's last token."""
import math

import pytest
import torch

from mxserve.ops import seqmix

pytestmark = pytest.mark.gpu
PAGE = 16


def reference(q, K, V, past, scale, window, keep, sink):
    """q [m, H, dk], K, V [n, G, .] in 64 bits -> [m, H, dv]."""
    m, H, _ = q.shape
    n, G, _ = K.shape
    i, j = past + torch.arange(m)[:, None], torch.arange(n)[None, :]
    seen = j <= i
    if window > 0:
        seen &= (i - j < window) | (j < keep)
    out = torch.empty(m, H, V.shape[2], dtype=torch.float64)
    for h in range(H):
        s = (q[:, h] @ K[:, h * G // H].t() * scale).masked_fill(~seen, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].double().expand(m, 1)], 1)
        out[:, h] = torch.softmax(s, -1)[:, :n] @ V[:, h * G // H]
    return out


def check(gpu, H, G, dk, dv, chunks, window=0, keep=0, sink=False, scale=None, pad=0, seed=0):
    g = torch.Generator().manual_seed(seed)
    scale = dk ** -0.5 if scale is None else scale
    T = sum(m for _, m in chunks)
    nb = [-(-(p + m) // PAGE) for p, m in chunks]
    ids = torch.randperm(sum(nb) + 3, generator=g)
    koff, voff = 8, 8 + G * PAGE * dk + 16
    cache = torch.randn(sum(nb) + 3, voff + G * PAGE * dv + 8, generator=g).bfloat16()
    bt = torch.full((len(chunks), max(nb) + 2), int(ids[-1]), dtype=torch.int32)  # entries past a sequence name some block
    used = 0
    for s, n in enumerate(nb):
        bt[s, :n] = ids[used:used + n]
        used += n
    kv = cache[:, koff:koff + G * PAGE * dk].view(-1, G, PAGE, dk), cache[:, voff:voff + G * PAGE * dv].view(-1, G, PAGE, dv)
    for s, (p, m) in enumerate(chunks):  # what lies behind the last token must not be read into the result
        b, o = bt[s, (p + m - 1) // PAGE], (p + m - 1) % PAGE + 1
        for t in kv:
            t[b, :, o:] = float("nan")
    wide = torch.randn(T, H * dk + pad, generator=g).bfloat16()
    q = wide[:, pad:]
    snk = torch.randn(H, generator=g) * 2 if sink else None
    qsl = torch.tensor([0] + [m for _, m in chunks]).cumsum(0).int()
    lens = torch.tensor([p + m for p, m in chunks], dtype=torch.int32)
    got = seqmix.window_attention(wide.to(gpu)[:, pad:], cache.to(gpu), bt.to(gpu), qsl.to(gpu), lens.to(gpu), koff, voff, H, G, dk, dv,
                                  PAGE, scale, window, keep, max(m for _, m in chunks), sink=None if snk is None else snk.to(gpu))
    got = got.cpu().double().view(T, H, dv)
    for s, (p, m) in enumerate(chunks):
        rows = [t[bt[s, :nb[s]].long()].transpose(1, 2).reshape(-1, G, t.shape[3])[:p + m].double() for t in kv]
        a = int(qsl[s])
        want = reference(q[a:a + m].double().view(m, H, dk), *rows, p, scale, window, keep, snk)
        # the result is rounded to bf16 (2^-9 of it); weights enter with 16 bits (2^-16 each, of values up to max |v|),
        # the exponents are fp32 sums of dk products: 2^-24 dk |s| <= 2^-14 here
        err = (got[a:a + m] - want).abs() - 2.0 ** -8 * want.abs()
        assert float(err.max()) <= 2.0 ** -13 * float(rows[1].abs().max()), (s, p, m, float(err.max()))


@pytest.mark.parametrize("dk,dv", [(16, 16), (64, 64), (48, 80), (96, 32), (128, 128), (112, 16), (32, 112), (64, 128)])
@pytest.mark.parametrize("H,G", [(4, 4), (6, 2), (8, 1)])
def test_head_sizes_and_groups(gpu, dk, dv, H, G):
    check(gpu, H, G, dk, dv, [(0, 70), (5, 33), (130, 16), (40, 1)], sink=True, seed=dk + dv)


@pytest.mark.parametrize("chunk", [(0, 16), (0, 31), (0, 32), (0, 33), (0, 63), (0, 64), (0, 65), (0, 127), (0, 128), (0, 129), (0, 300),
                                   (15, 17), (16, 16), (47, 81), (63, 65), (500, 40)])
@pytest.mark.parametrize("dim", [64, 128])
def test_borders_of_tiles_and_pages(gpu, chunk, dim):
    check(gpu, 4, 1, dim, dim, [chunk, (3, 2)], seed=chunk[0] + chunk[1])
    check(gpu, 3, 3, dim, dim, [chunk, (64, 1)], sink=True, seed=chunk[1])


@pytest.mark.parametrize("window,keep", [(1, 0), (16, 0), (17, 4), (40, 33), (64, 64), (65, 100), (200, 1), (1000, 4)])
@pytest.mark.parametrize("dim", [64, 128])
def test_windows_and_kept_tokens(gpu, window, keep, dim):
    check(gpu, 4, 2, dim, dim, [(0, 150), (333, 40), (77, 20), (250, 1)], window=window, keep=keep, sink=window % 2 == 0, seed=window)


def test_other_strides_and_scales(gpu):
    check(gpu, 4, 2, 64, 64, [(0, 40), (70, 50)], scale=-0.2, pad=4, sink=True)  # rows on 8-byte borders, a negative scale
    check(gpu, 2, 2, 64, 64, [(0, 40)], scale=0.0)
    check(gpu, 2, 1, 128, 64, [(9, 40)], scale=3.0, pad=12)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("H,G,dk,dv", [(4, 4, 64, 64), (8, 2, 64, 48), (2, 2, 128, 96), (4, 1, 96, 128)])
@pytest.mark.parametrize("past,new,window,keep", [(0, 140, 0, 0), (70, 200, 90, 5), (2100, 40, 0, 0)])
def test_a_token_reaches_only_queries_that_see_it(gpu, H, G, dk, dv, past, new, window, keep, bad):
    """A token with a value (or a key) that is no number: queries that do not see it give what they give without it, those that
    do are no numbers in that entry (a key: in all of them)."""
    g = torch.Generator().manual_seed(dk + new)
    n = past + new
    nb = -(-n // PAGE)
    koff, voff = 0, G * PAGE * dk
    cache = torch.randn(nb, voff + G * PAGE * dv, generator=g).bfloat16()
    q = torch.randn(new, H * dk, generator=g).bfloat16()
    bt = torch.arange(nb, dtype=torch.int32).view(1, nb)

    def run(c):
        return seqmix.window_attention(q.to(gpu), c.to(gpu), bt.to(gpu), torch.tensor([0, new], dtype=torch.int32, device=gpu),
                                       torch.tensor([n], dtype=torch.int32, device=gpu), koff, voff, H, G, dk, dv, PAGE, dk ** -0.5,
                                       window, keep, new, max_seq_len=n).cpu().float().view(new, H, dv)

    clean = run(cache)
    i = torch.arange(past, n)
    group = torch.arange(H) // (H // G) == G - 1
    for j in sorted({3, past + 1, past + 17, past + 31, past + 39, n - 30, n - 2}):
        seen = (i >= j) & ((i - j < window) | (j < keep) if window > 0 else torch.tensor(True))
        for off, d, col in ((voff, dv, dv - 1), (koff, dk, 2)):
            c = cache.clone()
            c[j // PAGE, off + ((G - 1) * PAGE + j % PAGE) * d + col] = bad
            y = run(c)
            hit = torch.zeros(new, H, dv, dtype=torch.bool)
            cols = torch.arange(dv) == col if off == voff else torch.ones(dv, dtype=torch.bool)
            hit |= seen[:, None, None] & group[None, :, None] & cols[None, None, :]
            # another tile's maximum may set the reference that weights are scaled by: fp32 roundings, one of bf16 at the end
            err = ((y - clean).abs() - 2.0 ** -7 * clean.abs())[~hit]
            assert not err.numel() or float(err.max()) <= 2.0 ** -12, (j, off == voff, float(err.max()))
            if bad != bad:
                assert not torch.isfinite(y[hit]).any(), (j, off == voff)
