"""Attention of single rows on the matrix cores against softmax in 64 bits: groups of query heads under, at and over the 16
columns of a product, head sizes that fill a product and that ride in zeroed entries, key counts around the tiles and the
waves' turns, windows with kept first tokens, sinks, value rows that lie apart, block sizes, and steps whose few rows are split
over workgroups."""
import math

import pytest
import torch

from mxserve.ops import seqmix

pytestmark = pytest.mark.gpu


def check(gpu, H, G, dk, dv, chunks, window=0, keep=0, sink=False, bs=16, vs=0, blocks=0):
    g = torch.Generator().manual_seed(H * 131 + dk + len(chunks))
    T, S = sum(m for _, m in chunks), len(chunks)
    nb = [-(-(p + m) // bs) for p, m in chunks]
    ids = torch.randperm(sum(nb) + 3, generator=g)
    vw = vs or dv
    koff, voff = 8, 8 + G * bs * dk + 16
    cache = torch.randn(sum(nb) + 3, voff + G * bs * vw + 8, generator=g).bfloat16()
    bt = torch.full((S, max(max(nb) + 2, blocks)), int(ids[-1]), dtype=torch.int32)
    used = 0
    for s, n in enumerate(nb):
        bt[s, :n] = ids[used:used + n]
        used += n
    K = cache[:, koff:koff + G * bs * dk].view(-1, G, bs, dk)
    V = cache[:, voff:voff + G * bs * vw].view(-1, G, bs, vw)
    for s, (p, m) in enumerate(chunks):  # what lies behind the last token must not be read into the result
        b, o = bt[s, (p + m - 1) // bs], (p + m - 1) % bs + 1
        K[b, :, o:] = float("nan")
        V[b, :, o:] = float("nan")
    q = torch.randn(T, H * dk + 8, generator=g).bfloat16()
    snk = torch.randn(H, generator=g) * 2 if sink else None
    qsl = torch.tensor([0] + [m for _, m in chunks]).cumsum(0).int()
    lens = torch.tensor([p + m for p, m in chunks], dtype=torch.int32)
    got = seqmix.window_attention(q.to(gpu)[:, 8:], cache.to(gpu), bt.to(gpu), qsl.to(gpu), lens.to(gpu), koff, voff, H, G, dk, dv, bs,
                                  dk ** -0.5, window, keep, max(m for _, m in chunks), None if snk is None else snk.to(gpu), vs)
    got = got.cpu().double().view(T, H, dv)
    for s, (p, m) in enumerate(chunks):
        Ks, Vs = (t[bt[s, :nb[s]].long()].transpose(1, 2).reshape(-1, G, t.shape[3])[:p + m].double() for t in (K, V))
        for i in range(m):
            j, pos = torch.arange(p + m), p + i
            seen = (j <= pos) & ((pos - j < window) | (j < keep) if window > 0 else torch.ones_like(j, dtype=torch.bool))
            qi = q[int(qsl[s]) + i, 8:].double().view(H, dk)
            for h in range(H):
                sc = (Ks[:, h * G // H] @ qi[h] * dk ** -0.5).masked_fill(~seen, -math.inf)
                if sink:
                    sc = torch.cat([sc, snk[h].double()[None]])
                want = torch.softmax(sc, 0)[:p + m] @ Vs[:, h * G // H, :dv]
                # half a bf16 step of the result; scores in fp32 sums move a weight by some 2^-20 of itself
                torch.testing.assert_close(got[int(qsl[s]) + i, h], want, rtol=2.0 ** -8, atol=2.0 ** -15)


@pytest.mark.parametrize("H,G,dk,dv", [(2, 2, 64, 64), (8, 2, 64, 64), (16, 1, 64, 64), (17, 1, 32, 64), (40, 2, 8, 8), (6, 2, 96, 40),
                                       (4, 2, 128, 128), (32, 1, 128, 64), (3, 1, 72, 104)])
@pytest.mark.parametrize("past", [0, 1, 14, 15, 16, 31, 32, 255, 256, 300, 1030])
def test_rows(gpu, H, G, dk, dv, past):
    check(gpu, H, G, dk, dv, [(past, 1), (past // 2, 2), (3, 1)], sink=past % 2 == 0)


@pytest.mark.parametrize("window,keep", [(1, 0), (5, 3), (32, 0), (100, 40), (256, 4), (1000, 0)])
@pytest.mark.parametrize("dk", [64, 128])
def test_windows(gpu, window, keep, dk):
    check(gpu, 8, 2, dk, dk, [(0, 1), (40, 3), (99, 1), (700, 1)], window, keep, sink=True)


@pytest.mark.parametrize("bs,vs", [(8, 0), (32, 0), (16, 96), (64, 128)])
def test_blocks_and_value_rows(gpu, bs, vs):
    check(gpu, 4, 1, 64, 48, [(0, 1), (77, 1), (500, 2)], bs=bs, vs=vs)


@pytest.mark.parametrize("rows", [1, 3, 16, 40])
@pytest.mark.parametrize("sink", [False, True])
def test_split_rows(gpu, rows, sink):
    check(gpu, 6, 3, 64, 64, [(37 * i % 900 + (900 if i == 0 else 0), 1) for i in range(rows)], sink=sink, blocks=300)
    check(gpu, 6, 3, 64, 64, [(37 * i % 900, 1) for i in range(rows)], 600, 10, sink=sink, blocks=300)


@pytest.mark.parametrize("H,G,dk,dv", [(16, 16, 64, 64), (40, 20, 32, 48), (16, 16, 128, 128), (16, 16, 96, 16)])
@pytest.mark.parametrize("chunks", [[(0, 5)] * 16, [(20, 2)] * 20, [(0, 15), (33, 1), (100, 2), (62, 3)] * 3, [(2040, 9)] + [(7, 4)] * 10])
def test_short_chunks_of_many_rows(gpu, H, G, dk, dv, chunks):
    """More rows and heads than the rows' form takes: chunks of fewer than 16 rows by tiles, weights with all their bits."""
    check(gpu, H, G, dk, dv, chunks)
    check(gpu, H, G, dk, dv, chunks, window=9, keep=3, sink=True)


@pytest.mark.parametrize("chunks", [[(0, 16)], [(0, 31), (5, 17)], [(33, 31)], [(40, 25)]])
def test_chunks_with_nothing_to_walk(gpu, chunks):
    """Chunks of 16 to 31 rows and at most 64 keys, in the rows' form, and just beyond."""
    check(gpu, 8, 2, 64, 64, chunks, sink=True)
