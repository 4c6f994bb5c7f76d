"""Chunk attention whose long walks are split into stretches against the same chunks in one walk: walks around the length from
which they split, short chunks and single tokens beside them, windows, sinks, and keys that every head expanded."""
import pytest
import torch

from mxserve.ops import seqmix

pytestmark = pytest.mark.gpu
# two sums of the same fp32 weights in another order, each rounded to bf16
TOL = dict(rtol=2.0 ** -7, atol=2.0 ** -10)
CHUNKS = [[(1000, 40)], [(700, 67), (701, 67), (1500, 1), (0, 17)], [(735, 33), (2000, 16), (10, 1), (0, 100)]]


@pytest.mark.parametrize("H,G,dk,dv", [(8, 2, 64, 64), (4, 4, 128, 128), (6, 2, 80, 48)])
@pytest.mark.parametrize("chunks", CHUNKS)
@pytest.mark.parametrize("window,keep", [(0, 0), (1100, 20), (900, 200)])
def test_paged(gpu, H, G, dk, dv, chunks, window, keep):
    g = torch.Generator().manual_seed(H + len(chunks))
    nb = [-(-(p + m) // 16) for p, m in chunks]
    T = sum(m for _, m in chunks)
    cache = torch.randn(sum(nb), G * 16 * (dk + dv), generator=g).bfloat16().to(gpu)
    bt = torch.zeros(len(chunks), max(nb), dtype=torch.int32)
    ids, u = torch.randperm(sum(nb), generator=g), 0
    for i, n in enumerate(nb):
        bt[i, :n] = ids[u:u + n]
        u += n
    q, sink = torch.randn(T, H * dk, generator=g).bfloat16().to(gpu), torch.randn(H, generator=g).to(gpu)
    qsl = torch.tensor([0] + [m for _, m in chunks]).cumsum(0).int().to(gpu)
    lens = torch.tensor([p + m for p, m in chunks], dtype=torch.int32)
    run = lambda span: seqmix.window_attention(q, cache, bt.to(gpu), qsl, lens.to(gpu), 0, G * 16 * dk, H, G, dk, dv, 16, dk ** -0.5,  # noqa: E731
                                               window, keep, max(m for _, m in chunks), sink, max_seq_len=span)
    torch.testing.assert_close(run(int(lens.max())).float(), run(0).float(), **TOL)


@pytest.mark.parametrize("chunks", CHUNKS)
@pytest.mark.parametrize("window", [0, 1100])
def test_expanded(gpu, chunks, window):
    g = torch.Generator().manual_seed(len(chunks))
    H, dn, dr, dv, rank = 4, 128, 64, 128, 64
    T, n = sum(m for _, m in chunks), sum(p + m for p, m in chunks)
    q, kv, rows = (torch.randn(*s, generator=g).bfloat16().to(gpu) for s in ((T, H * (dn + dr)), (n, H * (dn + dv)), (n, rank + dr)))
    base = torch.tensor([0] + [p + m for p, m in chunks]).cumsum(0)[:-1].int().to(gpu)
    qsl = torch.tensor([0] + [m for _, m in chunks]).cumsum(0).int().to(gpu)
    lens, sink = torch.tensor([p + m for p, m in chunks], dtype=torch.int32), torch.randn(H, generator=g).to(gpu)
    run = lambda span: seqmix.expanded_attention(q, kv, rows, base, qsl, lens.to(gpu), H, dn, dr, dv, 0.07,  # noqa: E731
                                                 max(m for _, m in chunks), sink, window, max_seq_len=span)
    torch.testing.assert_close(run(int(lens.max())).float(), run(0).float(), **TOL)
