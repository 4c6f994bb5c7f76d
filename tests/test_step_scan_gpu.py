"""Recurrences of single-token steps: every lane count of a column, columns that do not fill a wave, heads that share keys,
operands off their alignment, fresh and continued states, against the recurrence on the CPU."""
import pytest
import torch

from mxserve.ops import seqmix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,dk,dv,pad", [(2, 1, 32, 8, 8), (3, 3, 64, 40, 4), (4, 2, 128, 64, 3), (2, 2, 128, 128, 0), (1, 1, 256, 24, 8),
                                           (5, 5, 128, 1, 1), (2, 2, 64, 33, 8)])
@pytest.mark.parametrize("kind", ["state", "delta", "linear"])
def test_single_tokens(gpu, dt, H, G, dk, dv, pad, kind):
    if kind == "linear" and G != H:
        pytest.skip("a key head for every head")
    g = torch.Generator().manual_seed(H * dk + dv)
    S, off = 5, 8
    mk = lambda n, t=dt: torch.randn(S, n + pad, generator=g).to(t)[:, pad:]  # noqa: E731
    q, k, v = mk(G * dk), mk(G * dk), mk(H * dv)
    pool = torch.randn(S + 2, off + H * dk * dv + 4, generator=g)
    rows = torch.randperm(S + 2, generator=g)[:S].int()
    qsl, lens = torch.arange(S + 1).int(), torch.tensor([1, 7, 1, 30, 2], dtype=torch.int32)
    A, D = torch.randn(H, generator=g) * 0.5 - 1.0, torch.randn(H, generator=g)
    b, tb = mk(H), torch.randn(H, generator=g)
    a, cb, loga = mk(H * dk), torch.randn(H * dk, generator=g), -torch.rand(S, H * dk + pad, generator=g)[:, pad:]
    res = []
    for dev in ("cpu", gpu):
        on = lambda t: t if dev == "cpu" else torch.cat([torch.zeros(S, pad, dtype=t.dtype), t], 1).to(dev)[:, pad:]  # noqa: E731
        pl = pool.clone().to(dev)
        tail = (pl, rows.to(dev), off, qsl.to(dev), lens.to(dev), H)
        if kind == "state":
            y = seqmix.ssd_scan(on(v), on(k), on(q), on(b), tb.to(dev), A.to(dev), D.to(dev), *tail, G, dk, dv, 1)
        elif kind == "delta":
            y = seqmix.delta_scan(on(q), on(k), on(v), on(b), on(a), cb.to(dev), A.to(dev), *tail, G, dk, dv, dk ** -0.5, max_query_len=1)
        else:
            y = seqmix.gla_scan(on(q), on(k), on(v), on(loga), *tail, dk, dv, dk ** -0.5, 1)
        res.append((y.cpu(), pl.cpu()))
    for x, y in zip(*res):  # sums of up to 256 fp32 products of size one either way
        torch.testing.assert_close(y, x, rtol=1e-5, atol=3e-5)
