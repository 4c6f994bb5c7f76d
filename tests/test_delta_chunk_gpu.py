"""The delta rule in chunks of 32 tokens against the recurrence in 64 bits: token counts around chunks, several sequences with
states that go on from a slot, shared and own key heads, head sizes, and decays from almost none to a reset per token."""
import pytest
import torch

from mxserve.ops import seqmix

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def chunks_for_all(monkeypatch):
    monkeypatch.setattr(seqmix, "DELTA_CHUNK_TOKENS", 0)
    monkeypatch.setattr(seqmix, "DELTA_CHUNK_TOKENS_PER_SEQ", 0)


def reference(q, k, v, beta, a, dtb, A, state, before, new, H, G, dk, dv, scale, eps=1e-6):
    T = q.shape[0]
    unit = lambda t: (t.view(T, G, dk) * torch.rsqrt(t.view(T, G, dk).pow(2).sum(-1, keepdim=True) + eps)).repeat_interleave(H // G, 1)  # noqa: E731
    q, k, v, b = unit(q) * scale, unit(k), v.view(T, H, dv), torch.sigmoid(beta)
    g = torch.exp(-torch.exp(A).view(1, H, 1) * torch.nn.functional.softplus(a + dtb, threshold=1e9).view(T, H, dk))
    out, t = torch.empty(T, H, dv, dtype=torch.float64), 0
    for s, n in enumerate(new):
        if before[s] == 0:
            state[s] = 0
        for _ in range(n):
            st = state[s] * g[t].unsqueeze(1)
            u = b[t].view(H, 1) * (v[t] - (st * k[t].unsqueeze(1)).sum(-1))
            state[s] = st + u.unsqueeze(2) * k[t].unsqueeze(1)
            out[t] = (state[s] * q[t].unsqueeze(1)).sum(-1)
            t += 1
    return out.view(T, H * dv)


def run(gpu, H, G, dk, dv, before, new, a_mean=-2.0, shift=8, seed=0):
    g = torch.Generator().manual_seed(seed + H + dk)
    T, S, off = sum(new), len(new), 4
    q, k, v, b, a = (torch.randn(T, n + 8, generator=g).bfloat16() for n in (G * dk, G * dk, H * dv, H, H * dk))
    view = lambda t: t[:, shift:t.shape[1] - 8 + shift]  # noqa: E731
    dtb, A = torch.randn(H * dk, generator=g) - 1.0, torch.randn(H, generator=g) * 0.5 + a_mean
    pool = torch.randn(S + 1, off + H * dk * dv + 4, generator=g)
    rows = torch.randperm(S + 1, generator=g)[:S].int()
    qsl = torch.tensor([0] + new).cumsum(0).int()
    lens = torch.tensor([x + n for x, n in zip(before, new)], dtype=torch.int32)
    gp = pool.to(gpu)
    got = seqmix.delta_scan(*(view(t.to(gpu)) for t in (q, k, v, b, a)), dtb.to(gpu), A.to(gpu), gp, rows.to(gpu), off, qsl.to(gpu),
                            lens.to(gpu), H, G, dk, dv, dk ** -0.5, max_query_len=max(new))
    st = pool[rows.long(), off:off + H * dk * dv].double().view(S, H, dv, dk)
    want = reference(*(view(t).double() for t in (q, k, v, b, a)), dtb.double(), A.double(), st, before, new, H, G, dk, dv, dk ** -0.5)
    gst = gp.cpu()[rows.long(), off:off + H * dk * dv].double().view(S, H, dv, dk)
    return got.cpu().double(), want, gst, st, gp.cpu(), pool, rows


@pytest.mark.parametrize("H,G,dk,dv,shift", [(2, 2, 128, 128, 8), (4, 2, 64, 64, 8), (2, 1, 128, 16, 3), (2, 2, 64, 112, 4), (1, 1, 128, 96, 0)])
@pytest.mark.parametrize("before,new", [([0], [8]), ([5], [31]), ([0], [32]), ([0, 9, 0], [33, 64, 1]), ([3], [127]), ([0, 7], [300, 128]),
                                        ([1, 0, 2, 0], [1, 140, 1, 257])])
def test_chunks(gpu, H, G, dk, dv, shift, before, new):
    y, want, st, wst, pool, old, rows = run(gpu, H, G, dk, dv, before, new, shift=shift)
    # fp32 sums over 128 channels and up to 300 tokens whose writes depend on each other: a thousand roundings of 2^-24 at random
    torch.testing.assert_close(y, want, rtol=1e-5, atol=5e-5)
    torch.testing.assert_close(st, wst, rtol=1e-5, atol=5e-5)
    spare = [r for r in range(old.shape[0]) if r not in rows.tolist()]
    assert torch.equal(pool[spare], old[spare])
    assert torch.equal(pool[:, :4], old[:, :4]) and torch.equal(pool[:, -4:], old[:, -4:])


@pytest.mark.parametrize("a_mean", [-12.0, 2.0, 6.0])
def test_decays(gpu, a_mean):
    y, want, st, wst, *_ = run(gpu, 2, 1, 128, 64, [9, 0], [200, 150], a_mean)
    torch.testing.assert_close(y, want, rtol=1e-5, atol=1e-4)
    torch.testing.assert_close(st, wst, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("a_mean", [-8.0, -2.0, 0.0, 1.0, 2.0, 4.0, 6.0])
def test_no_further_off_than_token_by_token(gpu, monkeypatch, a_mean, dim):
    """From half lives of a thousand tokens to resets by each: the chunks' error against 64 bits, as a share of the norm of a head's
    outputs and state and on average over a thousand heads, is no larger than that of the walk by tokens."""
    H, T = 64, 80
    err = {0: [], 1 << 40: []}
    for seed in range(16):
        g = torch.Generator(device=gpu).manual_seed(seed)
        rnd = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
        q, k, v, b, a = (rnd(T, n).bfloat16() for n in (H * dim, H * dim, H * dim, H, H * dim))
        dtb, A = rnd(H * dim) - 1.0, rnd(H) * 0.5 + a_mean
        st = torch.zeros(1, H, dim, dim, dtype=torch.float64, device=gpu)
        with torch.device(gpu):
            want = reference(*(t.double() for t in (q, k, v, b, a, dtb, A)), st, [0], [T], H, H, dim, dim, dim ** -0.5)
        for least, e in err.items():
            monkeypatch.setattr(seqmix, "DELTA_CHUNK_TOKENS", least)
            pool = torch.zeros(1, H * dim * dim, device=gpu)
            ints = [torch.tensor(x, dtype=torch.int32, device=gpu) for x in ([0], [0, T], [T])]
            y = seqmix.delta_scan(q, k, v, b, a, dtb, A, pool, ints[0], 0, ints[1], ints[2], H, H, dim, dim, dim ** -0.5, max_query_len=T)
            share = lambda x, w, d: (x - w).norm(dim=d) / w.norm(dim=d)  # noqa: E731
            e.append(torch.stack([share(y.double().view(T, H, dim), want.view(T, H, dim), (0, 2)),
                                  share(pool.double().view(H, -1), st.view(H, -1), 1)], 1))
    chunks, tokens = (torch.cat(e).mean(0).tolist() for e in err.values())
    assert chunks[0] <= tokens[0] and chunks[1] <= tokens[1], (chunks, tokens)
