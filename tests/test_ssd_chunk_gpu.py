"""The state space in chunks on the matrix cores against the recurrence in 64 bits: chunk counts around tiles and pieces, heads
of every size that fills a workgroup, states that go on from a slot, and decays from almost none to a full reset per token."""
import pytest
import torch

from mxserve.ops import seqmix

pytestmark = pytest.mark.gpu


def reference(x, B, C, dt, dtb, A, D, state, before, new, G):
    """[T, H, P], [T, G, N] .. in 64 bits, state [S, H, P, N] in place -> y [T, H, P]."""
    H = x.shape[1]
    y, t = torch.empty_like(x), 0
    d = torch.nn.functional.softplus(dt + dtb, threshold=1e9)
    a = torch.exp(-torch.exp(A) * d)
    B, C = B.repeat_interleave(H // G, 1), C.repeat_interleave(H // G, 1)
    for s, n in enumerate(new):
        if before[s] == 0:
            state[s] = 0
        for _ in range(n):
            state[s] = a[t].view(H, 1, 1) * state[s] + (d[t].view(H, 1) * x[t]).unsqueeze(2) * B[t].unsqueeze(1)
            y[t] = (state[s] * C[t].unsqueeze(1)).sum(-1) + D.view(H, 1) * x[t]
            t += 1
    return y


def run(gpu, H, G, N, P, before, new, a_mean, seed=0):
    g = torch.Generator().manual_seed(seed + N + P)
    T, S, off = sum(new), len(new), 4
    x, B, C, dt = (torch.randn(T, n + 8, generator=g).mul(m).bfloat16()[:, 8:] for n, m in ((H * P, 1), (G * N, 0.3), (G * N, 0.3), (H, 1)))
    dtb, A, D = torch.randn(H, generator=g) - 1.0, torch.randn(H, generator=g) * 0.5 + a_mean, torch.randn(H, generator=g)
    pool = torch.randn(S + 1, off + H * P * N + 4, generator=g)
    rows = torch.randperm(S + 1, generator=g)[:S].int()
    qsl = torch.tensor([0] + new).cumsum(0).int()
    lens = torch.tensor([b + n for b, n in zip(before, new)], dtype=torch.int32)
    dev = [t.to(gpu) for t in (dtb, A, D)]
    gp = pool.to(gpu)
    on = lambda t: torch.cat([torch.zeros(T, 8, dtype=t.dtype), t], 1).to(gpu)[:, 8:]  # noqa: E731  (keeps the row stride)
    y = seqmix.ssd_scan(on(x), on(B), on(C), on(dt), *dev, gp, rows.to(gpu), off, qsl.to(gpu), lens.to(gpu), H, G, N, P, max(new))
    st = pool[rows.long(), off:off + H * P * N].double().view(S, H, P, N)
    want = reference(x.double().view(T, H, P), B.double().view(T, G, N), C.double().view(T, G, N), dt.double(), dtb.double(), A.double(),
                     D.double(), st, before, new, G)
    got_st = gp.cpu()[rows.long(), off:off + H * P * N].double().view(S, H, P, N)
    return y.cpu().double().view(T, H, P), want, got_st, st, gp.cpu(), pool, rows


@pytest.mark.parametrize("H,G,N,P", [(2, 1, 128, 64), (8, 2, 64, 32), (2, 2, 128, 128), (4, 2, 64, 64), (8, 1, 128, 32)])
@pytest.mark.parametrize("before,new", [([5], [63]), ([0], [64]), ([0, 9, 0], [64, 65, 1]), ([3], [127]), ([0, 7], [300, 128]),
                                        ([1, 0, 2, 0], [1, 140, 1, 257]), ([0, 4, 4, 4], [16, 15, 17, 33])])
def test_chunks(gpu, H, G, N, P, before, new):
    y, want, st, wst, pool, old, rows = run(gpu, H, G, N, P, before, new, -1.5)
    # fp32 sums over up to 300 tokens and 128 channels: a few hundred roundings of 2^-24, walking at random, on terms of size 30
    torch.testing.assert_close(y, want, rtol=1e-5, atol=1e-4)
    torch.testing.assert_close(st, wst, rtol=1e-5, atol=1e-4)
    spare = [r for r in range(old.shape[0]) if r not in rows.tolist()]
    assert torch.equal(pool[spare], old[spare])  # other slots and the slots' borders stay
    assert torch.equal(pool[:, :4], old[:, :4]) and torch.equal(pool[:, -4:], old[:, -4:])


@pytest.mark.parametrize("before,new", [([5] * 9 + [0], [1] * 9 + [512]), ([0, 3, 1, 8], [1, 300, 511, 2]), ([4, 0], [1024, 1])])
def test_a_spare_piece(gpu, before, new):
    """Counts of pieces that are multiples of 8: an empty one is put behind them."""
    piece, n = seqmix._scan_split(len(new), sum(new), max(new), 2 * 128 * 64, 2, 4 * 64, gpu, spare=True)[:2]
    assert n == -(-max(new) // piece) + 1 and n % 8 == 1
    y, want, st, wst, *_ = run(gpu, 2, 1, 128, 64, before, new, -1.5)
    torch.testing.assert_close(y, want, rtol=1e-5, atol=1e-4)
    torch.testing.assert_close(st, wst, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("H,G,N,P", [(64, 1, 128, 64), (64, 8, 64, 64), (32, 1, 64, 128), (2, 1, 128, 64)])
@pytest.mark.parametrize("before,new", [([0, 9] * 8, [8] * 16), ([3, 0, 1], [31, 30, 31]), ([0, 5] * 4, [9, 12, 1, 31, 8, 20, 2, 17])])
def test_short_chunks_of_many_heads(gpu, H, G, N, P, before, new):
    """Chunks of fewer than 32 tokens: in tiles where there are heads enough, token by token for the last line's two."""
    y, want, st, wst, pool, old, rows = run(gpu, H, G, N, P, before, new, -1.5)
    torch.testing.assert_close(y, want, rtol=1e-5, atol=1e-4)
    torch.testing.assert_close(st, wst, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("a_mean", [-12.0, 3.0, 7.0])
def test_decays(gpu, a_mean):
    """Half lives of a thousand tokens, and resets within a few or one, where the running sum of exponents is in the thousands."""
    y, want, st, wst, *_ = run(gpu, 4, 2, 128, 64, [9, 0], [200, 150], a_mean)
    torch.testing.assert_close(y, want, rtol=1e-5, atol=2e-4)
    torch.testing.assert_close(st, wst, rtol=1e-5, atol=2e-4)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("P,N,new", [(64, 128, [100]), (32, 64, [64, 70]), (128, 128, [700])])
def test_a_token_reaches_no_earlier_one(gpu, P, N, new, bad):
    """A token whose x, B, C or dt is no number: the outputs before it are what they are without it, its own and later ones are
    not numbers either (x: in its column alone)."""
    G, H = 1, max(2, 128 // P)
    g = torch.Generator().manual_seed(P)
    T, S = sum(new), len(new)
    ops = [torch.randn(T, n, generator=g).mul(m).bfloat16() for n, m in ((H * P, 1), (G * N, 0.3), (G * N, 0.3), (H, 1))]
    dev = [t.to(gpu) for t in (torch.randn(H, generator=g) - 1.0, torch.randn(H, generator=g) - 1.5, torch.randn(H, generator=g))]
    qsl = torch.tensor([0] + new).cumsum(0).int()
    lens = torch.tensor(new, dtype=torch.int32)

    def run(ops):
        pool = torch.zeros(S, H * P * N, device=gpu)
        y = seqmix.ssd_scan(*(t.to(gpu) for t in ops), *dev, pool, torch.arange(S, dtype=torch.int32, device=gpu), 0, qsl.to(gpu),
                            lens.to(gpu), H, G, N, P, max(new))
        return y.cpu(), pool.cpu().view(S, H * P, N)

    clean, st0 = run(ops)
    a = int(qsl[S - 1])  # the last sequence's
    for at in (a + 5, a + 31, a + 40, a + 63):
        for which in range(4):
            broken = [t.clone() for t in ops]
            col = P + 3 if which == 0 else 1
            broken[which][at, col] = bad
            y, st = run(broken)
            assert torch.equal(y[:at], clean[:at]), (which, at)
            if which == 0:
                others = torch.arange(H * P) != col
                assert torch.equal(y[:, others], clean[:, others]) and torch.equal(st[:, others], st0[:, others])
                assert not torch.isfinite(y[at:, col]).any() and not torch.isfinite(st[S - 1, col]).any()
            elif which == 2:  # C reads the state and leaves none of it behind
                assert not torch.isfinite(y[at]).any() and torch.equal(st, st0)
                assert torch.equal(y[at + 1:], clean[at + 1:])


@pytest.mark.parametrize("H,G,N,P", [(64, 8, 128, 64), (64, 4, 64, 128)])
@pytest.mark.parametrize("a_mean", [-8.0, -2.0, 0.0, 1.0, 2.0, 3.0, 7.0])
def test_no_further_off_than_token_by_token(gpu, a_mean, H, G, N, P):
    """From half lives of thousands of tokens to a reset by each: the error against 64 bits, as a share of the norm of a head's
    outputs and state and on average over a thousand heads, is no larger than that of the walk by tokens."""
    T = 80
    err = {"chunks": [], "tokens": []}
    for seed in range(16):
        g = torch.Generator(device=gpu).manual_seed(seed)
        rnd = lambda *s: torch.randn(*s, generator=g, device=gpu)  # noqa: E731
        x, B, C, dt = (rnd(T, n).mul(m).bfloat16() for n, m in ((H * P, 1), (G * N, 0.3), (G * N, 0.3), (H, 1)))
        dtb, A, D = rnd(H) - 1.0, rnd(H) * 0.5 + a_mean, rnd(H)
        st = torch.zeros(1, H, P, N, dtype=torch.float64, device=gpu)
        shaped = (t.double().view(T, *s) for t, s in ((x, (H, P)), (B, (G, N)), (C, (G, N)), (dt, (H,))))
        want = reference(*shaped, dtb.double(), A.double(), D.double(), st, [0], [T], G)
        odd = torch.zeros(T, H * P + 1, dtype=x.dtype, device=gpu)
        odd[:, 1:] = x  # no whole 16-byte pieces: token by token
        for way, xs in (("chunks", x), ("tokens", odd[:, 1:])):
            pool = torch.zeros(1, H * P * N, device=gpu)
            ints = [torch.tensor(v, dtype=torch.int32, device=gpu) for v in ([0], [0, T], [T])]
            y = seqmix.ssd_scan(xs, B, C, dt, dtb, A, D, pool, ints[0], 0, ints[1], ints[2], H, G, N, P, T)
            share = lambda v, w, d: (v - w).norm(dim=d) / w.norm(dim=d)  # noqa: E731
            err[way].append(torch.stack([share(y.double().view(T, H, P), want, (0, 2)),
                                         share(pool.double().view(H, -1), st.view(H, -1), 1)], 1))
    chunks, tokens = (torch.cat(e).mean(0).tolist() for e in err.values())
    assert chunks[0] <= tokens[0] and chunks[1] <= tokens[1], (chunks, tokens)


def test_softplus_of_a_sum(gpu):
    """The step sizes over the whole range, shown by a state that starts empty and one token: S = dt x B."""
    H, N, P, T = 2, 64, 64, 64
    worst = 0.0
    for bias in (-30.0, -9.5, -1.0, -1e-3, 0.0, 0.7, 3.3, 25.0):
        dt = torch.linspace(-60, 60, 4001).bfloat16()
        for v in dt[:: 211].tolist():
            x, B = torch.ones(T, H * P).bfloat16(), torch.zeros(T, N).bfloat16()
            B[0, 0] = 1.0
            x[1:] = 0.0
            d = torch.full((T, H), -1e30).bfloat16()
            d[0] = v
            pool = torch.zeros(1, H * P * N, device=gpu)
            ints = [torch.tensor(i, dtype=torch.int32, device=gpu) for i in ([0], [0, T], [T])]
            b = torch.full((H,), bias)
            seqmix.ssd_scan(x.to(gpu), B.to(gpu), B.to(gpu), d.to(gpu), b.to(gpu), torch.zeros(H, device=gpu), torch.zeros(H, device=gpu),
                            pool, ints[0], 0, ints[1], ints[2], H, 1, N, P, T)
            z = torch.tensor(v, dtype=torch.float64) + float(b[0])
            want = float(torch.clamp(z, min=0) + torch.log1p(torch.exp(-z.abs())))
            got = float(pool[0, 0])
            if want > 1e-36:
                worst = max(worst, abs(got - want) / want)
    assert worst <= 2.0 ** -23, worst  # one rounding (2^-24), and as much for what the steps before it keep of theirs
