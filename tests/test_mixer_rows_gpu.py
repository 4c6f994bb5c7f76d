"""The row-wise mixer kernels' wide forms (whole, aligned 16-byte pieces) against the PyTorch forms, at the sizes where
they begin and end."""
import pytest
import torch

from mxserve.ops import seqmix

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]


def tol(dt):  # fp32: sums of up to 8,192 terms in another order; bf16: one rounding of the result, and a tie that falls the other way
    return dict(rtol=1e-5, atol=2e-5) if dt == torch.float32 else dict(rtol=2.0 ** -7, atol=2.0 ** -8)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("T,W", [(1, 8), (3, 504), (5, 1024), (2, 2040), (64, 2048), (3, 2056), (2, 4096), (2, 8192), (2, 8200)])
def test_resid_update_rows(gpu, dt, T, W):
    g = torch.Generator().manual_seed(W)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x, a, b = rnd(T, W), rnd(T, W + 24).to(dt)[:, 8:8 + W], rnd(T, W).to(dt)
    wa, wb, nw, bias = (rnd(W).to(dt) for _ in range(4))
    for kw in (dict(a=a, norm_w=nw, a_scale=0.7, w_offset=1.0), dict(a=a, wa=wa, norm_w=nw), dict(a=None, norm_w=nw),
               dict(a=a, wa=wa, b=b, wb=wb, bias=bias, norm_w=nw), dict(a=a, bias=bias, assign=True, norm_w=nw),
               dict(a=a, wa=wa, wa_offset=1.0, cast_dtype=dt), dict(a=a)):
        xa = kw.pop("a")
        xc, xg = x.clone(), x.to(gpu)
        want = seqmix.resid_update(xc, xa, 1e-5, out_dtype=dt, **kw)
        got = seqmix.resid_update(xg, None if xa is None else xa.to(gpu), 1e-5, out_dtype=dt,
                                  **{k: v.to(gpu) if torch.is_tensor(v) else v for k, v in kw.items()})
        torch.testing.assert_close(xg.cpu(), xc, rtol=1e-5, atol=2e-5)
        assert (got is None) == (want is None)
        if want is not None:
            torch.testing.assert_close(got.cpu().float(), want.float(), **tol(dt))


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("T,V,pad", [(1, 8, 0), (3, 2047, 1), (2, 2048, 0), (2, 2056, 8), (65, 32000, 0), (1, 5001, 3)])
def test_softcap_rows(gpu, dt, T, V, pad):
    x = (20 * torch.randn(T, V + pad, generator=torch.Generator().manual_seed(V))).to(dt)[:, pad:]
    for cap in (0.0, 12.5):
        torch.testing.assert_close(seqmix.softcap(x.to(gpu), cap).cpu(), seqmix.softcap(x, cap), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("H,G,dk,dv,nf,nvf", [(4, 2, 8, 8, 2, 0), (6, 3, 16, 24, 8, 12), (32, 8, 64, 64, 32, 0), (5, 5, 64, 40, 9, 20),
                                              (2, 1, 512, 16, 256, 8), (3, 1, 24, 16, 12, 0), (2, 2, 1024, 8, 4, 4)])
@pytest.mark.parametrize("norm", [False, True])
def test_rotary_rows(gpu, dt, H, G, dk, dv, nf, nvf, norm):
    g = torch.Generator().manual_seed(H * dk + nf)
    T, bs, koff = 5, 16, 16
    voff = koff + G * bs * dk
    qkv = torch.randn(T, H * dk + G * (dk + dv), generator=g).to(dt)
    cache = torch.randn(3, voff + G * bs * dv + 8, generator=g).to(dt)
    pos, slots = torch.tensor([0, 7, 1000, 33, 5]), torch.tensor([40, 3, -1, 17, 0])
    fr, vf = torch.rand(nf, generator=g), torch.rand(nvf, generator=g) if nvf else None
    qn, kn = ((torch.randn(dk, generator=g)).to(dt) if norm else None for _ in range(2))
    res = {}
    for dev in ("cpu", gpu):
        x, c = qkv.clone().to(dev), cache.clone().to(dev)
        on = lambda t: None if t is None else t.to(dev)  # noqa: E731
        q, k, v = x.split([H * dk, G * dk, G * dv], dim=1)
        seqmix.rope_qkv_cache(q, k, v, on(pos), on(slots), c, koff, voff, H, G, dk, dv, bs, on(fr), on(qn), on(kn), 1e-5, on(vf))
        y = torch.zeros(T, H * dk + 8, dtype=dt, device=dev)
        seqmix.rope_rows(q, on(pos), H, dk, on(fr), -1.0, 0.7, y[:, 8:])
        res[str(dev)] = (x.cpu(), c.cpu(), y.cpu())
    for a, b in zip(*res.values()):
        # angles of up to 1,000 turned in fp32: 2^-24 * 1000 of a turn either way
        torch.testing.assert_close(a.float(), b.float(), **(dict(rtol=1e-4, atol=4e-4) if dt == torch.float32 else dict(rtol=2.0 ** -6, atol=2.0 ** -6)))


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("H,G,dk,dv,nf,nvf", [(6, 3, 16, 24, 8, 12), (32, 8, 64, 64, 32, 0), (5, 5, 64, 40, 9, 20), (128, 8, 128, 128, 64, 0),
                                              (3, 2, 512, 16, 256, 8), (4, 2, 64, 64, 32, 0), (16, 4, 8, 72, 4, 0)])
@pytest.mark.parametrize("norm", [False, True])
def test_rotary_of_many_rows(gpu, dt, H, G, dk, dv, nf, nvf, norm):
    """Enough tokens and heads for a lane per piece: a token's pieces in one workgroup and over several."""
    g = torch.Generator().manual_seed(H * dk + nf)
    bs, koff = 16, 16
    voff = koff + G * bs * dk
    for T in (255, 257) if H * dk >= 1024 else (800,):
        qkv = torch.randn(T, H * dk + G * (dk + dv), generator=g).to(dt)
        cache = torch.randn(T // bs + 1, voff + G * bs * dv + 8, generator=g).to(dt)
        pos, slots = torch.arange(T) % 97, torch.randperm(T, generator=g)
        slots[3] = -1
        fr, vf = torch.rand(nf, generator=g), torch.rand(nvf, generator=g) if nvf else None
        qn, kn = ((torch.randn(dk, generator=g)).to(dt) if norm else None for _ in range(2))
        res = {}
        for dev in ("cpu", gpu):
            x, c = qkv.clone().to(dev), cache.clone().to(dev)
            on = lambda t: None if t is None else t.to(dev)  # noqa: E731
            q, k, v = x.split([H * dk, G * dk, G * dv], dim=1)
            seqmix.rope_qkv_cache(q, k, v, on(pos), on(slots), c, koff, voff, H, G, dk, dv, bs, on(fr), on(qn), on(kn), 1e-5, on(vf))
            y = torch.zeros(T, H * dk + 8, dtype=dt, device=dev)
            seqmix.rope_rows(q, on(pos), H, dk, on(fr), -1.0, 0.7, y[:, 8:])
            res[str(dev)] = (x.cpu(), c.cpu(), y.cpu())
        for a, b in zip(*res.values()):
            # as above; a rotation of normed entries of up to 5 once more
            torch.testing.assert_close(a.float(), b.float(), **(dict(rtol=1e-4, atol=4e-4) if dt == torch.float32 else dict(rtol=2.0 ** -6, atol=2.0 ** -5)))


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("C", [8, 72, 2056])
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("lens", [[1], [8], [9], [1, 1, 1, 1, 1, 1, 1, 1, 1], [3, 4, 1, 2, 17], [7, 1, 8, 16]])
def test_convolution_rows(gpu, dt, C, taps, lens):
    g = torch.Generator().manual_seed(C + taps + len(lens))
    T, S = sum(lens), len(lens)
    x = torch.randn(T, C + 16, generator=g).to(dt)[:, 16:]
    w, b = torch.randn(taps, C, generator=g).to(dt), torch.randn(C, generator=g).to(dt)
    state = torch.randn(S + 2, 8 + max(taps - 1, 1) * C, generator=g)
    rows = torch.randperm(S + 2, generator=g)[:S].int()
    qsl = torch.tensor([0] + lens).cumsum(0).int()
    seq = torch.tensor([n + (0 if i % 2 else 9) for i, n in enumerate(lens)], dtype=torch.int32)
    for single in ([0, 1] if max(lens) == 1 else [0]):
        sc, sg = state.clone(), state.to(gpu)
        want = seqmix.causal_conv(x, w, b, sc, rows, 8, qsl, seq, True, 1 if single else max(lens))
        got = seqmix.causal_conv(x.to(gpu), w.to(gpu), b.to(gpu), sg, rows.to(gpu), 8, qsl.to(gpu), seq.to(gpu), True,
                                 1 if single else max(lens))
        torch.testing.assert_close(got.cpu().float(), want.float(), **tol(dt))
        torch.testing.assert_close(sg.cpu(), sc, rtol=0, atol=0)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("lens", [[3, 4, 1, 2, 17, 9], [1], [2001], [0, 7, 1, 8, 0, 16]])
@pytest.mark.parametrize("more", [0, 3])
def test_convolution_of_many_rows(gpu, dt, taps, lens, more):
    """Enough rows and channels for four rows a thread (and, in the last line, just too few for it): groups of four across
    borders of sequences, also of empty ones, and rows past the last sequence."""
    g = torch.Generator().manual_seed(taps + len(lens) + more)
    for C, least in ((2056, 1840 if dt == torch.bfloat16 else 920), (2056, 1770 if dt == torch.bfloat16 else 880)):
        n = lens * max(1, -(-least // sum(lens)))
        T, S = sum(n) + more, len(n)
        x, b = torch.randn(T, C + 16, generator=g).to(dt)[:, 16:], torch.randn(C, generator=g).to(dt)
        w = torch.randn(taps, C, generator=g).to(dt)
        state = torch.randn(S + 2, 8 + (taps - 1) * C, generator=g)
        rows = torch.randperm(S + 2, generator=g)[:S].int()
        qsl = torch.tensor([0] + n).cumsum(0).int()
        seq = torch.tensor([m + (0 if i % 2 else 9) for i, m in enumerate(n)], dtype=torch.int32)
        sg = state.to(gpu)
        got = seqmix.causal_conv(x.to(gpu), w.to(gpu), b.to(gpu), sg, rows.to(gpu), 8, qsl.to(gpu), seq.to(gpu), True, max(2, max(n)))
        sc, end, last = state.clone(), qsl.clone(), S - 1
        seqmix.causal_conv(x[:T - more], w, b, sc, rows, 8, qsl, seq, True, max(n))
        torch.testing.assert_close(sg.cpu(), sc, rtol=0, atol=0)
        if more:  # they go on as the last sequence's
            end[S] = T
            seq = seq + torch.tensor([0] * last + [more], dtype=torch.int32)
        want = seqmix.causal_conv(x, w, b, state.clone(), rows, 8, end, seq, True, T)
        torch.testing.assert_close(got.cpu().float(), want.float(), **tol(dt))


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("taps", [2, 4])
@pytest.mark.parametrize("lens", [[3], [5, 2], [4, 9, 0], [1, 1, 1]])
@pytest.mark.parametrize("more", [1, 2, 7])
def test_convolution_rows_past_the_last_sequence(gpu, dt, taps, lens, more):
    """x holds more rows than the sequences have: those go on as the last sequence's, and no sequence behind it is looked up."""
    C, T, S = 72, sum(lens) + more, len(lens)
    g = torch.Generator().manual_seed(T)
    x, w = torch.randn(T, C, generator=g).to(dt), torch.randn(taps, C, generator=g).to(dt)
    state = torch.randn(S, (taps - 1) * C, generator=g)
    rows = torch.arange(S, dtype=torch.int32)
    qsl = torch.tensor([0] + lens).cumsum(0).int()
    seq = torch.tensor([n + 9 for n in lens], dtype=torch.int32)
    on = [t.to(gpu) for t in (rows, qsl, seq)]
    got = seqmix.causal_conv(x.to(gpu), w.to(gpu), None, state.to(gpu), on[0], 0, on[1], on[2], True, max(max(lens), 2)).cpu()
    longer = qsl.clone()
    longer[S] = T
    want = seqmix.causal_conv(x, w, None, state.clone(), rows, 0, longer, seq + torch.tensor([0] * (S - 1) + [more]), True, T)
    torch.testing.assert_close(got.float(), want.float(), **tol(dt))


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("N,groups,wn", [(16, 2, 16), (128, 16, 8), (384, 8, 48), (384, 3, 384), (2048, 16, 128), (4096, 8, 4096), (1024, 1, 1024),
                                         (4096, 1, 4096), (8192, 2, 8192), (6144, 2, 6144)])
def test_gated_norm_rows(gpu, dt, N, groups, wn):
    g = torch.Generator().manual_seed(N + groups)
    o, z, w = torch.randn(3, N, generator=g), torch.randn(3, N + 8, generator=g).to(dt)[:, 8:], torch.randn(wn, generator=g).to(dt)
    for act, first in (("silu", True), ("sigmoid", False), ("silu", False)):
        want, got = torch.zeros(3, N + 16, dtype=dt), torch.zeros(3, N + 16, dtype=dt, device=gpu)
        seqmix.gated_norm(o, z, w, 1e-5, groups, act, first, dt, 0.5, want[:, 16:])
        seqmix.gated_norm(o.to(gpu), z.to(gpu), w.to(gpu), 1e-5, groups, act, first, dt, 0.5, got[:, 16:])
        torch.testing.assert_close(got.cpu().float(), want.float(), **tol(dt))
