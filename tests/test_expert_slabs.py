"""Routed experts in slabs: the batched products over slabs against one product pair per expert, for even, skewed and empty
choices; the kernels that fill the slabs and clip the projections, at rows of whole pieces and at others."""
import pytest
import torch

from mxserve.models.feedforward import CappedExpert, RoutedExperts
from mxserve.ops import seqmix

DTYPES = [torch.float32, torch.bfloat16]


def block(E, top, W, ff, dev, dt, weigh, seed):
    g = torch.Generator().manual_seed(seed)
    f = RoutedExperts("", W, E, top, ff, 7.0, CappedExpert("shared.", W, ff, 7.0), weigh=weigh)
    w = {n: (torch.randn(s, generator=g) * s[-1] ** -0.5).to(dt).to(dev) for n, s in f.shapes().items()}
    f.finish_weights(w)
    return f, w, g


def both_routes(dev, dt, E, top, W, ff, T, weigh, skew):
    f, w, g = block(E, top, W, ff, dev, dt, weigh, T + E)
    h = torch.randn(T, W, generator=g).to(dt).to(dev)
    f.BATCHED_MAX_TOKENS = f.BATCHED_MAX_ROWS = 0
    if skew:  # every token's first choices are the same experts
        route = f.route
        f.route = lambda h, w: (route(h, w)[0], torch.arange(top, dtype=torch.int32, device=dev).repeat(T, 1), None)
    out = {}
    for gain in (0.0, 1e9):
        f.SLAB_GAIN_S = gain
        out[gain] = f.forward(h, w).float().cpu()
    # the same rows through products of other shapes: fp32 sums in another order, one rounding to dt after each product
    tol = dict(rtol=1e-4, atol=1e-4) if dt == torch.float32 else dict(rtol=2.0 ** -6, atol=2.0 ** -6)
    torch.testing.assert_close(out[0.0], out[1e9], **tol)


@pytest.mark.parametrize("weigh", ["input", "output"])
@pytest.mark.parametrize("E,top,T,skew", [(4, 2, 33, False), (6, 1, 40, False), (5, 5, 7, False), (4, 2, 33, True), (3, 1, 1, False)])
def test_routes_agree(E, top, T, skew, weigh):
    both_routes(torch.device("cpu"), torch.float32, E, top, 24, 16, T, weigh, skew)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("E,top,W,ff,T,skew", [(8, 2, 256, 128, 300, False), (8, 2, 100, 36, 77, False), (8, 2, 256, 128, 300, True),
                                               (3, 3, 64, 64, 65, False), (16, 4, 128, 64, 1000, False)])
@pytest.mark.parametrize("weigh", ["input", "output"])
def test_routes_agree_gpu(gpu, dt, E, top, W, ff, T, skew, weigh):
    both_routes(gpu, dt, E, top, W, ff, T, weigh, skew)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("W,pad", [(8, 0), (2048, 8), (2048, 1), (37, 0), (4, 4)])
def test_slabs(gpu, dt, W, pad):
    g = torch.Generator().manual_seed(W)
    T, k, E = 50, 3, 7
    h = torch.randn(T, W + pad, generator=g).to(dt)[:, pad:]
    ids = torch.stack([torch.randperm(E - 1, generator=g)[:k] for _ in range(T)]).int()  # the last expert gets nothing
    wt = torch.rand(T, k, generator=g)
    offs, inv = seqmix.expert_align(ids.to(gpu), E)
    cap = int((offs[1:] - offs[:-1]).max()) + 2
    for weights in (wt, None):
        xs, index = seqmix.gather_slabs(h.to(gpu), None if weights is None else weights.to(gpu), ids.to(gpu), offs, inv, cap)
        index = index.cpu().long()
        assert torch.equal(index // cap, ids.reshape(-1).long()) and index.unique().numel() == T * k
        want = h.float().repeat_interleave(k, 0) * (1.0 if weights is None else weights.reshape(-1, 1))
        torch.testing.assert_close(xs.view(E * cap, W).cpu()[index].float(), want.to(dt).float(), rtol=0, atol=0)
    got = seqmix.spread_scaled(h.to(gpu), wt.to(gpu), ids.to(gpu), E).cpu()
    torch.testing.assert_close(got.float(), seqmix.spread_scaled(h, wt, ids, E).float(), rtol=0, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("F,pad", [(8, 0), (4, 0), (5, 0), (136, 8), (136, 1), (2560, 0)])
def test_capped(gpu, dt, F, pad):
    gu = torch.randn(33, 2 * F + pad, generator=torch.Generator().manual_seed(F)).mul(6).to(dt)[:, pad:]
    gu[0, 0], gu[1, F] = float("inf"), float("-inf")
    got, want = seqmix.capped_glu(gu.to(gpu), 7.0), seqmix.capped_glu(gu, 7.0)
    torch.testing.assert_close(got.cpu().float(), want.float(), **(dict(rtol=1e-5, atol=1e-5) if dt == torch.float32 else dict(rtol=2.0 ** -7, atol=1e-5)))


@pytest.mark.parametrize("E,top,W,ff,counts,slabs", [
    (8, 2, 2048, 2560, [16] * 8, True), (8, 2, 2048, 2560, [1024] * 8, True), (8, 2, 2048, 2560, [4096, 4096] + [0] * 6, False),
    (128, 1, 128, 64, [4096] + [0] * 127, False), (128, 1, 128, 64, [32] * 128, True), (8, 2, 256, 512, [8192, 8192] + [0] * 6, False),
    (8, 2, 256, 512, [300, 212] + [0] * 6, True), (64, 6, 2048, 1408, [96] * 64, True), (8, 2, 4096, 7168, [8192] * 8, False)])
def test_when_slabs_pay(E, top, W, ff, counts, slabs):
    """Neither many empty rows, however few their operations, nor more memory than SLAB_MAX_BYTES."""
    offs = [0]
    for n in counts:
        offs.append(offs[-1] + n)
    cap = RoutedExperts("", W, E, top, ff, 7.0).slab_rows(offs, 2)
    assert cap == (max(counts) if slabs else 0)
    assert E * cap * (2 * W + 3 * ff) * 2 <= RoutedExperts.SLAB_MAX_BYTES
