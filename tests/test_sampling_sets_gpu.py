"""The sampler's top-k / top-p sets at the sizes where its forms change (a row in registers or read again by every pass,
16-byte aligned or not) and for rows whose histogram bins overflow: every sampled token lies in the exact set, and is the
Gumbel maximum of it."""
import pytest
import torch

from mxserve import ops
from mxserve.ops import reference as ref

pytestmark = pytest.mark.gpu


def exact_set(row: torch.Tensor, t: float, k: int, p: float, slack: float) -> torch.Tensor:
    """The tokens that may be sampled, in 64 bits; slack widens (> 0) or narrows (< 0) the nucleus by that share, more
    than the kernel's 2^-46 fixed-point shares (2^-29 of a row) and the rounding of their exponentials (2^-22 each, and
    2^-24 of the exponent) can move it."""
    z = row.double()
    keep = torch.isfinite(z)
    if 0 < k < z.numel():
        keep &= z >= torch.topk(z, k).values[-1]
    if p < 1.0:
        q = torch.softmax(z / t, -1)
        s, order = torch.sort(z, descending=True)
        before = torch.cumsum(q[order], 0) - q[order]
        first = before < p + slack
        first[0] = True
        keep &= z >= s[first][-1]
    return keep


def rows_of(kind: str, B: int, V: int, g: torch.Generator) -> torch.Tensor:
    if kind == "flat":
        return torch.randn(B, V, generator=g) * 0.8
    if kind == "peaked":
        return torch.randn(B, V, generator=g) * 4.0
    if kind == "equal":
        return torch.full((B, V), 1.25)
    if kind == "steps":  # few values, each of them many times: fuller than a bin's list
        return torch.randint(0, 3, (B, V), generator=g).float() * 0.5
    x = torch.randn(B, V, generator=g) * 2.0  # "masked": most tokens are not allowed
    x[:, torch.rand(V, generator=g) < 0.7] = float("-inf")
    x[:, V // 2] = 3.0
    return x


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 8), (torch.bfloat16, 1001), (torch.bfloat16, 32768), (torch.bfloat16, 32776),
                                     (torch.bfloat16, 131072), (torch.bfloat16, 151936), (torch.bfloat16, 163848),
                                     (torch.float32, 1), (torch.float32, 1003), (torch.float32, 32000), (torch.float32, 50000),
                                     (torch.float32, 70000)])
@pytest.mark.parametrize("kind", ["flat", "peaked", "equal", "steps", "masked"])
def test_sampled_tokens_are_the_sets_maxima(gpu, dtype, V, kind):
    g = torch.Generator().manual_seed(V)
    cases = [(0.7, 0, 0.95), (0.7, 0, 0.5), (1.3, 0, 1e-4), (1.0, 1, 1.0), (1.0, 40, 1.0), (0.9, 700, 0.9), (0.01, 0, 0.9), (1.0, 0, 1.0)]
    if kind == "equal":
        cases = cases[:1] + cases[-2:]
    B = len(cases)
    logits = rows_of(kind, B, V, g).to(dtype)
    t = torch.tensor([c[0] for c in cases])
    k = torch.tensor([c[1] for c in cases], dtype=torch.int32)
    p = torch.tensor([c[2] for c in cases])
    seeds, steps = torch.arange(5, 5 + B), torch.full((B,), 2, dtype=torch.int64)
    ids = ops.sample(*(x.to(gpu) for x in (logits, t, p, k, seeds, steps))).cpu()
    u = ref.uniform_noise(seeds, steps, V).double()
    for i, (ti, ki, pi) in enumerate(cases):
        wide = exact_set(logits[i].float(), float(t[i]), ki, float(p[i]), 2e-6)
        narrow = exact_set(logits[i].float(), float(t[i]), ki, float(p[i]), -2e-6)
        score = logits[i].double() / float(t[i]) - torch.log(-torch.log(u[i]))
        got = int(ids[i])
        assert 0 <= got < V and bool(wide[got]), (kind, V, cases[i], got)
        # fp32 scores: two hardware logarithms of about 2^-22 relative error each, around values of up to |z| / t
        tol = 1e-5 * max(1.0, float(score[wide].abs().max()))
        assert float(score[got]) >= float(score[narrow].max()) - tol, (kind, V, cases[i])


@pytest.mark.parametrize("V", [131072, 262144, 300007])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_many_small_shares_count(gpu, dtype, V):
    """131,000 tokens of 2^-34 of the likeliest one's share are 8e-6 of the whole and move the border of a nucleus that ends
    among the tokens before them.  The second token lies where the row's noise makes it the maximum, so that the sample tells."""
    for seed in range(1000):
        u = ref.uniform_noise(torch.tensor([seed]), torch.tensor([2]), V)[0].double()
        noise = -torch.log(-torch.log(u))
        if float(noise.max()) > 16.0:
            break
    mid, first = int(noise.argmax()), int(noise.argmin())
    z = torch.full((V,), -34 * 0.6931471805599453)
    others = [v for v in (7, 7777, 77777, 100003) if v not in (mid, first)]
    z[others], z[mid], z[first] = -14.25, -13.75, 0.0
    z = z.to(dtype)
    share = torch.exp(z.double() - float(z[first]))
    p = float((share[first] + 0.5 * share[mid]) / share.sum())  # half way into the second token: fp32 steps of p are 6e-8
    assert abs(float(torch.tensor(p)) - p) < 0.1 * float(share[mid])
    one = lambda x, t: torch.tensor([x], dtype=t, device=gpu)  # noqa: E731
    got = ops.sample(z.view(1, V).to(gpu), one(1.0, torch.float32), one(p, torch.float32), one(0, torch.int32),
                     one(seed, torch.int64), one(2, torch.int64))
    assert int(got[0]) == mid


@pytest.mark.parametrize("V", [5, 8, 1000, 8192, 8200, 24576, 32768, 32776, 65544, 163848])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_of_one_pass(gpu, dtype, V):
    """Greedy rows and draws without a set, which no register form holds: every place of a row can win, the last one too."""
    g = torch.Generator().manual_seed(V)
    best = sorted({0, V // 2, V - 1, V * 3 // 4, min(V - 1, 8191), min(V - 1, 16384)})
    B = 2 * len(best)
    z = (torch.randn(B, V, generator=g) * 0.5).clamp(-2, 2).to(dtype)
    temp = torch.tensor([0.0, 0.8] * len(best))
    seeds, steps = torch.arange(B), torch.full((B,), 3)
    for i, v in enumerate(best):
        z[2 * i, v] = 3.0
    got = ops.sample(z.to(gpu), temp.to(gpu), torch.ones(B, device=gpu), torch.zeros(B, dtype=torch.int32, device=gpu),
                     seeds.to(gpu), steps.to(gpu)).cpu()
    assert got[::2].tolist() == best
    noise = -torch.log(-torch.log(ref.uniform_noise(seeds[1::2], steps[1::2], V).double()))
    score = z[1::2].double() / 0.8 + noise
    # the kernel's noise is two fp32 logarithms: 2^-20 of a score of at most 20
    assert (score.max(-1).values - score.gather(1, got[1::2, None])[:, 0] <= 2e-5).all()
