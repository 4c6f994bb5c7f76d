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
