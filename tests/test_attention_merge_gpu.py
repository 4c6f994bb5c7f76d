"""Merges of split attention rows: partition counts around the eight that a merge has in flight."""
import pytest
import torch

from mxserve import ops
from mxserve.ops import reference as ref, seqmix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[1], [257], [900, 3], [1791, 2049, 2304], [4500]])
def test_decode_partitions(gpu, lens):
    g = torch.Generator().manual_seed(len(lens) + lens[0])
    B, H, G, D = len(lens), 8, 2, 64
    nb = [-(-n // 16) for n in lens]
    kv = torch.randn(sum(nb), 2, G, 16, D, generator=g).bfloat16()
    bt = torch.zeros(B, max(nb), dtype=torch.int32)
    ids, u = torch.randperm(sum(nb), generator=g), 0
    for i, n in enumerate(nb):
        bt[i, :n] = ids[u:u + n]
        u += n
    q = torch.randn(B, H, D, generator=g).bfloat16()
    sl, qsl = torch.tensor(lens, dtype=torch.int32), torch.arange(B + 1).int()
    got = ops.paged_attention_decode(q.to(gpu), kv.to(gpu), bt.to(gpu), sl.to(gpu), D ** -0.5, max(lens))
    want = ref.paged_attention(q, kv, bt, qsl, sl, D ** -0.5)
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=2.0 ** -6, atol=2.0 ** -7)  # weights and result in bf16


@pytest.mark.parametrize("rank", [16, 64, 512])
@pytest.mark.parametrize("rows,ctx", [(1, 40), (1, 300), (3, 200), (70, 260), (9, 1000)])
def test_latent_stretches(gpu, rank, rows, ctx):
    g = torch.Generator().manual_seed(rank + rows)
    H, dk = 4, rank + 16
    nb = -(-ctx // 16)
    cache = torch.randn(rows * nb, 16 * dk, generator=g).bfloat16()
    bt = torch.randperm(rows * nb, generator=g).int().view(rows, nb)
    q = torch.randn(rows, H * dk, generator=g).bfloat16()
    sl = torch.randint(1, ctx + 1, (rows,), generator=g).int()  # some stretches hold no keys
    qsl = torch.arange(rows + 1).int()
    args = (0, H, dk, rank, 16, dk ** -0.5, 1, ctx)
    got = seqmix.latent_attention(q.to(gpu), cache.to(gpu), bt.to(gpu), qsl.to(gpu), sl.to(gpu), *args)
    want = seqmix.latent_attention(q.float(), cache.float(), bt, qsl, sl, *args)
    torch.testing.assert_close(got.cpu().float(), want, rtol=2.0 ** -7, atol=2.0 ** -7)  # values of size one, result in bf16
