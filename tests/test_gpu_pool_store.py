"""Pooled rows of completed blocks, several rows a block of the launch (csrc/attention_pooled.hip)."""
import pytest
import torch

from inferllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("lens, pool, dk, dv", [([1], 1, 8, 4), ([7], 8, 128, 128), ([8, 1], 8, 96, 40), ([17, 9, 40], 12, 20, 256),
                                                ([65, 130], 3, 128, 64), ([100], 16, 256, 12)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_means_of_completed_blocks(lens, pool, dk, dv, dtype):
    """Sums in position order in float32, one rounding of the mean: exactly torch's, added in that order.  Rows that no block
    belongs to stay."""
    nkv, page, per = 2, 16, 12
    g = torch.Generator().manual_seed(sum(lens) + pool)
    table = torch.randperm(len(lens) * per, generator=g).int().view(len(lens), per)
    caches = [torch.randn(table.numel(), nkv, page, n, generator=g).to(dtype) for n in (dk, dv)]
    pos = torch.cat([torch.arange(n) for n in lens]).int()
    slot = torch.cat([torch.full((n,), i) for i, n in enumerate(lens)]).int()
    pooled = [torch.full_like(c, 7.0) for c in caches]
    want = [p.clone() for p in pooled]
    for i, n in enumerate(lens):
        for b in range(n // pool):
            for c, w in zip(caches, want):
                s = torch.zeros(nkv, c.shape[-1])
                for j in range(b * pool, (b + 1) * pool):
                    s += c[table[i, j // page], :, j % page].float()
                w[table[i, b // page], :, b % page] = (s * (torch.tensor(1.0) / pool)).to(dtype)
    on = [t.to(DEV) for t in (pos, slot, *caches, *pooled, table)]
    ops.pool_store(*on, page, nkv, dk, dv, pool)
    assert torch.equal(on[4].cpu(), want[0]) and torch.equal(on[5].cpu(), want[1])
