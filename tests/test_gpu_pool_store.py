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


@pytest.mark.parametrize("T, pool, dk, dv, shift", [(9, 8, 128, 128, 0), (17, 5, 64, 8, 0), (8, 13, 256, 256, 0), (33, 3, 36, 20, 0),
                                                    (9, 7, 128, 64, 1), (8, 1, 7, 250, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_sequences_that_complete_a_block_together(T, pool, dk, dv, shift, dtype):
    """One token of every sequence, each the last of its block (a block of the launch has up to 8 means to form), eight or four
    columns a thread and one, rows that do not lie on 16 bytes."""
    nkv, page = 2, 16
    per = -(-3 * pool // page)
    g = torch.Generator().manual_seed(T + pool)

    def rows(n, fill=None):
        t = torch.randn(T * per * nkv * page * n + shift, generator=g) if fill is None else torch.full((T * per * nkv * page * n + shift,), fill)
        return t.to(dtype)[shift:].view(T * per, nkv, page, n)
    table = torch.randperm(T * per, generator=g).int().view(T, per)
    caches, pooled = [rows(n) for n in (dk, dv)], [rows(n, 7.0) for n in (dk, dv)]
    pos, slot = torch.tensor([pool * (1 + i % 3) - 1 for i in range(T)]).int(), torch.randperm(T, generator=g).int()
    want = [p.clone() for p in pooled]
    for p, s in zip(pos.tolist(), slot.tolist()):
        for c, w in zip(caches, want):
            a = torch.zeros(nkv, c.shape[-1])
            for j in range(p + 1 - pool, p + 1):
                a += c[table[s, j // page], :, j % page].float()
            b = p // pool
            w[table[s, b // page], :, b % page] = (a * (torch.tensor(1.0) / pool)).to(dtype)

    def put(t):                                   # (a view that begins `shift` elements into its memory)
        flat = torch.empty(t.numel() + shift, dtype=t.dtype, device=DEV)
        return flat[shift:].view(t.shape).copy_(t)
    on = [pos.to(DEV), slot.to(DEV), *map(put, caches), *map(put, pooled), table.to(DEV)]
    ops.pool_store(*on, page, nkv, dk, dv, pool)
    assert torch.equal(on[4].cpu(), want[0]) and torch.equal(on[5].cpu(), want[1])
