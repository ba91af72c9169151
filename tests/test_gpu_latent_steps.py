"""Single tokens over the latent cache at the edges of the kernels for wide latents (csrc/latent_attention.hip), against plain
torch: queries through W_uk, the walk of four waves a block, the merge that asks for everything at once."""
import pytest
import torch

import kernel_refs as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B, H, Rk, dr, dv, window", [
    (1, 16, 512, 64, 128, 0),        # five steps of scores a wave, the last in part
    (2, 3, 272, 8, 33, 0),           # row groups and steps past the end, one value dim in the last block
    (3, 17, 512, 192, 40, 50),       # a second group of heads with one, eight steps a wave, a window
    (8, 16, 384, 128, 128, 0),       # 128 heads of rows: the most that the merge for few takes
    (9, 16, 384, 128, 64, 0),        # ... and one row more
    (33, 16, 512, 64, 32, 0),        # more than 512 heads of rows: queries by blocks of 512 dims
    (2, 2, 512, 552, 16, 0)])        # keys wider than the four waves' steps
@pytest.mark.parametrize("dn", [1, 130])
def test_wide_latents(B, H, Rk, dr, dv, window, dn, monkeypatch):
    from inferllm_amd.kernels import ops
    g, page, per, bf = torch.Generator().manual_seed(B * 1000 + Rk + dr), 64, 6, torch.bfloat16
    lens = torch.tensor([1 + (i * 61 + 31) % 380 for i in range(B)], dtype=torch.int32)
    table = torch.randperm(B * per, generator=g).view(B, per).to(torch.int32)
    cache = torch.randn(B * per, page, Rk + dr, generator=g).to(bf)
    ct = cache[:, :, :Rk].transpose(1, 2).contiguous().unsqueeze(-1)
    y = torch.randn(B, H * (dn + dr) + Rk + dr + H, generator=g).to(bf)
    gate_off = y.shape[1] - H
    wuk, wuv = ((torch.randn(n, Rk, generator=g) * Rk ** -0.5).to(bf) for n in (H * dn, H * dv))
    put = lambda t: t.cuda()  # noqa: E731
    slot = torch.randperm(B, generator=g).to(torch.int32)
    qa = ops.latent_absorb_q(put(y), put(wuk), H, dn, dr, Rk, bf)
    want = R.latent_absorb_q(y, wuk, H, dn, dr, Rk, torch.float32).double()
    # a result's rounding, 2^-9 of it
    assert float((qa.double().cpu() - want).abs().max()) <= 2 ** -8 * float(want.abs().max())
    qa = (qa.float() * (0.3 / float(want.std()))).to(bf)
    scale = (Rk + dr) ** -0.5
    want = R.latent_attn_decode(qa.cpu(), y, wuv, gate_off, cache, table, page, 0, slot, lens, 0, H, dr, Rk, dv, scale, window, 1).double()
    real = torch.empty
    for nsplit in (1, 5, 12, 17, 64):
        with monkeypatch.context() as m:             # (what no range writes may not be read)
            m.setattr(torch, "empty", lambda *a, **k: real(*a, **k).fill_(float("nan")))
            got = ops.latent_attn_decode(qa, put(y), put(wuv), gate_off, put(cache), put(table), page, 0, put(slot), put(lens), 0, H,
                                         dr, Rk, dv, scale, window, nsplit, put(ct)).double().cpu()
        assert bool(torch.isfinite(got).all()), nsplit
        # a weight's and a result's rounding, 2^-9 each
        assert float((got - want).norm() / want.norm()) < 2 ** -7, nsplit


@pytest.mark.parametrize("R_", [8, 24, 64, 200, 320, 512])
@pytest.mark.parametrize("B", [32, 33])
def test_queries_on_either_side_of_512_heads_of_rows(B, R_):
    from inferllm_amd.kernels import ops
    g, H, dn, dr, bf = torch.Generator().manual_seed(B + R_), 16, 72, 12, torch.bfloat16
    y = torch.randn(B, H * (dn + dr) + R_ + dr + H, generator=g).to(bf)
    wuk = (torch.randn(H * dn, R_, generator=g) * R_ ** -0.5).to(bf)
    got = ops.latent_absorb_q(y.cuda(), wuk.cuda(), H, dn, dr, R_, torch.float32).double().cpu()
    want = R.latent_absorb_q(y, wuk, H, dn, dr, R_, torch.float32).double()
    # float32 sums of dn products in another order: 2 dn 2^-24 of the sum of their sizes
    size = R.latent_absorb_q(y.abs(), wuk.abs(), H, dn, dr, R_, torch.float32).double()
    assert bool(((got - want).abs() <= 2 * dn * 2.0 ** -24 * size).all())
