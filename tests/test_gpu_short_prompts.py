"""Products of a short prompt's rows (csrc/gemm_short.hip) against float32 on the same bfloat16 operands: sums of K products in
float32 and one rounding of the result, 2^-8 of the largest value of the tensor with the rotation's or the activation's float32
steps (the activation's error is the sums': below 2^-16 of the largest gate times the largest up, which 2^-8 covers).  And the
rule: which calls go there, on any machine."""
import json

import pytest
import torch

from inferllm_amd.kernels import ops
from inferllm_amd.kernels.plan import Plan

DEV = "cuda"


def _weight(rows, K, mode, **geometry):
    g = torch.Generator(device=DEV).manual_seed(rows + K)
    w = (torch.randn(rows, K, device=DEV, generator=g) * K ** -0.5).to(torch.bfloat16)
    return ops.decode_weight(w, mode, True, **geometry)


# rows at the edges of the kernel's tiles of 32 rows, K of one, two and four parts with a ragged last one, heads whose tiles end
# within a block's, whole prompts with pages in a ring (a row that a later row overwrites is left out) and without
@pytest.mark.gpu
@pytest.mark.parametrize("M, K, nh, nkv, hd, ring", [
    (17, 512, 1, 1, 16, 0), (32, 576, 5, 1, 16, 2), (33, 1024, 4, 2, 48, 0), (129, 1088, 6, 2, 128, 2), (160, 2048, 16, 4, 128, 0),
    (193, 4096, 32, 8, 128, 3), (256, 1280, 3, 3, 80, 0)])
def test_qkv_of_a_short_prompt(M, K, nh, nkv, hd, ring):
    page, a = 32, M // 3
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
    w = _weight((nh + 2 * nkv) * hd, K, "qkv", nh=nh, nkv=nkv, hd=hd)
    table = torch.randn(M, hd // 2, 2, device=DEV, generator=g)
    pos = torch.cat([torch.arange(a), torch.arange(M - a)]).int().to(DEV)
    slot = torch.cat([torch.ones(a), torch.zeros(M - a)]).int().to(DEV)
    lengths = torch.tensor([M - a, a], dtype=torch.int32, device=DEV)
    pages = ring or -(-M // page)
    where = torch.randperm(2 * pages, generator=torch.Generator().manual_seed(M)).view(2, pages).int().to(DEV)
    caches = [torch.zeros(2 * pages, nkv, page, hd, dtype=torch.bfloat16, device=DEV) for _ in range(4)]
    assert ops.qkv_short_fits(x, w, hd)
    y = ops.qkv_short(x, w, table, pos, slot, lengths, *caches[:2], where, page, ring, nh, nkv, hd)
    want = x.float() @ w.plain.float().t()
    ops.rope_store(want, table, hd, 0, pos, slot, None, None, None, None, 1, 0, nh, nkv, hd)
    assert (y.float() - want).abs().max() <= 2.0 ** -8 * want.abs().max()
    # the cache holds these very rows, where the general kernel stores them (rotation by the angle 0)
    still = torch.tensor([1.0, 0.0], device=DEV).expand(M, hd // 2, 2).contiguous()
    ops.rope_store(y.clone(), still, hd, 0, pos, slot, lengths, *caches[2:], where, page, ring, nh, nkv, hd)
    assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])


@pytest.mark.gpu
@pytest.mark.parametrize("M, F, K, limit", [(129, 8, 512, 0.0), (144, 1000, 1088, 1.5), (160, 2816, 1024, 0.0), (161, 264, 2048, 0.5),
                                            (192, 8192, 2048, 0.0)])
def test_gate_and_up_of_a_short_prompt(M, F, K, limit):
    x = torch.randn(M, K, device=DEV, generator=torch.Generator(device=DEV).manual_seed(M)).to(torch.bfloat16)
    w = _weight(2 * F, K, "gate_up")
    assert ops.gate_up_short_fits(x, w)
    y = ops.gate_up_act(x, w, limit)
    gate, up = (x.float() @ w.plain.float().t()).split(F, 1)
    if limit:
        gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
        want = gate * torch.sigmoid(1.702 * gate) * (up + 1)
    else:
        want = torch.nn.functional.silu(gate) * up
    assert (y.float() - want).abs().max() <= 2.0 ** -8 * want.abs().max()


@pytest.mark.gpu
def test_what_a_short_prompts_kernels_leave_to_the_general_path():
    x = torch.zeros(130, 512, dtype=torch.bfloat16, device=DEV)
    gate_up, qkv = _weight(2 * 48, 512, "gate_up"), _weight(48, 512, "qkv", nh=1, nkv=1, hd=16)
    assert ops.gate_up_short_fits(x, gate_up) and ops.qkv_short_fits(x, qkv, 16)
    for other in (x[:16], x.float(), x.new_zeros(257, 512), x.new_zeros(130, 1024)[:, ::2], x.new_zeros(130 * 512 + 1)[1:].view(130, 512),
                  x.new_zeros(130, 576)):
        assert not ops.gate_up_short_fits(other, gate_up) and not ops.qkv_short_fits(other, qkv, 16)
    assert not ops.gate_up_short_fits(x[:128], gate_up) and not ops.gate_up_short_fits(x.new_zeros(193, 512), gate_up)
    assert not ops.gate_up_short_fits(x, gate_up.plain) and not ops.gate_up_short_fits(x, qkv)
    assert not ops.qkv_short_fits(x, qkv.plain, 16) and not ops.qkv_short_fits(x, gate_up, 16)


def test_a_pinned_plan_keeps_the_products_of_short_prompts_that_it_was_made_with():
    shape = (22016, 4096)
    old = Plan.fixed().to_dict()
    del old["short"]
    assert all(Plan.from_dict(json.loads(json.dumps(old))).keeps_short(M, *shape) for M in (17, 160, 256))
    own = Plan(cuts={("pad", 5, *shape): ("pad", 256), (1, 12288, 4096): ()})
    assert [own.keeps_short(M, *shape) for M in (128, 129, 160, 161)] == [False, True, True, False]
    assert own.keeps_short(32, 12288, 4096)
    for plan in (own, Plan.fixed(), Plan()):
        again = Plan.from_dict(json.loads(json.dumps(plan.to_dict())))
        assert again == plan and again.short is plan.short
    assert not Plan.fixed().keeps_short(160, *shape) and not Plan().keeps_short(160, *shape)


# csrc/gemm_tiles.hip with blocks of 128 columns: parts of K of 16 stages and more, of unequal length, a ragged last block, and the
# rows at the edges of both variants
@pytest.mark.gpu
@pytest.mark.parametrize("M, N, K, splits", [(129, 4096, 8192, 8), (192, 8196, 3136, 3), (193, 4132, 7232, 7), (256, 16384, 2048, 2), (1, 8320, 4096, 3)])
def test_cut_products_of_wide_blocks(M, N, K, splits):
    """Any order of K float32 sums: K 2^-24 of the sum of magnitudes."""
    g = torch.Generator(device=DEV).manual_seed(M)
    x, w = (torch.randn(n, K, device=DEV, generator=g).to(torch.bfloat16) for n in (M, N))
    planes = ops.linear_cut(x, w)
    assert planes.shape == (splits, M, N)
    want, room = (x.double() @ w.double().t(), K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()))
    assert bool(((planes.double().sum(0) - want).abs() <= room).all())


def test_small_and_narrow_matrices_of_a_short_prompt_stay_with_the_vendor_gemm():
    """(N, K) and the rows up to which q|k|v goes to the kernel: each side measured faster there."""
    assert [ops.qkv_short_rows(N, K) for N, K in ((768, 768), (1280, 8192), (1536, 1024), (4096, 2048), (6144, 2048), (7680, 2560),
                                                   (3072, 4096), (12288, 4096))] == [96, 96, 160, 160, 160, 256, 256, 256]
