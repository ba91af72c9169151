"""The choice and grouping of few tokens in one kernel (csrc/moe.hip) against the two kernels."""
import pytest
import torch

from inferllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _tiles(idx, grouped):
    """{expert: its pairs}, every tile within its expert's places and its size."""
    order, tiles, max_tiles, rows, _ = grouped
    order, tiles = order.cpu(), tiles.cpu()
    got = {}
    for i in range(int(tiles[3 * max_tiles])):
        e, first, n = (int(v) for v in tiles[3 * i:3 * i + 3])
        assert 1 <= n <= rows
        got.setdefault(e, []).extend(int(p) for p in order[first:first + n])
    return {e: sorted(p) for e, p in got.items()}


@pytest.mark.parametrize("T, NE, top, real", [(1, 1, 1, 1), (1, 64, 6, 64), (3, 20, 2, 17), (8, 64, 6, 64), (16, 64, 16, 60),
                                              (15, 40, 1, 40), (16, 16, 16, 12)])
@pytest.mark.parametrize("score", ["softmax", "sigmoid"])
@pytest.mark.parametrize("kind", ["plain", "corrected", "ties", "infinite"])
def test_choice_and_grouping_in_one_kernel(T, NE, top, real, score, kind):
    g = torch.Generator(device=DEV).manual_seed(T * NE + top)
    z = torch.randn(T, NE, device=DEV, generator=g)
    corr = torch.randn(NE, device=DEV, generator=g) * 0.1 if kind == "corrected" else None
    if kind == "ties":
        z = z.round()
    if kind == "infinite":
        z[T // 2, NE // 2] = -float("inf")
        corr = torch.where(torch.arange(NE, device=DEV) == NE - 1, -float("inf"), 0.0)
    idx, wt = ops.moe_route(z, corr, top, score, 0.7)
    grouped = ops._moe_group(idx, real, torch.bfloat16, 256, 128)
    idx2, wt2, grouped2 = ops._moe_route_group(z, corr, top, score, 0.7, real, torch.bfloat16, 256, 128)
    assert torch.equal(idx, idx2) and torch.equal(wt, wt2) and grouped[2:] == grouped2[2:]
    want = {}
    for p, e in enumerate(idx.flatten().tolist()):
        if 0 <= e < real:
            want.setdefault(e, []).append(p)
    assert _tiles(idx, grouped) == want == _tiles(idx2, grouped2)


@pytest.mark.parametrize("T, E, top, NEr, dtype", [(1, 8, 1, 4, torch.bfloat16), (8, 2048, 6, 64, torch.bfloat16), (3, 2056, 9, 5, torch.bfloat16),
                                                   (130, 4, 8, 6, torch.float32), (5, 1028, 16, 30, torch.float32)])
@pytest.mark.parametrize("weights, shared", [(True, True), (False, False), (True, False)])
def test_combine_with_choices_that_are_no_experts(T, E, top, NEr, dtype, weights, shared):
    """Choices from NEr on give the token's own row; the rows of Y that belong to them are never used (NaN here)."""
    g = torch.Generator(device=DEV).manual_seed(T * E)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    h, y = rnd(T, E).to(dtype), rnd(T * top, E).to(dtype)
    idx = torch.randint(0, NEr + 3, (T, top), device=DEV, generator=g).int()
    y[(idx.flatten() >= NEr)] = float("nan")
    wt = rnd(T, top) if weights else None
    sh, sg = (rnd(T, E).to(dtype), rnd(E).to(dtype)) if shared else (None, None)
    got = ops.moe_combine(h, idx, wt, y, NEr, sh, sg)
    rows = torch.where((idx < NEr)[..., None], y.view(T, top, E).double(), h.double()[:, None])
    want = (rows * (wt.double()[..., None] if weights else 1.0)).sum(1)
    size = (rows.abs() * (wt.double().abs()[..., None] if weights else 1.0)).sum(1)
    if shared:
        gate = torch.sigmoid((h.double() * sg.double()).sum(1, keepdim=True))
        want, size = want + gate * sh.double(), size + 8 * sh.double().abs()         # (the gate's own sum of E products)
    assert bool(((got.double() - want).abs() <= (top + 4 + (E if shared else 0)) * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("T, E, top, dtype", [(3, 264, 2, torch.bfloat16), (131, 2056, 1, torch.bfloat16), (9, 12, 2, torch.float32)])
def test_combine_of_one_or_two_choices(T, E, top, dtype):
    test_combine_with_choices_that_are_no_experts(T, E, top, 4, dtype, True, True)
