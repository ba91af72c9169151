"""A parallel block's products of few rows: the last two added to the residual rows with the next norms' operands, and the first
two side by side (csrc/gemm_skinny.hip)."""
import pytest
import torch

from inferllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bf16(*shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, device=DEV, generator=g) * scale).to(torch.bfloat16)


# (2056, ...) has whole tiles at every number of rows, the others halves of tiles up to 8; one piece of K and many, a last tile of 8
@pytest.mark.parametrize("N, K, K2", [(48, 128, 896), (72, 1024, 256), (2048, 2048, 8192), (2056, 384, 1024)])
@pytest.mark.parametrize("wt", [torch.float32, torch.bfloat16])
def test_the_sum_into_the_stream_with_the_next_norms(N, K, K2, wt):
    eps = 1e-6
    x, x2 = _bf16(16, K, seed=1), _bf16(16, K2, seed=2)
    a, b = (ops.decode_weight(_bf16(N, k, seed=k, scale=0.05), "plain", True) for k in (K, K2))
    norms = [((1 + 0.1 * _bf16(N, seed=s).float()).to(wt), eps) for s in (3, 4)]
    use = ops.decode_weight(_bf16(256, N // 128 * 128 or 8, seed=5, scale=0.1), "plain", True) if N % 128 == 0 else None
    stream = torch.randn(16, N, device=DEV, generator=torch.Generator(device=DEV).manual_seed(6))
    got = {}
    for M in (1, 7, 8, 9, 16):
        pair = ops.Product(x[:M], a), ops.Product(x2[:M], b)
        want = stream[:M] + ops.linear_sum(*pair)
        for given in ((None, None), (norms[0], None), tuple(norms)):
            y = stream[:M].clone()
            left = ops.linear_sum(*pair, y, *given)
            assert torch.equal(y, want)                              # one float32 addition a number
            rows = [r for r in (left, left.second if left is not None else None) if r is not None]
            assert len(rows) == sum(g is not None for g in given)
            for r, (w, _) in zip(rows, norms):
                assert r.made_for(w, eps) and torch.equal(r.xb, (want * w.float()).to(torch.bfloat16))
                # (a float32 sum of N squares)
                exact = want.double().square().sum(1)
                assert bool(((r.ssq.double().sum(1) - exact).abs() <= N * 2.0 ** -24 * exact).all())
        got[M] = (y, *(ops.linear(r, use) for r in rows if use is not None))
        assert all(torch.equal(g[:1], o) for g, o in zip(got[M], got[1]))          # a row's bits do not depend on the others
    assert all(torch.equal(g[:8], o) for g, o in zip(got[16], got[8]))


@pytest.mark.parametrize("N, N2, K", [(16, 8, 128), (40, 2064, 256), (3648, 8192, 2048), (5128, 72, 640)])
@pytest.mark.parametrize("act", ["", "relu_squared", "gelu_tanh"])
@pytest.mark.parametrize("normed", [False, True])
def test_two_first_products(N, N2, K, act, normed):
    """Each output as its own product gives it, within the orders of a float32 sum of K products and bfloat16's rounding; a row
    has the same bits whatever the others; an infinity in one operand's row stays there."""
    a, b = (ops.decode_weight(_bf16(n, K, seed=n, scale=K ** -0.5), "plain", True) for n in (N, N2))
    x, x2 = _bf16(16, K, seed=1), _bf16(16, K, seed=2)

    def rows(M):
        if not normed:
            return x[:M].contiguous(), x2[:M].contiguous()
        stream = x[:M].float().contiguous()
        ssq = stream.square().view(M, 8, -1).sum(2).contiguous()
        w = torch.ones(K, device=DEV)
        return tuple(ops.NormedRows(stream, w, 1e-6, torch.bfloat16, t[:M].contiguous(), ssq) for t in (x, x2))

    f = {"": lambda z: z, "relu_squared": lambda z: z.relu().square(),
         "gelu_tanh": lambda z: torch.nn.functional.gelu(z, approximate="tanh")}[act]
    got = {}
    for M in (1, 8, 9, 16):
        h, h2 = rows(M)
        assert ops.linear_pair_fits(h, a, h2, b, act)
        got[M] = ops.linear_pair(h, a, h2, b, act)
        rs = torch.rsqrt(x[:M].double().square().mean(1, keepdim=True) + 1e-6) if normed else 1.0
        wants = (x[:M].double() * rs) @ a.plain.double().t(), f((x2[:M].double() * rs) @ b.plain.double().t())
        for y, want in zip(got[M], wants):
            assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -14 * want.abs().max()).all())
        assert all(torch.equal(y[:1], o) for y, o in zip(got[M], got[1]))
    if not normed:
        x2[3, 5] = float("inf")
        y, z = ops.linear_pair(*(v for p in zip(rows(16), (a, b)) for v in p), "")
        plain = ops.linear_pair(x, a, x, b, "")
        assert torch.equal(y, plain[0]) and not bool(torch.isfinite(z[3]).any()) and bool(torch.isfinite(z[[0, 1, 2, 4, 15]]).all())


def test_rows_that_are_not_a_pair():
    K = 256
    a, b = (ops.decode_weight(_bf16(n, K, seed=n), "plain", True) for n in (64, 32))
    x = _bf16(17, K, seed=1)
    stream, w, ssq = x[:4].float().contiguous(), torch.ones(K, device=DEV), torch.ones(4, 8, device=DEV)
    n = ops.NormedRows(stream, w, 1e-6, torch.bfloat16, x[:4].contiguous(), ssq)
    other = ops.NormedRows(stream, w, 1e-6, torch.bfloat16, x[:4].contiguous(), ssq.clone())
    fits = ops.linear_pair_fits
    assert fits(n, a, n, b, "") and fits(x[:16], a, x[:16], b, "gelu_tanh")
    assert not fits(x, a, x, b, "") and not fits(n, a, x[:4], b, "") and not fits(n, a, other, b, "") and not fits(n, a, n, b, "xielu")
    assert not fits(x[:4].float(), a, x[:4].float(), b, "") and not fits(x[:4], a.plain, x[:4], b, "")
    assert not fits(x[:4], ops.decode_weight(a.plain, "gate_up", True), x[:4], b, "") and not fits(x[:4], a, x[:5], b, "")
