"""Single tokens through mixers with a matrix of state a head in one launch (csrc/mixer_steps.hip), against what stands around the
plain gated rule as separate steps in plain torch (tests/kernel_refs.py), in 64 bits."""
import pytest
import torch

import kernel_refs as R

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]
# rows past a wave's in the last waves and columns past the last 64, one row or column, the smallest and largest of each size
SIZES = [(1, 1), (40, 9), (64, 64), (65, 65), (128, 128), (129, 130), (256, 256), (250, 193)]


def _near(got, want, dtype):
    # float32: sums of up to 256 terms in another order (16 parts); bfloat16 results: half an ulp, 2^-9, and a tie's other side
    rel = 1e-5 if dtype == torch.float32 else 2.0 ** -8
    got, want = got.double().cpu(), want.double()
    assert got.shape == want.shape
    assert float((got - want).abs().max()) <= rel * float(want.abs().max()), float((got - want).abs().max() / want.abs().max())


def _slots(B, g):
    return torch.randperm(B + 2, generator=g)[:B].to(torch.int32), torch.arange(B + 1, dtype=torch.int32)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dk,dv", SIZES)
def test_matrix_memory_step(dk, dv, dtype):
    from inferllm_amd.kernels import ops
    g = torch.Generator().manual_seed(dk * 300 + dv)
    B, H, cap = 3, 5, 3.0
    i_off = 2 * H * dk + H * dv
    z_off = i_off + 2 * H + 1
    U = torch.randn(B, z_off + H * dv, generator=g).to(dtype)
    bias, w = torch.randn(2, H, generator=g), torch.randn(H * dv, generator=g).to(dtype)
    m, S = torch.randn(B + 2, H, generator=g), torch.randn(B + 2, H, dk, dv + 1, generator=g)
    slot, cu = _slots(B, g)
    m_got, S_got = m.cuda(), S.cuda()
    got = ops.memory_step(U.cuda(), i_off, i_off + H, z_off, bias[0].cuda(), bias[1].cuda(), cap, m_got, S_got, slot.cuda(),
                          w.cuda(), H, dk, dv, 1e-5)
    q, k, v, beta, dec, em = R.memory_prepare(U, i_off, i_off + H, bias[0], bias[1], cap, m, cu, slot, B, H, dk, dv)
    want = R.memory_finish(R.delta_scan(q, k, v, beta, dec, S, cu, slot, B, 1, correct=False), em, w, U, z_off, 1e-5, torch.float32)
    _near(got, want, dtype)
    _near(S_got, S, torch.float32)
    _near(m_got, m, torch.float32)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("ra", [4, 16, 28])
@pytest.mark.parametrize("dk,dv", SIZES)
def test_gated_linear_attention_step(dk, dv, ra, dtype):
    from inferllm_amd.kernels import ops
    g = torch.Generator().manual_seed(dk * 300 + dv + ra)
    B, H, tau = 3, 5, 7.0
    a_off = -(-(2 * H * dk + 2 * H * dv) // 4) * 4
    cols = (1, H * dk + 1, 2 * H * dk, 2 * H * dk + H * dv)
    U = torch.randn(B, a_off + ra, generator=g).to(dtype)
    w2, zb = (torch.randn(H * dk, ra, generator=g) * 0.5).to(dtype), torch.randn(H * dk, generator=g)
    w, S = torch.randn(dv, generator=g).to(dtype), torch.randn(B + 2, H, dk, dv, generator=g)
    slot, cu = _slots(B, g)
    S_got = S.cuda()
    assert ops.gla_step_fits(U.cuda(), a_off, w2.cuda(), dk, dv, dtype)
    got = ops.gla_step(U.cuda(), *cols, a_off, w2.cuda(), zb.cuda(), tau, S_got, slot.cuda(), w.cuda(), H, dk, dv, 1e-5)
    Z = U[:, a_off:].double() @ w2.double().t()
    ins = R.gla_prepare(U, *cols[:3], Z, zb, tau, H, dk, dv)
    want = R.delta_finish(R.delta_scan(*ins, S, cu, slot, B, 1, correct=False), w, U, cols[3], "silu", 1e-5, torch.float32)
    _near(got, want, dtype)
    _near(S_got, S, torch.float32)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("G,H,taps,groups", [(2, 4, 4, 4), (3, 3, 1, 1), (1, 6, 8, 2)])
@pytest.mark.parametrize("N,dv", SIZES)
def test_state_space_step(N, dv, G, H, taps, groups, dtype):
    from inferllm_amd.kernels import ops
    g = torch.Generator().manual_seed(N * 300 + dv + taps)
    B, inner, C = 3, H * dv, H * dv + 2 * G * N
    U = torch.randn(B, 2 * inner + 2 * G * N + H + 3, generator=g).to(dtype)
    cols = (inner + 1, 2 * inner + 2 * G * N + 2, 0)
    conv_w, conv_b = torch.randn(C, taps, generator=g), torch.randn(C, generator=g)
    tail = torch.randn(B + 2, max(taps - 1, 1), C, generator=g).to(dtype)
    a_log, dt_bias, D = torch.randn(3, H, generator=g)
    w, S = torch.randn(inner, generator=g).to(dtype), torch.randn(B + 2, H, N, dv, generator=g)
    slot, cu = _slots(B, g)
    t_got, S_got = tail.cuda(), S.cuda()
    got = ops.ssm_step(U.cuda(), *cols, conv_w.cuda(), conv_b.cuda(), t_got, S_got, slot.cuda(), a_log.cuda(), dt_bias.cuda(),
                       D.cuda(), w.cuda(), groups, 1e-5, G, H, N, dv)
    q, k, v, step, dec = R.ssm_prepare(U, cols[0], cols[1], conv_w, conv_b, tail, slot, a_log, dt_bias, G, H, N, dv, update_tail=True)
    o = R.delta_scan(q, k, v, step, dec, S, cu, slot, B, 1, correct=False)
    _near(got, R.ssm_finish(o, v, D, U, 0, w, groups, 1e-5, torch.float32), dtype)
    _near(S_got, S, torch.float32)
    assert torch.equal(t_got.cpu(), tail)


@pytest.mark.parametrize("H, dk, lens", [(3, 8, [64, 1, 65]), (2, 4, [63, 500]), (1, 4, [128])])
def test_matrix_memory_gates_of_long_runs(H, dk, lens):
    """Maxima by a scan of 64 tokens: its edges, gates that stay far below the maximum for many tokens (whose decays add up) and
    gates that take it over."""
    from inferllm_amd.kernels import ops
    g = torch.Generator().manual_seed(sum(lens))
    T, n, cap = sum(lens), len(lens), 15.0
    i_off = 3 * H * dk
    U = torch.randn(T, i_off + 2 * H, generator=g) * 4
    U[::7, i_off:i_off + H] -= 40.0
    slot = torch.randperm(n + 1, generator=g)[:n].to(torch.int32)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    bias, m = torch.randn(2, H, generator=g), torch.randn(n + 1, H, generator=g)
    m_got = m.cuda()
    got = ops.memory_prepare(U.cuda(), i_off, i_off + H, bias[0].cuda(), bias[1].cuda(), cap, m_got, cu.cuda(), slot.cuda(), n, H, dk, dk)
    want = R.memory_prepare(U, i_off, i_off + H, bias[0], bias[1], cap, m, cu, slot, n, H, dk, dk)
    for a, b in zip(got[3:], want[3:]):      # weight, decay, exp(-m): exponentials of numbers up to 15, whose sums of up to 64 round
        assert bool(((a.double().cpu() - b.double()).abs() <= 64 * 15 * 2.0 ** -24 * b.double().abs() + 1e-30).all())
    torch.testing.assert_close(m_got.cpu(), m, atol=64 * 15 * 2.0 ** -24, rtol=0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H, dv, groups", [(2, 4, 1), (4, 12, 2), (3, 100, 1), (8, 128, 2), (64, 64, 8), (33, 124, 1), (5, 66, 1)])
def test_state_space_finish_four_columns_a_load(H, dv, groups, dtype):
    from inferllm_amd.kernels import ops
    g = torch.Generator().manual_seed(H * dv)
    T, inner = 5, H * dv
    o, x, D = torch.randn(T, H, dv, generator=g), torch.randn(T, H, dv, generator=g), torch.randn(H, generator=g)
    Z, w = torch.randn(T, inner + 8, generator=g).to(dtype), torch.randn(inner, generator=g).to(dtype)
    got = ops.ssm_finish(o.cuda(), x.cuda(), D.cuda(), Z.cuda(), 4, w.cuda(), groups, 1e-5, torch.float32)
    _near(got, R.ssm_finish(o, x, D, Z, 4, w, groups, 1e-5, torch.float32), torch.float32)


@pytest.mark.parametrize("nb, cb", [(2, 64), (3, 128), (1, 192), (2, 256), (1, 320), (1, 4096)])
def test_recurrent_gates_of_many_rows(nb, cb):
    """16 rows and up to 256 outputs a block: slices, waves and whole blocks without outputs, a last tile of one row."""
    from inferllm_amd.kernels import ops
    g = torch.Generator().manual_seed(cb)
    T, C = 145, nb * cb
    u, wt = torch.randn(T, C, generator=g), torch.randn(2, nb, cb, cb, generator=g) * cb ** -0.5
    rb, ib, lam = torch.randn(3, C, generator=g)
    for got, want in zip(ops.lru_gates(*(t.cuda() for t in (u, wt, rb, ib, lam)), 8.0), R.lru_gates(u, wt, rb, ib, lam, 8.0)):
        _near(got, want, torch.float32)
