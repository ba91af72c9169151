"""Each HIP kernel alone against its plain torch contract (tests/kernel_refs.py),
at sizes other than the engine's tiny models: widths and vocabularies that are no
power of two, head sizes in steps of 16 (and 24), odd head and group counts.
Shapes include those of the reference's own op tests (test/GPU/test_opr.cpp:9-119)."""
import math

import pytest
import torch

import kernel_refs as R

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


def ops():
    from inferllm_amd.kernels import ops as o
    return o


def tol(dtype):
    return (2e-5, 2e-5) if dtype == torch.float32 else (2e-2, 2e-2)


def close(got, want, dtype, scale=1.0):
    a, r = tol(dtype)
    assert got.shape == want.shape
    torch.testing.assert_close(got.double().cpu(), want.double().cpu(), atol=a * scale, rtol=r)


def rnd(*shape, dtype=torch.float32, seed=0, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * std).to(dtype)


def test_every_entry_point_is_declared_and_a_wrong_call_raises():
    """The loader gives each function of api.h its argument types: a call with too few arguments
    or with a float where a size is meant raises instead of launching on garbage."""
    import ctypes
    lib = ops()._lib()
    assert lib.illm_version.argtypes == [] and lib.illm_embed.argtypes[-1] is ctypes.c_void_p
    with pytest.raises(TypeError):
        lib.illm_silu_mul(None, None, 0, 4)
    with pytest.raises(ctypes.ArgumentError):
        lib.illm_silu_mul(None, None, 0, 4.5, 8, None)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("V,E,ids", [(10, 128, [1, 9, 3, 3]), (411, 80, [0, 410, 7]), (1000, 4100, [999])])
def test_embed(dtype, V, E, ids):
    table = rnd(V, E, dtype=dtype)
    t = torch.tensor(ids, dtype=torch.int32)
    got = ops().embed(t.to(DEV), table.to(DEV))
    assert torch.equal(got.cpu(), R.embed(t, table))       # rows are copied bit for bit


@pytest.mark.parametrize("out_dtype", DTYPES)
@pytest.mark.parametrize("w_dtype", DTYPES)
@pytest.mark.parametrize("T,E,eps", [(4, 4096, 1e-5), (3, 80, 1e-6), (1, 1001, 3e-2), (70, 96, 1e-5), (2, 6000, 1e-5), (2, 9000, 1e-5), (5, 1536, 1e-6)])
def test_add_rmsnorm(out_dtype, w_dtype, T, E, eps):
    x = rnd(T, E, seed=1) * 0.05            # small rows: eps matters
    w = (1 + rnd(E, seed=2) * 0.1).to(w_dtype)
    for delta_dtype in (None, torch.float32, torch.bfloat16):
        delta = None if delta_dtype is None else rnd(T, E, seed=3, std=0.05).to(delta_dtype)
        xr, xg = x.clone(), x.clone().to(DEV)
        want = R.add_rmsnorm(xr, delta, w, eps, out_dtype)
        got = ops().add_rmsnorm(xg, None if delta is None else delta.to(DEV), w.to(DEV), eps, out_dtype)
        close(got, want, out_dtype)
        close(xg, xr, torch.float32)          # the sum is written back
        if T > 2:
            idx = torch.tensor([T - 1, 0], dtype=torch.int32)
            xr2, xg2 = x.clone(), x.clone().to(DEV)
            want = R.add_rmsnorm(xr2, delta, w, eps, out_dtype, idx)
            got = ops().add_rmsnorm(xg2, None if delta is None else delta.to(DEV), w.to(DEV), eps,
                                    out_dtype, idx.to(DEV))
            close(got, want, out_dtype)
            assert torch.equal(xg2.cpu(), x)   # gathered rows leave x alone


@pytest.mark.parametrize("out_dtype", DTYPES)
@pytest.mark.parametrize("S,T,E", [(1, 3, 80), (3, 20, 96), (8, 64, 4096), (5, 17, 6000), (2, 3, 8196), (13, 4, 1536)])
def test_add_rmsnorm_adds_planes(out_dtype, S, T, E):
    """delta as the planes of a product whose K was split: their sum is added, in float32."""
    x = rnd(T, E, seed=1)
    w = (1 + rnd(E, seed=2) * 0.1).to(torch.bfloat16)
    planes = rnd(S, T, E, seed=3) * torch.linspace(0.5, 2.0, S)[:, None, None]
    xr, xg = x.clone(), x.clone().to(DEV)
    want = R.add_rmsnorm(xr, planes, w, 1e-5, out_dtype)
    got = ops().add_rmsnorm(xg, planes.to(DEV), w.to(DEV), 1e-5, out_dtype)
    close(got, want, out_dtype)
    close(xg, xr, torch.float32, scale=4.0)
    idx = torch.tensor([T - 1, 0, T // 2], dtype=torch.int32)
    xg2 = x.clone().to(DEV)
    got = ops().add_rmsnorm(xg2, planes.to(DEV), w.to(DEV), 1e-5, out_dtype, idx.to(DEV))
    close(got, R.add_rmsnorm(x.clone(), planes, w, 1e-5, out_dtype, idx), out_dtype)
    assert torch.equal(xg2.cpu(), x)


@pytest.mark.parametrize("T,E", [(129, 1028), (160, 2048), (256, 2052), (129, 4096), (257, 4092), (300, 4100), (512, 8192)])
def test_norm_of_a_row_among_129_to_512_and_among_more(T, E):
    """From 129 rows on, a row's normed values and its sum have the same bits whatever the number of rows."""
    many = 520
    x, w = rnd(many, E, seed=1), (1 + rnd(E, seed=2) * 0.1).to(DEV)
    for planes, dtype in ((0, torch.bfloat16), (1, torch.bfloat16), (3, torch.float32)):
        delta = rnd(planes, many, E, seed=3).to(dtype) if planes else None
        got = []
        for n in (T, many):
            xs = x[:n].contiguous().to(DEV)
            d = None if delta is None else delta[:, :n].contiguous().to(DEV)
            out = ops().add_rmsnorm(xs, d if planes != 1 else d[0], w, 1e-5, torch.float32)
            got.append((out, xs))
        assert torch.equal(got[0][0], got[1][0][:T]) and torch.equal(got[0][1], got[1][1][:T])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,F", [(4, 10), (5, 130), (3, 11008), (1, 173), (70, 64), (2, 2056)])
def test_silu_mul(dtype, T, F):
    gu = rnd(T, 2 * F, dtype=dtype, std=3.0)
    gu[0, 0] = 0.0; gu[0, 1] = -60.0; gu[0, 2] = 40.0
    close(ops().silu_mul(gu.to(DEV)), R.silu_mul(gu), dtype, scale=10)


def make_cache(n_pages, nkv, page, hd, dtype):
    return (torch.full((n_pages, nkv, page, hd), float("nan"), dtype=dtype),
            torch.full((n_pages, nkv, page, hd), float("nan"), dtype=dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,hd,rot,pairing", [(4, 2, 24, 24, 0), (3, 3, 16, 16, 1), (8, 1, 128, 128, 0),
                                                    (5, 5, 48, 32, 0), (2, 1, 256, 256, 1), (32, 8, 64, 64, 0), (3, 1, 48, 48, 0), (2, 2, 32, 16, 0)])
def test_rope_store(dtype, nh, nkv, hd, rot, pairing):
    from inferllm_amd.parts.position import rotary_table
    page, max_pos = 8, 64
    table = rotary_table(12345.0, rot, max_pos, "cpu")
    lens = [13, 1, 20]
    slots = [2, 0, 3]
    pos = [p for n in lens for p in range(n)]
    slot = [s for n, s in zip(lens, slots) for _ in range(n)]
    T = len(pos)
    qkv = rnd(T, (nh + 2 * nkv) * hd, dtype=dtype, seed=5)
    pt = torch.full((5, 4), 11, dtype=torch.int32)
    pt[2, :2] = torch.tensor([7, 3]); pt[0, :1] = 9; pt[3, :3] = torch.tensor([0, 5, 1])
    slot_len = torch.tensor([1, 0, 13, 20, 0], dtype=torch.int32)
    kc, vc = make_cache(12, nkv, page, hd, dtype)
    rp, rs = torch.tensor(pos, dtype=torch.int32), torch.tensor(slot, dtype=torch.int32)
    q_ref, kc_ref, vc_ref = qkv.clone(), kc.clone(), vc.clone()
    R.rope_store(q_ref, table, rot, pairing, rp, rs, slot_len, kc_ref, vc_ref, pt, page, 0, nh, nkv, hd)
    q_g, kc_g, vc_g = qkv.to(DEV), kc.to(DEV), vc.to(DEV)
    ops().rope_store(q_g, table.to(DEV), rot, pairing, rp.to(DEV), rs.to(DEV), slot_len.to(DEV),
                     kc_g, vc_g, pt.to(DEV), page, 0, nh, nkv, hd)
    close(q_g, q_ref, dtype, scale=4)
    for got, want in ((kc_g, kc_ref), (vc_g, vc_ref)):
        got, want = got.cpu(), want
        assert torch.equal(torch.isnan(got), torch.isnan(want))      # exactly the same rows are written
        close(torch.nan_to_num(got), torch.nan_to_num(want), dtype, scale=4)
    # position 0 leaves the row as it is
    first = [0, 13, 14]
    assert torch.equal(q_g.cpu()[first], qkv[first])


@pytest.mark.parametrize("dtype", DTYPES)
def test_rope_store_window_ring(dtype):
    """A ring of pages: rows that a later row of the same step overwrites are skipped."""
    nh, nkv, hd, page, ring = 2, 2, 16, 4, 3
    n = 23
    qkv = rnd(n, (nh + 2 * nkv) * hd, dtype=dtype, seed=9)
    pt = torch.tensor([[4, 2, 6]], dtype=torch.int32)
    slot_len = torch.tensor([n], dtype=torch.int32)
    rp = torch.arange(n, dtype=torch.int32); rs = torch.zeros(n, dtype=torch.int32)
    kc, vc = make_cache(8, nkv, page, hd, dtype)
    kr, vr = kc.clone(), vc.clone()
    R.rope_store(qkv.clone(), None, 0, 0, rp, rs, slot_len, kr, vr, pt, page, ring, nh, nkv, hd)
    kg, vg = kc.to(DEV), vc.to(DEV)
    ops().rope_store(qkv.to(DEV), None, 0, 0, rp.to(DEV), rs.to(DEV), slot_len.to(DEV), kg, vg,
                     pt.to(DEV), page, ring, nh, nkv, hd)
    assert torch.equal(torch.nan_to_num(kg.cpu()), torch.nan_to_num(kr))
    assert torch.equal(torch.nan_to_num(vg.cpu()), torch.nan_to_num(vr))
    # the last ring*page - (page - 1 - (n-1) % page) positions are there, e.g. position n-1
    view = qkv.view(n, nh + 2 * nkv, hd)
    assert torch.equal(kg.cpu()[int(pt[0, ((n - 1) // page) % ring]), :, (n - 1) % page], view[n - 1, nh:nh + nkv])


@pytest.mark.parametrize("xd,wd,yd", [(torch.float32,) * 3, (torch.bfloat16,) * 3,
                                      (torch.bfloat16, torch.bfloat16, torch.float32),
                                      (torch.bfloat16, torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("M,N,K", [(1, 2, 128), (4, 128, 128), (70, 411, 80), (65, 64, 1001), (3, 1000, 172)])
def test_gemm_generic(xd, wd, yd, M, N, K):
    x, w = rnd(M, K, dtype=xd, seed=1), rnd(N, K, dtype=wd, seed=2)
    got = ops().gemm_generic(x.to(DEV), w.to(DEV), yd)
    close(got, R.linear(x, w, yd), yd, scale=math.sqrt(K))


def test_gemm_generic_row_bits_do_not_depend_on_batch():
    x, w = rnd(70, 300, seed=1), rnd(130, 300, seed=2)
    whole = ops().gemm_generic(x.to(DEV), w.to(DEV), torch.float32).cpu()
    for r in (0, 17, 69):
        alone = ops().gemm_generic(x[r:r + 1].to(DEV), w.to(DEV), torch.float32).cpu()
        assert torch.equal(alone[0], whole[r])


def test_gemm_identity_and_linearity():
    x = rnd(5, 96, seed=3)
    eye = torch.eye(96)
    assert torch.equal(ops().gemm_generic(x.to(DEV), eye.to(DEV), torch.float32).cpu(), x)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,hd,lens,window", [
    (4, 4, 16, [7], 0), (4, 2, 24, [5, 11, 2], 0), (16, 16, 8, [2], 0), (32, 2, 128, [5, 70], 0),
    (3, 1, 48, [33, 64, 1, 100], 0), (2, 2, 256, [40], 0), (4, 2, 32, [90, 17], 13), (5, 5, 16, [130], 64)])
def test_attn_prefill(dtype, nh, nkv, hd, lens, window):
    T = sum(lens)
    qkv = rnd(T, (nh + 2 * nkv) * hd, dtype=dtype, seed=7)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    scale = 1.0 / math.sqrt(hd)
    got = ops().attn_prefill(qkv.to(DEV), cu.to(DEV), len(lens), max(lens), nh, nkv, hd, scale, window)
    want = R.attn_prefill(qkv, cu, len(lens), max(lens), nh, nkv, hd, scale, window)
    close(got, want, dtype, scale=2)


@pytest.mark.parametrize("nh,nkv,hd,lens,window", [
    (4, 4, 128, [300, 129, 128, 1], 0), (8, 1, 64, [257, 64], 0), (3, 3, 96, [200], 0), (6, 2, 32, [127, 130], 0),
    (2, 1, 160, [70], 0), (4, 2, 128, [400], 100), (2, 2, 64, [333, 5], 64), (5, 5, 224, [66], 0), (2, 2, 192, [129], 7),
    # head sizes that are no multiple of 32: the last block of dims is half used
    (4, 2, 80, [300, 129, 1], 0), (3, 1, 16, [200, 65], 0), (2, 2, 48, [333], 40), (6, 3, 112, [257], 0),
    (2, 1, 144, [130], 0), (1, 1, 240, [70, 3], 0), (2, 2, 176, [129], 9), (2, 1, 208, [64], 0),
    # more blocks than the chip holds at once (heaviest first, not paired), and a long sequence
    (32, 8, 128, [600, 130, 577, 64], 0), (2, 1, 128, [2500, 40], 0)])
def test_attn_prefill_mfma(nh, nkv, hd, lens, window):
    """The matrix-core kernels over several blocks of 128 query rows and tiles of 64 keys: the one
    with one LDS buffer, the one with two (head sizes up to 128), and the library's own choice."""
    dtype = torch.bfloat16
    T = sum(lens)
    qkv = rnd(T, (nh + 2 * nkv) * hd, dtype=dtype, seed=17)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    scale = 1.0 / math.sqrt(hd)
    want = R.attn_prefill(qkv, cu, len(lens), max(lens), nh, nkv, hd, scale, window)
    lib = ops()._lib()
    try:
        for which in (0, 2, 1):
            lib.illm_set_prefill_two_buffers(which)
            got = ops().attn_prefill(qkv.to(DEV), cu.to(DEV), len(lens), max(lens), nh, nkv, hd, scale, window)
            close(got, want, dtype, scale=2)
    finally:
        lib.illm_set_prefill_two_buffers(1)


@pytest.mark.parametrize("nh,nkv,hd,lens,window", [
    (4, 4, 128, [300, 129, 128, 1], 0), (8, 1, 64, [257, 64], 0), (3, 3, 96, [200], 0), (6, 2, 32, [127, 130], 0),
    (4, 2, 128, [400], 100), (2, 2, 64, [333, 5], 64), (2, 1, 32, [300], 7), (3, 1, 96, [31, 32, 33, 161], 33),
    (32, 8, 128, [600, 130, 577, 64], 0), (2, 1, 128, [1500, 40], 0)])
def test_attn_prefill_f32_matrix_cores(nh, nkv, hd, lens, window):
    """Float32 prompts with head sizes 32 to 128: the kernel on the matrix cores' float32
    instruction (blocks of 128 query rows, tiles of 32 keys) and the multiply-add kernel, both
    within the float32 budget of the plain implementation."""
    T = sum(lens)
    qkv = rnd(T, (nh + 2 * nkv) * hd, seed=19)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    scale = 1.0 / math.sqrt(hd)
    want = R.attn_prefill(qkv, cu, len(lens), max(lens), nh, nkv, hd, scale, window)
    lib = ops()._lib()
    try:
        for on in (1, 0):
            lib.illm_set_attn_f32_mfma(on)
            got = ops().attn_prefill(qkv.to(DEV), cu.to(DEV), len(lens), max(lens), nh, nkv, hd, scale, window)
            close(got, want, torch.float32, scale=2)
    finally:
        lib.illm_set_attn_f32_mfma(1)


def test_attn_prefill_f32_finds_one_far_key():
    """One early key is made to stand out for a late query of another block and wave: the
    output is that key's value; a query before the key does not see it."""
    nh, nkv, hd, n = 2, 1, 128, 700
    qkv = rnd(n, (nh + 2 * nkv) * hd, seed=3)
    view = qkv.view(n, nh + 2 * nkv, hd)
    view[37, nh] = view[650, 1] * 30
    cu = torch.tensor([0, n], dtype=torch.int32)
    got = ops().attn_prefill(qkv.to(DEV), cu.to(DEV), 1, n, nh, nkv, hd, 1.0, 0).cpu().view(n, nh, hd)
    torch.testing.assert_close(got[650, 1], view[37, nh + nkv], atol=1e-4, rtol=1e-4)
    assert not torch.allclose(got[30, 1], view[37, nh + nkv], atol=0.1)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,hd,starts,rows,page", [
    (4, 2, 32, [0, 70, 5], [40, 30, 1], 64), (8, 8, 128, [200, 0], [130, 64], 64), (3, 1, 48, [17, 64], [9, 200], 64),
    (6, 2, 24, [3], [5], 16), (2, 2, 256, [63], [66], 64), (32, 8, 128, [1000, 37, 0], [300, 27, 129], 64),
    (5, 5, 96, [130, 0], [131, 300], 32), (4, 1, 64, [31], [290], 16),
    (4, 2, 80, [70, 0], [200, 130], 64), (2, 1, 16, [5], [300], 64), (3, 3, 112, [129], [64], 128), (2, 1, 240, [64], [70], 64)])
def test_attn_prefill_paged(dtype, nh, nkv, hd, starts, rows, page):
    """A step's rows that go on from tokens the cache holds (a prompt cut into steps): attention
    over the paged cache at absolute positions, several sequences with different starts (0
    among them: a sequence that begins while others go on).  Stale rows of the pages are NaN."""
    lens = [s + r for s, r in zip(starts, rows)]
    pt, kc, vc, slots, _ = paged_case(dtype, nkv, hd, lens, page)
    for b, sl in enumerate(slots.tolist()):                    # rows beyond a sequence's end: NaN
        lp, r = divmod(lens[b], page)
        if r:
            kc[int(pt[sl, lp]), :, r:] = float("nan"); vc[int(pt[sl, lp]), :, r:] = float("nan")
    kc[-1] = float("nan"); vc[-1] = float("nan")
    T = sum(rows)
    qkv = rnd(T, (nh + 2 * nkv) * hd, dtype=dtype, seed=11)
    qkv[:, nh * hd:] = float("nan")                            # k and v come from the cache alone
    cu = torch.tensor([0] + list(torch.tensor(rows).cumsum(0)), dtype=torch.int32)
    st = torch.tensor(starts, dtype=torch.int32)
    scale = 1.0 / math.sqrt(hd)
    want = R.attn_prefill_paged(qkv, cu, slots, st, kc, vc, pt, page, 0, len(rows), max(rows), nh, nkv, hd,
                                scale, 0)
    lib = ops()._lib()
    try:
        # the library's own choice, and for bfloat16 the kernel with two LDS buffers forced
        # (head sizes 32 to 128 in steps of 32; the others do not have it)
        for which in ((1, 2) if dtype == torch.bfloat16 else (1,)):
            lib.illm_set_prefill_two_buffers(which)
            got = ops().attn_prefill_paged(qkv.to(DEV), cu.to(DEV), slots.to(DEV), st.to(DEV), kc.to(DEV),
                                           vc.to(DEV), pt.to(DEV), page, 0, len(rows), max(rows), nh, nkv, hd,
                                           scale, 0)
            assert torch.isfinite(got.float()).all()
            close(got, want, dtype, scale=2)
    finally:
        lib.illm_set_prefill_two_buffers(1)


def test_attn_prefill_paged_long_steps_with_a_window_ring():
    """Steps of 1,100 rows that go on from 1,500 and from 0 tokens (the kernel with two LDS buffers
    is the library's choice from 1,024 rows on): all keys, and a window of 500 keys over a ring of
    26 pages, which the longer sequence's 2,600 positions wrap round."""
    dtype, nh, nkv, hd, page = torch.bfloat16, 4, 2, 128, 64
    starts, rows = [1500, 0], [1100, 1030]
    lens = [s + r for s, r in zip(starts, rows)]
    qkv = rnd(sum(rows), (nh + 2 * nkv) * hd, dtype=dtype, seed=13)
    qkv[:, nh * hd:] = float("nan")
    cu = torch.tensor([0] + list(torch.tensor(rows).cumsum(0)), dtype=torch.int32)
    st = torch.tensor(starts, dtype=torch.int32)
    scale = 1.0 / math.sqrt(hd)
    for window, ring in ((0, 0), (500, 26)):
        pt, kc, vc, slots, _ = paged_case(dtype, nkv, hd, lens, page, ring=ring)
        got = ops().attn_prefill_paged(qkv.to(DEV), cu.to(DEV), slots.to(DEV), st.to(DEV), kc.to(DEV), vc.to(DEV),
                                       pt.to(DEV), page, ring, len(rows), max(rows), nh, nkv, hd, scale, window)
        want = R.attn_prefill_paged(qkv, cu, slots, st, kc, vc, pt, page, ring, len(rows), max(rows),
                                    nh, nkv, hd, scale, window)
        close(got, want, dtype, scale=2)


def test_attn_prefill_finds_one_far_key():
    """One early key is made to stand out for a late query: the output is that key's value."""
    nh, nkv, hd, n = 2, 1, 128, 700
    dtype = torch.bfloat16
    qkv = rnd(n, (nh + 2 * nkv) * hd, dtype=dtype, seed=3)
    view = qkv.view(n, nh + 2 * nkv, hd)
    view[37, nh] = view[650, 1].float().mul(30).to(dtype)          # key 37 matches query row 650, head 1
    cu = torch.tensor([0, n], dtype=torch.int32)
    got = ops().attn_prefill(qkv.to(DEV), cu.to(DEV), 1, n, nh, nkv, hd, 1.0, 0).cpu().view(n, nh, hd)
    close(got[650, 1], view[37, nh + nkv], dtype)
    assert not torch.allclose(got[30, 1].float(), view[37, nh + nkv].float(), atol=0.1)   # hidden from row 30


def paged_case(dtype, nkv, hd, lens, page, ring=0, seed=3):
    """Random cache contents laid out through a shuffled page table."""
    B = len(lens)
    per_seq = max((n + page - 1) // page for n in lens) if not ring else ring
    n_pages = B * per_seq + 3
    g = torch.Generator().manual_seed(seed)
    perm = torch.randperm(n_pages - 1, generator=g)[: B * per_seq].reshape(B, per_seq)
    pt = torch.full((B + 2, per_seq), n_pages - 1, dtype=torch.int32)
    slots = list(range(B, 0, -1))                    # slot numbers differ from batch order
    for b, s in enumerate(slots):
        pt[s] = perm[b].to(torch.int32)
    kc, vc = rnd(n_pages, nkv, page, hd, dtype=dtype, seed=seed + 1), rnd(n_pages, nkv, page, hd, dtype=dtype, seed=seed + 2)
    return pt, kc, vc, torch.tensor(slots, dtype=torch.int32), torch.tensor(lens, dtype=torch.int32)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,hd,lens,window,nsplit", [
    (4, 4, 16, [7], 0, 1), (4, 2, 24, [5, 11, 2], 0, 2), (32, 2, 128, [300, 70], 0, 3),
    (3, 1, 48, [33, 64, 1, 600], 0, 4), (2, 2, 256, [257], 0, 2), (4, 2, 32, [90, 17, 700], 13, 2),
    (5, 5, 16, [130, 520], 64, 5)])
def test_attn_decode(dtype, nh, nkv, hd, lens, window, nsplit):
    page = 16
    ring = 0
    if window:
        ring = (window + page - 2) // page + 1
    pt, kc, vc, slots, seq_len = paged_case(dtype, nkv, hd, lens, page, ring)
    B = len(lens)
    qkv = rnd(B, (nh + 2 * nkv) * hd, dtype=dtype, seed=11)
    scale = 1.0 / math.sqrt(hd)
    got = ops().attn_decode(qkv.to(DEV), kc.to(DEV), vc.to(DEV), pt.to(DEV), page, ring, slots.to(DEV),
                            seq_len.to(DEV), nh, nkv, hd, scale, window, nsplit)
    want = R.attn_decode(qkv, kc, vc, pt, page, ring, slots, seq_len, nh, nkv, hd, scale, window, nsplit)
    close(got, want, dtype, scale=2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nh,nkv,hd,lens,window", [(4, 2, 24, [1, 255, 256], 0), (6, 2, 256, [33, 512, 600], 0),
                                                   (3, 3, 120, [600, 90], 70)])
def test_one_range_of_keys_needs_no_merge(dtype, nh, nkv, hd, lens, window):
    """The general kernel as the only range of its sequence writes the result itself: the same bits as with
    further, empty ranges and a merge, where all keys are in the first 256 of a table that could hold more."""
    page = 16
    pt, kc, vc, slots, seq_len = paged_case(dtype, nkv, hd, lens, page)
    pt = torch.cat([pt, torch.full((pt.shape[0], 64), kc.shape[0] - 1, dtype=torch.int32)], dim=1)
    qkv = rnd(len(lens), (nh + 2 * nkv) * hd, dtype=dtype, seed=11)
    got = {n: ops().attn_decode(qkv.to(DEV), kc.to(DEV), vc.to(DEV), pt.to(DEV), page, 0, slots.to(DEV),
                                seq_len.to(DEV), nh, nkv, hd, 1.0 / math.sqrt(hd), window, n).cpu() for n in (1, 4)}
    for b, n in enumerate(lens):
        if n <= 256:
            assert torch.equal(got[1][b], got[4][b])
    want = R.attn_decode(qkv, kc, vc, pt, page, 0, slots, seq_len, nh, nkv, hd, 1.0 / math.sqrt(hd), window, 1)
    close(got[1], want, dtype, scale=2)


@pytest.mark.parametrize("nh,nkv,hd,lens,window,nsplit", [
    (32, 32, 128, [600, 1, 64, 65], 0, 1), (32, 8, 128, [300, 70], 0, 3), (4, 4, 16, [7, 200], 0, 2),
    (8, 1, 64, [1000], 0, 32), (6, 2, 24, [5, 11, 130], 0, 2), (16, 1, 256, [257, 31], 0, 2),
    (5, 5, 96, [130, 520], 70, 5), (12, 4, 32, [90, 17, 700], 13, 2), (3, 3, 8, [129], 0, 1),
    (20, 2, 48, [333], 0, 4), (64, 8, 128, [1000, 63], 0, 5), (32, 8, 64, [129], 0, 1), (6, 3, 96, [70, 700], 0, 3),
    (34, 2, 32, [200], 0, 2), (8, 2, 160, [90, 300], 50, 2), (10, 5, 224, [65], 0, 1),
    # long contexts, the most splits, both kernels (plain and grouped heads)
    (8, 8, 128, [8192, 16001], 0, 16), (16, 2, 128, [12000, 5], 0, 16)])
def test_attn_decode_bf16_pages_of_64(nh, nkv, hd, lens, window, nsplit):
    """The fast bfloat16 kernel (pages of 64 rows, as the engine's cache has them); stale rows
    of the pages are NaN and must not leak into the result."""
    dtype, page = torch.bfloat16, 64
    ring = (window + page - 2) // page + 1 if window else 0
    pt, kc, vc, slots, seq_len = paged_case(dtype, nkv, hd, lens, page, ring)
    for b, s in enumerate(slots.tolist()):
        n = lens[b]
        if not ring:
            lp, r = divmod(n, page)
            if r:
                kc[int(pt[s, lp]), :, r:] = float("nan"); vc[int(pt[s, lp]), :, r:] = float("nan")
    kc[-1] = float("nan"); vc[-1] = float("nan")
    B = len(lens)
    qkv = rnd(B, (nh + 2 * nkv) * hd, dtype=dtype, seed=11)
    scale = 1.0 / math.sqrt(hd)
    want = R.attn_decode(qkv, kc, vc, pt, page, ring, slots, seq_len, nh, nkv, hd, scale, window, nsplit)
    for waves in (1, 2, 3, 8):                  # waves of a block that share a key range
        got = ops().attn_decode(qkv.to(DEV), kc.to(DEV), vc.to(DEV), pt.to(DEV), page, ring, slots.to(DEV),
                                seq_len.to(DEV), nh, nkv, hd, scale, window, nsplit, waves)
        close(got, want, dtype, scale=2)


@pytest.mark.parametrize("nh,nkv,hd,lens,window,nsplit", [(32, 8, 128, [650, 90, 3000], 0, 4), (12, 4, 32, [90, 17, 700], 13, 2),
                                                          (64, 8, 128, [1000, 63], 0, 5), (34, 2, 64, [200, 129], 0, 1)])
def test_both_grouped_head_decode_kernels_agree(nh, nkv, hd, lens, window, nsplit):
    """Grouped heads up to head size 128 run with both products on the matrix cores; the kernel
    with P.V on the vector units (which larger head sizes still use) must give the same."""
    o = ops()
    dtype, page = torch.bfloat16, 64
    ring = (window + page - 2) // page + 1 if window else 0
    pt, kc, vc, slots, seq_len = paged_case(dtype, nkv, hd, lens, page, ring)
    qkv = rnd(len(lens), (nh + 2 * nkv) * hd, dtype=dtype, seed=11)
    args = (qkv.to(DEV), kc.to(DEV), vc.to(DEV), pt.to(DEV), page, ring, slots.to(DEV), seq_len.to(DEV),
            nh, nkv, hd, 1.0 / math.sqrt(hd), window, nsplit, 4)
    new = o.attn_decode(*args)
    try:
        o._lib().illm_set_gqa_pv_on_matrix_cores(0)
        old = o.attn_decode(*args)
    finally:
        o._lib().illm_set_gqa_pv_on_matrix_cores(1)
    want = R.attn_decode(qkv, kc, vc, pt, page, ring, slots, seq_len, nh, nkv, hd, 1.0 / math.sqrt(hd), window, nsplit)
    close(new, want, dtype, scale=2)
    close(old, want, dtype, scale=2)
    close(new, old.float(), dtype, scale=2)


def test_linear_add_over_a_short_k_in_one_piece_a_wave():
    """K up to 4096 with at most 512 tiles runs with 8 waves that each take their share of K at
    once; the looping variant sums in another order and must agree to rounding."""
    o = ops()
    for M, N, K in ((8, 4096, 4096), (16, 2048, 1024), (3, 520, 4096), (1, 8192, 2048)):
        x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
        nw = (1 + rnd(N, seed=4) * 0.3).to(torch.bfloat16)
        into = rnd(M, N, seed=3) * 10
        wc = _plain_copy(w.to(DEV))
        outs = []
        for on in (1, 0):
            try:
                o._lib().illm_set_skinny_one_shot(on)
                dev = into.clone().to(DEV)
                rows = o.linear_add(x.to(DEV), wc, dev, (nw.to(DEV), 1e-5))
            finally:
                o._lib().illm_set_skinny_one_shot(1)
            outs.append((dev, rows))
        want = into.double() + R.linear(x, w, torch.float64)
        for dev, rows in outs:
            torch.testing.assert_close(dev.double().cpu(), want, atol=2e-4 * math.sqrt(K), rtol=1e-5)
            close(rows.xb, want * nw.double(), torch.bfloat16, scale=float(want.abs().max()))
            torch.testing.assert_close(rows.ssq.double().sum(1).cpu(), (want ** 2).sum(1), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("ydt", DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 2, 128), (4, 128, 128), (8, 4096, 4096), (1, 32000, 4096), (16, 411, 80),
                                   (17, 100, 1000), (33, 64, 1008), (48, 31, 8), (64, 4096, 11008), (7, 12288, 4096),
                                   (64, 33, 40)])
def test_gemm_skinny(ydt, M, N, K):
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
    got = ops().gemm_skinny_bf16(x.to(DEV), w.to(DEV), ydt)
    close(got, R.linear(x, w, ydt), ydt, scale=math.sqrt(K))
    if ydt == torch.float32:       # float32 out keeps the accumulator: far tighter than bfloat16
        torch.testing.assert_close(got.double().cpu(), R.linear(x, w, torch.float64), atol=2e-4 * math.sqrt(K), rtol=1e-4)


@pytest.mark.parametrize("M,F,K", [(1, 11008, 4096), (8, 172, 64), (16, 200, 80), (3, 33, 1000), (40, 50, 64)])
def test_gate_up_silu(M, F, K):
    x = rnd(M, K, dtype=torch.bfloat16, seed=1)
    w = rnd(2 * F, K, dtype=torch.bfloat16, seed=2, std=0.2)
    got = ops().gate_up_silu(x.to(DEV), w.to(DEV))
    g, u = R.linear(x, w[:F], torch.float64), R.linear(x, w[F:], torch.float64)
    want = g / (1 + torch.exp(-g)) * u
    close(got, want, torch.bfloat16, scale=max(1.0, float(want.abs().max())))
    swapped = u / (1 + torch.exp(-u)) * g
    assert not torch.allclose(got.double().cpu(), swapped, atol=0.1 * float(want.abs().max()))


@pytest.mark.parametrize("ydt", DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (8, 100, 136), (16, 33, 1000), (5, 320, 96), (3, 7, 4), (9, 11008, 4096),
                                   (17, 100, 136), (64, 320, 96), (100, 33, 1000), (128, 4096, 512)])
def test_gemv_rows_f32(ydt, M, N, K):
    """The 32-bit path's product of few rows: float32 sums, W read once for every 16 rows; a
    row's result is the same bits whatever rows stand beside it."""
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    assert ops().gemv_rows_f32_fits(x.to(DEV), w.to(DEV))
    got = ops().gemv_rows_f32(x.to(DEV), w.to(DEV), ydt)
    want = R.linear(x, w, torch.float64)
    if ydt == torch.float32:
        torch.testing.assert_close(got.double().cpu(), want, atol=2e-6 * math.sqrt(K) * 4, rtol=1e-5)
    else:
        close(got, want, ydt, scale=math.sqrt(K))
    if ydt == torch.float32 and M > 1:
        alone = ops().gemv_rows_f32(x[M - 1:].contiguous().to(DEV), w.to(DEV), ydt)
        assert torch.equal(alone[0], got[M - 1])
    if K % 32 or M < ops().ROWS_F32_MFMA_FROM:
        assert torch.equal(ops().linear(x.to(DEV), w.to(DEV), ydt), got)
    assert not ops().gemv_rows_f32_fits(rnd(129, K).to(DEV), w.to(DEV))
    assert not ops().gemv_rows_f32_fits(x.to(DEV).to(torch.bfloat16), w.to(DEV))


@pytest.mark.parametrize("ydt", DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (8, 100, 160), (16, 33, 992), (5, 320, 96), (3, 7, 32), (9, 11008, 4096),
                                   (17, 100, 256), (64, 320, 96), (100, 33, 1024), (128, 4096, 512), (70, 16400, 64),
                                   (33, 22016, 4096)])
def test_gemm_rows_f32_mfma(ydt, M, N, K):
    """The 32-bit path's product of up to 128 rows on the matrix cores' float32 instruction:
    float32 accuracy, edges, one and two tiles of W a block with the same bits, and a row's result
    the same bits whatever rows stand beside it."""
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    assert ops().gemm_rows_f32_mfma_fits(x.to(DEV), w.to(DEV))
    got = ops().gemm_rows_f32_mfma(x.to(DEV), w.to(DEV), ydt)
    if M >= ops().ROWS_F32_MFMA_FROM:
        parted = ops().gemm_f32_split_pays(x.to(DEV), w.to(DEV))      # (`linear` has another kernel for large matrices)
        route = ops().gemm_f32_split(x.to(DEV), w.to(DEV), ydt) if parted else got
        assert torch.equal(ops().linear(x.to(DEV), w.to(DEV), ydt), route)
    want = R.linear(x, w, torch.float64)
    if ydt == torch.float32:
        torch.testing.assert_close(got.double().cpu(), want, atol=2e-6 * math.sqrt(K) * 4, rtol=1e-5)
    else:
        close(got, want, ydt, scale=math.sqrt(K))
    lib = ops()._lib()
    try:
        for tiles in (1, 2):
            lib.illm_set_rows_f32_tiles(tiles)
            assert torch.equal(ops().gemm_rows_f32_mfma(x.to(DEV), w.to(DEV), ydt), got)
    finally:
        lib.illm_set_rows_f32_tiles(0)
    if M > 1:
        alone = ops().gemm_rows_f32_mfma(x[M - 1:].contiguous().to(DEV), w.to(DEV), ydt)
        assert torch.equal(alone[0], got[M - 1])
    assert not ops().gemm_rows_f32_mfma_fits(rnd(129, K).to(DEV), w.to(DEV))
    assert not ops().gemm_rows_f32_mfma_fits(rnd(M, K + 16).to(DEV), rnd(N, K + 16).to(DEV))


@pytest.mark.parametrize("M,N,K,S", [(1, 64, 32, 1), (9, 1027, 2048, 1), (16, 130, 96, 3), (17, 4096, 64, 2), (33, 129, 224, 7),
                                     (65, 65, 160, 1), (96, 16400, 64, 1), (100, 500, 512, 4), (128, 1028, 992, 8),
                                     (129, 12288, 96, 1), (257, 300, 416, 2), (400, 7, 352, 1)])
def test_gemm_f32_split(M, N, K, S):
    """The float32 product in bfloat16 parts, whole and as planes: within the rounding of float32 sums (a sum of K / 32
    stages and a few more, each within 2^-23 of the sum of absolute products), edges of the tiles, a row's bits the
    same alone and among others, and infinities, NaN and the largest numbers as plain multiply-adds have them."""
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    xd, wd = x.to(DEV), w.to(DEV)
    assert ops().gemm_f32_split_fits(xd, wd)
    got = ops()._f32_split(xd, wd, torch.float32, S)
    whole = got.sum(0) if S > 1 else got
    bound = 2.0 ** -23 * (K / 32 + 16) * (x.double().abs() @ w.double().abs().t())
    assert bool(((whole.double().cpu() - R.linear(x, w, torch.float64)).abs() <= bound).all())
    alone = ops()._f32_split(xd[M - 1:].contiguous(), wd, torch.float32, S)
    assert torch.equal(alone[..., 0, :], got[..., M - 1, :])
    direct = ops().gemm_f32_split(xd, wd, torch.float32)          # with the library's own number of parts
    assert bool(((direct.double().cpu() - R.linear(x, w, torch.float64)).abs() <= bound).all())
    close(ops().gemm_f32_split(xd, wd, torch.bfloat16), R.linear(x, w, torch.float64), torch.bfloat16, scale=math.sqrt(K))
    x[0, 3], w[1, 5], w[N - 1, K - 1] = float("inf"), float("nan"), 3.4028e38
    got = ops().gemm_f32_split(x.to(DEV), w.to(DEV), torch.float32).cpu()
    want = ops().gemm_generic(x.to(DEV), w.to(DEV), torch.float32).cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert not ops().gemm_f32_split_fits(rnd(M, K + 16).to(DEV), rnd(N, K + 16).to(DEV))


@pytest.mark.parametrize("N,K", [(12288, 2048), (4096, 4096), (1024, 8192), (4098, 4096), (2048, 2048), (4096, 1024), (12288, 512), (1028, 2080)])
def test_f32_rows_alone_and_among_others(N, K):
    """A row of a float32 product has the same bits in steps of 9 to 128 rows, and in steps of more, with the parts of K
    as planes or one after the other: from `linear` and, where it takes them, as `linear_cut`'s planes added in order."""
    x, w = rnd(1100, K, seed=1).to(DEV), rnd(N, K, seed=2).to(DEV)
    for sizes in ((128, 9, 16, 17, 64, 65, 100), (1100, 129, 200, 257, 384, 500, 640, 900)):
        want = ops().linear(x[:sizes[0]].contiguous(), w)
        for M in sizes:
            rows = x[:M].contiguous()
            assert torch.equal(ops().linear(rows, w), want[:M])
            if ops().linear_cut_fits(rows, w):
                planes = ops().linear_cut(rows, w)
                got = planes[0].clone()
                for p in planes[1:]:
                    got += p
                assert torch.equal(got, want[:M])


@pytest.mark.parametrize("K", [64, 512])
@pytest.mark.parametrize("M,N", [(17, 130), (129, 68)])
def test_gemm_f32_split_over_the_range_of_float32(M, N, K):
    """The parts hold a float32 number exactly from the smallest normal one up: rows and matrices of any magnitude
    (beyond 2^104, and where the sums pass 2^80, by plain multiply-adds), subnormals among larger numbers, and operands
    of one sign whose left-out products of parts all add up.  Errors within what float32 sums of K products may
    have, 2^-24 for each addition of the sum of absolute products, and 2^-24 of it for what is left out."""
    g = torch.Generator().manual_seed(1)
    for ex, ew in ((0, 0), (-118, 0), (-124, 0), (-124, 100), (0, -122), (60, -125), (100, -100), (112, -100), (-100, 112), (60, 58)):
        x, w = torch.randn(M, K, generator=g).clamp(-4, 4) * 2.0 ** ex, torch.randn(N, K, generator=g).clamp(-4, 4) * 2.0 ** ew
        x[0, ::2] *= 2.0 ** -20
        got = ops().gemm_f32_split(x.to(DEV), w.to(DEV), torch.float32).double().cpu()
        bound = 2.0 ** -24 * (K + 1) * (x.double().abs() @ w.double().abs().t()) + 2.0 ** -148
        assert bool(((got - x.double() @ w.double().t()).abs() <= bound).all()), (ex, ew)
    one = torch.tensor([0x3f807fc0], dtype=torch.int32).view(torch.float32)
    x, w = one.expand(M, K).contiguous(), -one.expand(N, K).contiguous()
    want = x.double() @ w.double().t()
    err = lambda y: float(((y.double().cpu() - want) / want).abs().max())  # noqa: E731
    assert err(ops().gemm_f32_split(x.to(DEV), w.to(DEV), torch.float32)) <= 2.0 ** -24 * (K / 32 + 2)


def test_gemm_f32_split_in_pieces(monkeypatch):
    """Rows in pieces of at most so much scratch: the bits of one call, with the parts of K of all rows."""
    for M, N, K in ((300, 4098, 2048), (513, 130, 1056), (700, 12288, 512)):
        x, w = rnd(M, K, seed=1).to(DEV), rnd(N, K, seed=2).to(DEV)
        for dtype in DTYPES:
            want = ops()._f32_split(x, w, dtype, 1)
            monkeypatch.setattr(ops(), "F32_SPLIT_SCRATCH", 6 * K * 256)
            assert len(ops()._f32_split_pieces(M, K)) > 1
            assert torch.equal(ops()._f32_split(x, w, dtype, 1), want)
            monkeypatch.undo()


def test_gemm_f32_split_takes_no_longer_for_nan():
    """Sums that are no finite numbers are taken again on the float32 instruction: a prompt whose activations have all
    become NaN takes a few times as long as a sound one, not a hundred times."""
    x, w = rnd(256, 4096, seed=1).to(DEV), rnd(4096, 4096, seed=2).to(DEV)

    def least(f, rows):
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record(); f(rows, w, torch.float32); b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times[1:])
    bad = torch.full_like(x, float("nan"))
    assert ops().gemm_f32_split(bad, w, torch.float32).isnan().all()
    limit = 2 * least(ops().gemm_f32_mfma, x) + 2 * least(ops().gemm_f32_split, x)
    for rows in (bad, torch.full_like(x, float("inf")), torch.full_like(x, 3e38)):
        assert least(ops().gemm_f32_split, rows) <= limit
    x[7, 100] = float("nan")
    got = ops().gemm_f32_split(x, w, torch.float32)
    assert got[7].isnan().all() and int(got.isnan().sum()) == 4096


@pytest.mark.parametrize("M,N,K", [(1, 16, 32), (8, 24, 96), (3, 2048, 1056), (8, 2040, 4096), (7, 520, 2048), (5, 100, 1024),
                                   (8, 2048, 8192), (9, 2048, 1024), (16, 40, 64)])
def test_skinny_half_tiles_and_activations(M, N, K):
    """Products of up to 8 rows with half a tile a block (odd numbers of k-steps, a last tile of few rows, a block's waves
    more than its pieces) against whole tiles and 64 bits, a norm taken by the product, and activations on its sums."""
    x, w = rnd(M, K, seed=1).to(torch.bfloat16), rnd(N, K, seed=2).to(torch.bfloat16)
    tiled = ops().decode_weight(w.to(DEV), "plain", True)
    assert isinstance(tiled, ops().Weight)
    want = R.linear(x, w, torch.float64)
    bound = 2.0 ** -23 * (K / 32 + 32) * (x.double().abs() @ w.double().abs().t())
    lib = ops()._lib()
    acts = {"relu_squared": lambda t: t.clamp(min=0) ** 2,
            "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh")}
    normed = ops().NormedRows(x.float().to(DEV), torch.ones(K, device=DEV), 1e-5, torch.bfloat16, x.to(DEV),
                              (x.float() ** 2).view(M, K // 32, 32).sum(-1).contiguous().to(DEV))
    scale = torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5)
    try:
        for half in (0, 1, -1):
            lib.illm_set_skinny_half(half)
            got = ops().linear(x.to(DEV), tiled, torch.float32).double().cpu()
            assert bool(((got - want).abs() <= bound).all())
            got = ops().linear(normed, tiled, torch.float32).double().cpu()
            assert bool(((got - want * scale).abs() <= 2 * bound * scale + 1e-12).all())
            for name, act in acts.items():
                for rows in (x.to(DEV), normed):
                    z = want * (scale if rows is normed else 1.0)
                    close(ops().linear_act(rows, tiled, name), act(z), torch.bfloat16, scale=float(act(z).abs().max()))
                    close(ops().linear_act(rows, w.to(DEV), name), act(z), torch.bfloat16, scale=float(act(z).abs().max()))
    finally:
        lib.illm_set_skinny_half(-1)
    many = rnd(40, K, seed=3).to(torch.bfloat16).to(DEV)              # beyond the few rows: a kernel of its own
    assert torch.equal(ops().linear_act(many, tiled, "gelu_tanh"), ops().gelu_tanh(ops().linear(many, tiled)))


@pytest.mark.parametrize("N,K", [(2048, 8192), (2040, 4096), (512, 1056), (520, 2048), (1030, 2080), (64, 1024)])
def test_skinny_rows_alone_and_among_16(N, K):
    """A row's sums have the same bits in steps of 1 to 16 rows: with half a tile a block (up to 8 rows) as with whole
    ones, and as a norm's consumer."""
    x, w = rnd(16, K, seed=1).to(torch.bfloat16).to(DEV), rnd(N, K, seed=2).to(torch.bfloat16).to(DEV)
    tiled, nw = ops().decode_weight(w, "plain", True), torch.ones(K, device=DEV)
    ssq = (x.float() ** 2).view(16, K // 32, 32).sum(-1)
    want = ops().linear(x, tiled, torch.float32)
    lib = ops()._lib()
    normed = lambda M: ops().NormedRows(x[:M].float(), nw, 1e-5, torch.bfloat16, x[:M].contiguous(), ssq[:M].contiguous())
    want_normed = ops().linear(normed(16), tiled, torch.float32)
    try:
        for half in (1, 0, -1):
            lib.illm_set_skinny_half(half)
            for M in (1, 3, 7, 8, 9):
                assert torch.equal(ops().linear(x[:M].contiguous(), tiled, torch.float32), want[:M])
                assert torch.equal(ops().linear(normed(M), tiled, torch.float32), want_normed[:M])
    finally:
        lib.illm_set_skinny_half(-1)


@pytest.mark.parametrize("name", ["relu_squared", "gelu_tanh"])
@pytest.mark.parametrize("N,K", [(2048, 1056), (100, 1024), (4104, 96)])
def test_an_activation_in_the_product_and_behind_it(name, N, K):
    """`linear_act` of 1 to 16 rows: the same bits whatever their number, and no further from 64 bits than the product
    rounded to bfloat16 and the activation of that; more rows are those two."""
    x, w = rnd(20, K, seed=1).to(torch.bfloat16), rnd(N, K, seed=2, std=K ** -0.5).to(torch.bfloat16)
    z = x.double() @ w.double().t()
    want = z.clamp(min=0) ** 2 if name == "relu_squared" else torch.nn.functional.gelu(z, approximate="tanh")
    off = lambda y: float((y.double().cpu() - want[:len(y)]).norm())  # noqa: E731
    xd, act = x.to(DEV), getattr(ops(), name)
    for W in (w.to(DEV), ops().decode_weight(w.to(DEV), "plain", True)):
        whole = ops().linear_act(xd[:16].contiguous(), W, name)
        assert off(whole) <= off(act(ops().linear(xd[:16].contiguous(), W)))
        for M in (1, 5, 8, 9):
            assert torch.equal(ops().linear_act(xd[:M].contiguous(), W, name), whole[:M])
        rows = xd[:17].contiguous()
        assert torch.equal(ops().linear_act(rows, W, name), act(ops().linear(rows, W)))


@pytest.mark.parametrize("d,window,chunk,own", [(128, 0, 0, 1), (128, 0, 96, 0), (64, 70, 0, 0), (64, 0, 0, 1)])
def test_capped_prompt_alone_and_among_others(d, window, chunk, own):
    """A prompt's attention has the same bits whatever prompts stand beside it in the step."""
    nh, nkv, lens = 16, 4, [300] + [128] * 70
    T, B, page = sum(lens), len(lens), 64
    rows = rnd(T, (nh + 2 * nkv) * d, seed=1).to(torch.bfloat16).to(DEV)
    table = torch.arange(B * 5, dtype=torch.int32, device=DEV).view(B, 5)
    kc, vc = (rnd(B * 5, nkv, page, d, seed=s).to(torch.bfloat16).to(DEV) for s in (2, 3))
    got = []
    for n in (1, B):
        cu = torch.tensor([0] + torch.tensor(lens[:n]).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
        slot, start = torch.arange(n, dtype=torch.int32, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV)
        got.append(ops().attn_cap_rows(rows[:sum(lens[:n])].contiguous(), cu, slot, start, kc, vc, table, page, 0, n, 300, nh,
                                       nkv, d, d, d ** -0.5, 0.0, window, chunk=chunk,
                                       own=(nh * d, (nh + nkv) * d) if own else None))
    assert torch.equal(got[0], got[1][:300])


@pytest.mark.parametrize("d,window,chunk,keep", [(128, 50, 0, 70), (64, 0, 90, 0), (40, 33, 0, 0), (128, 0, 0, 0)])
def test_capped_prompt_over_pages_of_any_size(d, window, chunk, keep):
    """Rows over the cache (steps that go on from it, shuffled pages, kept pages, rings that have gone round) have the
    same bits whether pages are whole tiles of keys (64, 96: looked up once a tile) or not (20, 48), and are right."""
    nh, nkv, starts, lens = 4, 2, [0, 45, 500], [70, 33, 140]
    T, B = sum(lens), len(lens)
    g = torch.Generator().manual_seed(1)
    q = rnd(T, nh * d, seed=1).to(torch.bfloat16)
    k, v = (rnd(B, 640, nkv, d, seed=s).to(torch.bfloat16) for s in (2, 3))
    cu = torch.tensor([0, 70, 103, 243], dtype=torch.int32)
    slot, start = torch.tensor([2, 0, 1], dtype=torch.int32), torch.tensor(starts, dtype=torch.int32)
    gate = rnd(T, nh * d + 4, seed=4).to(torch.bfloat16)
    outs = []
    for page in (64, 96, 48, 20):
        kept = -(-keep // page)
        ring = -(-(140 + 50) // page) + 1 if window else 0
        per = kept + ring if ring else -(-640 // page)
        table = torch.randperm(B * per, generator=g).view(B, per).to(torch.int32)
        kc, vc = (torch.zeros(B * per, nkv, page, d, dtype=torch.bfloat16) for _ in range(2))
        for b in range(B):
            for pos in range(starts[b] + lens[b]):
                at, r = R.cache_offsets(table, int(slot[b]), pos, page, ring, kept)
                kc[at, :, r], vc[at, :, r] = k[b, pos], v[b, pos]
        args = (page, ring, B, max(lens), nh, nkv, d, d, d ** -0.5, 0.0, window)
        dev = [t.to(DEV) for t in (q, cu, slot, start, kc, vc, table)]
        outs.append(ops().attn_cap_rows(*dev, *args, chunk=chunk, keep=keep, kept=kept, gate=gate.to(DEV), gate_off=4).cpu())
    want = R.attn_cap_rows(q, cu, slot, start, kc, vc, table, *args, chunk=chunk, keep=keep, kept=kept, gate=gate, gate_off=4)
    close(outs[-1], want, torch.bfloat16)
    for got in outs[:-1]:
        assert torch.equal(got, outs[-1])


@pytest.mark.parametrize("dt,taps,shape", [(torch.bfloat16, 4, (2, 4, 8, 16)), (torch.float32, 3, (1, 2, 4, 36)), (torch.bfloat16, 2, (2, 2, 6, 20))])
def test_ssm_prepare_rows(dt, taps, shape):
    """A state-space mixer's inputs of prompts, four channels a thread, against the kernel of a channel a thread (which
    odd offsets still take): the same bits, sequences of 1 to 40 rows, tails of earlier steps."""
    G, H, N, dv = shape
    lens, C = [1, 2, 40, 3, 17], H * dv + 2 * G * N
    T = sum(lens)
    slot = torch.cat([torch.full((n,), 4 - i, dtype=torch.int32) for i, n in enumerate(lens)]).to(DEV)
    cols = rnd(T, C + H, seed=1)
    wide, odd = torch.zeros(T, C + H + 8), torch.zeros(T, C + H + 8)
    wide[:, 4:4 + C + H], odd[:, 3:3 + C + H] = cols, cols
    wide[:, 4 + C:4 + C + H], odd[:, 3 + C:3 + C + H] = cols[:, C:], cols[:, C:]
    tail = rnd(5, taps - 1, C, seed=2).to(dt).to(DEV)
    w, b, a, db = (t.to(DEV) for t in (rnd(C, taps, seed=3), rnd(C, seed=4), rnd(H, seed=5), rnd(H, seed=6)))
    run = lambda U, off: ops().ssm_prepare(U.to(dt).to(DEV), off, off + C, w, b, tail, slot, a, db, G, H, N, dv)
    for x, y in zip(run(wide, 4), run(odd, 3)):
        assert torch.equal(x, y)


@pytest.mark.parametrize("E", [4, 96, 1024, 1028, 4096, 8196, 33])
def test_embed_widths(E):
    """Rows of the table by four columns a thread, and one (E odd)."""
    for dt in DTYPES:
        table = rnd(50, E, seed=1).to(dt).to(DEV)
        ids = torch.tensor([0, 49, 7, 7, 60, -1], dtype=torch.int32, device=DEV)
        want = table[ids.long().clamp(0, 49)].float() * 0.5
        assert torch.equal(ops().embed(ids, table, 0.5), want)


def test_zero_slot():
    """A slot's row of every state tensor to zeros: 19 tensors (more than a launch takes), rows of 1 byte to 100 KB
    that begin on and off 16 bytes, and nothing beside them."""
    shapes = [(1,), (3,), (5, 7), (16,), (33,), (64, 129), (25000,), (2, 3, 4), (1021,)]
    ts = [torch.ones((4,) + sh, dtype=dt, device=DEV) for sh in shapes for dt in (torch.float32, torch.bfloat16)]
    ts.append(torch.ones((4, 17), dtype=torch.uint8, device=DEV))
    for slot in (0, 2, 3):
        for t in ts:
            t.fill_(1)
        ops().zero_slot(ts, slot)
        for t in ts:
            want = torch.ones_like(t)
            want[slot] = 0
            assert torch.equal(t, want)


@pytest.mark.parametrize("ydt", DTYPES)
@pytest.mark.parametrize("M,N,K", [(129, 128, 16), (130, 33, 48), (200, 411, 80), (257, 129, 1008), (1, 5, 32),
                                   (300, 1000, 4096), (2048, 130, 512)])
def test_gemm_f32_mfma(ydt, M, N, K):
    """The 32-bit path's product of many rows, on the matrix cores' float32 instruction: float32
    accuracy (a product with operands rounded to a shorter type would miss this budget by two
    orders), edges that are no multiple of the tile, and a row's result the same bits wherever
    it stands in the batch."""
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    assert ops().gemm_f32_mfma_fits(x.to(DEV), w.to(DEV))
    got = ops().gemm_f32_mfma(x.to(DEV), w.to(DEV), ydt)
    want = R.linear(x, w, torch.float64)
    if ydt == torch.float32:
        torch.testing.assert_close(got.double().cpu(), want, atol=2e-6 * math.sqrt(K) * 4, rtol=1e-5)
    else:
        close(got, want, ydt, scale=math.sqrt(K))
    if ydt == torch.float32 and M > 2:
        part = ops().gemm_f32_mfma(x[M // 2 + 1:].contiguous().to(DEV), w.to(DEV), ydt)
        assert torch.equal(part, got[M // 2 + 1:])
    if M > 128:
        assert torch.equal(ops().linear(x.to(DEV), w.to(DEV), ydt), got)
    assert not ops().gemm_f32_mfma_fits(rnd(M, K + 8).to(DEV), rnd(N, K + 8).to(DEV))
    assert not ops().gemm_f32_mfma_fits(x.to(DEV).to(torch.bfloat16), w.to(DEV))


@pytest.mark.parametrize("M,N,K", [(1, 1, 16), (64, 64, 32), (65, 129, 48), (129, 64, 64), (192, 520, 80), (130, 1030, 112),
                                   (257, 65, 4096)])
def test_gemm_f32_mfma_tiles(M, N, K):
    """Both block sizes of the many-row float32 product and its kernel of short K (16) give the same bits, at edges of
    their tiles, of a stage of 32 k and of the eight column tiles that go round the chip; against 64 bits within
    sums of K products in any order (each within K 2^-24 of the sum of their magnitudes)."""
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    want = x.double() @ w.double().t()
    room = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    got = []
    lib = ops()._lib()
    try:
        for tile in (16, 64, 128):
            lib.illm_set_f32_tile(tile)
            got.append(ops().gemm_f32_mfma(x.to(DEV), w.to(DEV), torch.float32))
    finally:
        lib.illm_set_f32_tile(0)
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
    assert bool(((got[0].double().cpu() - want).abs() <= room).all())


@pytest.mark.parametrize("nh,nkv,lens", [(8, 8, [70, 1, 200]), (16, 2, [129, 40]), (5, 5, [3, 300, 64, 130]), (12, 4, [128, 127])])
def test_attn_prefill_ragged_batches(nh, nkv, lens):
    """Every (sequence, head) pair of a ragged batch is worked on once, whether 8 divides the heads (an
    XCD takes the same heads of every sequence) or not: each sequence's rows are the bits of the
    sequence alone."""
    hd, T = 64, sum(lens)
    qkv = rnd(T, (nh + 2 * nkv) * hd, seed=3).to(torch.bfloat16).to(DEV)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    got = ops().attn_prefill(qkv, i32(cu), len(lens), max(lens), nh, nkv, hd, 0.125, 0)
    close(got, R.attn_prefill(qkv.cpu(), torch.tensor(cu), len(lens), max(lens), nh, nkv, hd, 0.125, 0), torch.bfloat16)
    for a, b in zip(cu, cu[1:]):
        alone = ops().attn_prefill(qkv[a:b].contiguous(), i32([0, b - a]), 1, b - a, nh, nkv, hd, 0.125, 0)
        assert torch.equal(got[a:b], alone)


@pytest.mark.parametrize("T,E,F,NE,top,act", [(1, 64, 64, 2, 1, "silu"), (9, 128, 192, 4, 2, "clamped_swish"), (129, 192, 64, 1, 1, "silu"),
                                              (300, 64, 320, 3, 2, "silu"), (257, 256, 128, 2, 2, "relu_squared"), (40, 448, 64, 5, 5, "silu")])
def test_moe_tiles_of_128_pairs(T, E, F, NE, top, act):
    """The experts' products in tiles of up to 128 pairs give the bits of the kernel for 16 pairs (the same
    products summed over k in the same order), at tiles of one row, whole ones and remainders, column
    blocks that are not full, with and without gates and weights on the input."""
    o = ops()
    gated = act != "relu_squared"
    g = torch.Generator().manual_seed(5)
    h = rnd(T, E, dtype=torch.bfloat16, seed=1).to(DEV)
    wu = (rnd(NE, F * (2 if gated else 1), E, seed=2) * 0.1).to(torch.bfloat16).to(DEV)
    wd = (rnd(NE, E, F, seed=3) * 0.1).to(torch.bfloat16).to(DEV)
    idx = torch.stack([torch.randperm(NE, generator=g)[:top] for _ in range(T)]).to(torch.int32).to(DEV)
    wt = torch.rand(T, top, generator=g).to(DEV) if act == "clamped_swish" else None
    real, got = o._moe_tiling, []
    try:
        for rows in (16, 128):
            o._moe_tiling = lambda dtype, e, f, np, n: (True, rows, max(1, min(np, np // rows + n)))
            got.append(o.moe_experts(h, idx, wu, wd, None, act, 7.0 if act == "clamped_swish" else 0.0, wt))
    finally:
        o._moe_tiling = real
    assert torch.equal(got[0], got[1]) and bool(torch.isfinite(got[1].float()).all())
    assert real(torch.bfloat16, E, F, 24 * NE, NE)[1] == 128 and real(torch.bfloat16, E, F + 32, 24 * NE, NE)[1] != 128


@pytest.mark.parametrize("T,E,F,NE,top,act", [(1, 64, 64, 2, 1, "silu"), (193, 192, 320, 1, 1, "clamped_swish"), (400, 448, 128, 3, 2, "silu"),
                                              (385, 128, 192, 2, 2, "relu_squared"), (130, 64, 576, 5, 5, "silu")])
def test_moe_tiles_of_192_pairs(T, E, F, NE, top, act):
    """Tiles of up to 192 pairs in turns of two groups of waves give the bits of the kernel for 16 pairs: one stage of
    64 k, odd and even numbers of them, tiles of one row, whole ones and remainders, columns that end inside a block."""
    o = ops()
    gated = act != "relu_squared"
    g = torch.Generator().manual_seed(6)
    h = rnd(T, E, dtype=torch.bfloat16, seed=1).to(DEV)
    wu = (rnd(NE, F * (2 if gated else 1), E, seed=2) * 0.1).to(torch.bfloat16).to(DEV)
    wd = (rnd(NE, E, F, seed=3) * 0.1).to(torch.bfloat16).to(DEV)
    idx = torch.stack([torch.randperm(NE, generator=g)[:top] for _ in range(T)]).to(torch.int32).to(DEV)
    wt = torch.rand(T, top, generator=g).to(DEV) if act == "clamped_swish" else None
    real, got = o._moe_tiling, []
    try:
        for rows in (16, 192):
            o._moe_tiling = lambda dtype, e, f, np, n: (True, rows, max(1, min(np, np // rows + n)))
            got.append(o.moe_experts(h, idx, wu, wd, None, act, 7.0 if act == "clamped_swish" else 0.0, wt))
    finally:
        o._moe_tiling = real
    assert torch.equal(got[0], got[1]) and bool(torch.isfinite(got[1].float()).all())
    wide = lambda per, n: o._moe_wide(2048, 1408, per * n, n)  # noqa: E731
    assert [wide(*c) for c in ((24, 64), (111, 64), (112, 64), (112, 8), (400, 8))] == [False, False, True, False, False]


@pytest.mark.parametrize("T,E,F,NE,top,act", [(8, 64, 64, 9, 1, "silu"), (17, 192, 96, 8, 2, "clamped_swish"), (90, 64, 320, 3, 2, "relu_squared"),
                                              (12, 2048, 64, 16, 3, "silu"), (20, 4160, 64, 9, 2, "relu_squared")])
def test_moe_products_of_few_tokens_by_whole_lines(T, E, F, NE, top, act):
    """Experts' products of 8 tiles and more of up to 16 pairs, read by whole lines, give a token the bits that it has
    alone, where fewer tiles go to the kernel that reads 64 bytes of 16 rows: one step of 64 k and odd numbers of them,
    full tiles and tiles of one pair, columns that end inside a block, 8 and 16 columns a wave."""
    o, gated = ops(), act != "relu_squared"
    g = torch.Generator().manual_seed(5)
    h = rnd(T, E, dtype=torch.bfloat16, seed=1).to(DEV)
    wu = (rnd(NE, F * (2 if gated else 1), E, seed=2) * 0.1).to(torch.bfloat16).to(DEV)
    wd = (rnd(NE, E, F, seed=3) * 0.1).to(torch.bfloat16).to(DEV)
    idx = torch.stack([torch.randperm(NE, generator=g)[:top] for _ in range(T)]).to(torch.int32).to(DEV)
    wt = torch.rand(T, top, generator=g).to(DEV) if act == "clamped_swish" else None
    real, lim = o._moe_tiling, 7.0 if act == "clamped_swish" else 0.0
    try:
        o._moe_tiling = lambda dtype, e, f, np, n: (True, 16, max(1, min(np, np // 16 + n)))
        assert min(T * top, T * top // 16 + NE) >= 8 > top
        got = o.moe_experts(h, idx, wu, wd, None, act, lim, wt).view(T, top, E)
        for t in range(T):
            alone = o.moe_experts(h[t:t + 1], idx[t:t + 1], wu, wd, None, act, lim, None if wt is None else wt[t:t + 1])
            assert torch.equal(got[t], alone)
    finally:
        o._moe_tiling = real
    assert bool(torch.isfinite(got.float()).all())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("E", [1024, 1032, 2048, 2056, 4104])
def test_moe_combine_of_wide_rows(E, dtype):
    """Rows around a block's columns (1,024 in float32, 2,048 in bfloat16): with few tokens several blocks a token, the
    same bits as among 129, where one block walks them all."""
    o, T, top = ops(), 129, 3
    h, y, sh = (rnd(n, E, dtype=dtype, seed=i).to(DEV) for i, n in enumerate((T, T * top, T)))
    sg, g = rnd(E, seed=4).to(DEV), torch.Generator().manual_seed(5)
    idx, wt = torch.randint(0, 5, (T, top), generator=g).to(torch.int32), torch.rand(T, top, generator=g)
    every = o.moe_combine(h, idx.to(DEV), wt.to(DEV), y, 4, sh, sg)
    some = o.moe_combine(h[:128], idx[:128].to(DEV), wt[:128].to(DEV), y[:128 * top], 4, sh[:128], sg)
    assert torch.equal(some, every[:128])
    d = lambda t: t.double().cpu()  # noqa: E731
    rows = torch.where((idx < 4)[:, :, None], d(y).view(T, top, E), d(h)[:, None])
    want = (rows * wt.double()[:, :, None]).sum(1) + torch.sigmoid(d(h) @ d(sg))[:, None] * d(sh)
    assert float((d(every) - want).abs().max()) <= (E + 200) * 2.0 ** -24 * float(want.abs().max())


@pytest.mark.parametrize("dtype", DTYPES)
def test_moe_combine_of_views_that_begin_anywhere(dtype):
    """The weighted sum reads 16 bytes at a time only from addresses that are multiples of 16: views that begin
    elsewhere (by column, a gate's sum in another order) are as close to 64 bits."""
    o, T, E, top = ops(), 5, 64, 3
    h, y, sh, sg = rnd(T, E, dtype=dtype, seed=1), rnd(T * top, E, dtype=dtype, seed=2), rnd(T, E, dtype=dtype, seed=3), rnd(E, seed=4)
    idx = torch.randint(0, 5, (T, top), generator=torch.Generator().manual_seed(5)).to(torch.int32)
    wt = torch.rand(T, top, generator=torch.Generator().manual_seed(6))
    rows = torch.where((idx < 4)[:, :, None], y.double().view(T, top, E), h.double()[:, None])
    want = (rows * wt.double()[:, :, None]).sum(1) + torch.sigmoid(h.double() @ sg.double())[:, None] * sh.double()

    def off(t):
        return torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:].view(t.shape).copy_(t)
    on = [t.to(DEV) for t in (h, y, sh)]
    for k in range(4):
        a, b, c = [off(t) if i == k else t for i, t in enumerate(on)]
        got = o.moe_combine(a, idx.to(DEV), wt.to(DEV), b, 4, c, sg.to(DEV)).double().cpu()
        # a sum of 64 products through a sigmoid, five more products: a few hundred roundings of 2^-24
        assert float((got - want).abs().max()) <= 300 * 2.0 ** -24 * float(want.abs().max())


def test_moe_experts_of_views_that_begin_anywhere():
    """Rows and experts' matrices whose first element is no multiple of 16 bytes give the bits of copies that are,
    with the pairs grouped beforehand and not."""
    o, T, E, F, NE, top = ops(), 130, 128, 192, 3, 2
    h, wu, wd = (rnd(*s, dtype=torch.bfloat16, seed=i).to(DEV) * 0.3 for i, s in enumerate([(T, E), (NE, 2 * F, E), (NE, E, F)]))
    idx = torch.stack([torch.randperm(NE)[:top] for _ in range(T)]).to(torch.int32).to(DEV)
    want = o.moe_experts(h, idx, wu, wd)

    def off(t):
        v = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:].view(t.shape)
        return v.copy_(t)
    plan = o._moe_group(idx, NE, h.dtype, E, F)
    assert plan[3] == 128 and o._moe_group(idx, NE, h.dtype, E, F, False)[3] == 64
    for a, b, c in ((off(h), wu, wd), (h, off(wu), wd), (h, wu, off(wd))):
        assert torch.equal(o.moe_experts(a, idx, b, c), want)
        assert torch.equal(o.moe_experts(a, idx, b, c, plan), want)


@pytest.mark.parametrize("xdt", DTYPES)
@pytest.mark.parametrize("T,NE,K", [(1, 1, 4), (8, 64, 2048), (9, 65, 2052), (16, 7, 6144), (17, 33, 260), (100, 64, 512)])
def test_few_outputs_rows(xdt, T, NE, K):
    """A router's product at the edges of its two kernels (up to 16 tokens, eight turns of 256 k; 8 tokens a block,
    4 outputs a wave); float32 sums in any order (K 2^-24 of the sum of magnitudes)."""
    x, w = rnd(T, K, dtype=xdt, seed=1), rnd(NE, K, seed=2)
    got = ops().few_outputs_f32(x.to(DEV), w.to(DEV)).double().cpu()
    room = (K + 8) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert bool(((got - x.double() @ w.double().t()).abs() <= room).all())


@pytest.mark.parametrize("xdt", DTYPES)
@pytest.mark.parametrize("NE,K", [(64, 2048), (7, 6144), (33, 260), (5, 4), (65, 2050), (3, 61)])
def test_few_outputs_of_a_row_alone_and_among_others(xdt, NE, K):
    """A row's sums are the same bits alone, among 16 (the most of one kernel), 17 and 100 rows: a token's
    near-tied experts don't hang on its company."""
    x, w = rnd(100, K, dtype=xdt, seed=1).to(DEV), rnd(NE, K, seed=2).to(DEV)
    every = ops().few_outputs_f32(x, w)
    for T in (1, 2, 3, 15, 16, 17, 99):
        for at in (0, 100 - T):
            assert torch.equal(ops().few_outputs_f32(x[at:at + T].contiguous(), w), every[at:at + T]), (T, at)


def test_moe_route_places():
    """The choice by places: ties go to the lower index, as in the search that odd scores (not finite, or
    more than 64 outputs) take; weights are the scores."""
    o = ops()
    for NE in (1, 5, 64, 65):
        z = (rnd(50, NE, seed=4) * 2).round().div(2).to(DEV)                 # many equal scores
        want = torch.sort(torch.softmax(z.double().cpu(), -1).float(), dim=-1, descending=True, stable=True)
        for top in sorted({1, min(3, NE), min(4, NE), min(6, NE)}):          # (3 of 64: searches, 4: places)
            idx, wt = o.moe_route(z, None, top)
            assert torch.equal(idx.long().cpu(), want.indices[:, :top])
            torch.testing.assert_close(wt.cpu(), want.values[:, :top], atol=0, rtol=1e-5)


@pytest.mark.parametrize("rule", ["plain", "delta", "bonus", "removal"])
@pytest.mark.parametrize("G,H,dk,dv,vector", [(2, 4, 128, 20, False), (3, 3, 40, 17, True), (1, 1, 5, 3, False), (2, 2, 17, 16, True),
                                              (1, 2, 130, 33, True)])
def test_gated_scan_chunks(rule, G, H, dk, dv, vector):
    """The recurrences for long runs: chunks of 8 tokens that end anywhere, blocks of 16 columns that are
    not full, every count of rows a part, a decay a row or one for all; against a plain walk in 64 bits
    (2,000 roundings of sums of a few units), and a run in two steps leaves the same bits."""
    if rule == "removal":
        G = H
    lens = [16, 17, 33, 3, 24]
    T = sum(lens)
    q, k, v = rnd(T, G, dk, seed=1) * dk ** -0.5, rnd(T, G, dk, seed=2) * dk ** -0.5, rnd(T, H, dv, seed=3)
    g = torch.Generator().manual_seed(4)
    beta, dec = torch.rand(T, H, generator=g), torch.rand(T, H, dk if vector else 1, generator=g) * 0.4 + 0.6
    rem = rnd(T, H, dk, seed=5) * dk ** -0.5 if rule == "removal" else None
    start = rnd(len(lens), H, dk, dv, seed=6) * 0.5
    want, r = torch.zeros(T, H, dv, dtype=torch.float64), 0
    S = start.double().clone()
    for b, n in enumerate(lens):
        for t in range(r, r + n):
            kk, qq = k[t].double().repeat_interleave(H // G, 0), q[t].double().repeat_interleave(H // G, 0)
            vt, bt, gt = v[t].double(), beta[t].double()[:, None], dec[t].double()[:, :, None]
            if rule == "bonus":
                want[t] = (S[b] * qq[:, :, None]).sum(1) + bt * vt
                S[b] = S[b] * gt + kk[:, :, None] * vt[:, None]
                continue
            if rule == "removal":
                read = bt * (S[b] * kk[:, :, None]).sum(1)
                S[b] = S[b] * gt + kk[:, :, None] * vt[:, None] - rem[t].double()[:, :, None] * read[:, None]
            else:
                S[b] = S[b] * gt
                u = bt * (vt - ((S[b] * kk[:, :, None]).sum(1) if rule == "delta" else 0.0))
                S[b] = S[b] + kk[:, :, None] * u[:, None]
            want[t] = (S[b] * qq[:, :, None]).sum(1)
        r += n

    def run(spans, states):
        """the rows `spans` (begin, end) of every sequence, its state in `states`"""
        rows = torch.cat([torch.arange(a, b) for a, b in spans])
        cu = [0]
        for a, b in spans:
            cu.append(cu[-1] + b - a)
        i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
        d = [x[rows].contiguous().to(DEV) if x is not None else None for x in (q, k, v, beta, dec, rem)]
        o = torch.empty(len(rows), H, dv, device=DEV)
        lib, p = ops()._lib(), ops()._p
        assert lib.illm_gated_scan(p(d[0]), p(d[1]), p(d[2]), p(d[3]), p(d[4]), dec.shape[2], p(states), p(i32(cu)),
                                   p(i32(list(range(len(lens))))), p(o), len(lens), max(max(b - a for a, b in spans), 16), G, H, dk, dv,
                                   {"plain": 0, "delta": 1, "bonus": 2, "removal": 0}[rule], p(d[5]), ops()._stream()) == 0
        return o.cpu()

    ends = [sum(lens[:i + 1]) for i in range(len(lens))]
    spans = [(e - n, e) for e, n in zip(ends, lens)]
    whole = start.clone().to(DEV)
    got = run(spans, whole)
    scale = want.abs().max()
    assert float((got.double() - want).abs().max() / scale) < 2000 * 2.0 ** -24
    assert float((whole.double().cpu() - S).abs().max() / S.abs().max()) < 2000 * 2.0 ** -24
    halves = start.clone().to(DEV)
    cuts = [(a, a + (b - a) // 2) for a, b in spans]
    first, second = run(cuts, halves), run([(m, b) for (_, m), (_, b) in zip(cuts, spans)], halves)
    assert torch.equal(halves, whole)
    assert torch.equal(torch.cat([first[:cuts[0][1]], second[:lens[0] - cuts[0][1]]]), got[:lens[0]])


def _decode_copy(w, mode="plain", **geometry):
    o = ops()
    return o.Weight(w, o.tile_weight(w, o.tile_rows(w.shape[0], mode, **geometry)), mode)


def test_tile_rows_cover_every_row_once():
    o = ops()
    for rows, N in ((o.tile_rows(100), 100), (o.tile_rows(2 * 44, "gate_up"), 88),
                    (o.tile_rows((6 + 2 * 3) * 48, "qkv", nh=6, nkv=3, hd=48), 12 * 48)):
        assert rows.shape[1] == 16
        kept = rows[rows >= 0]
        assert sorted(kept.tolist()) == list(range(N))
    g = o.tile_rows(2 * 44, "gate_up")
    assert g[5, :8].tolist() == [40, 41, 42, 43, -1, -1, -1, -1] and g[5, 8:12].tolist() == [84, 85, 86, 87]
    q = o.tile_rows((2 + 2) * 32, "qkv", nh=2, nkv=1, hd=32)
    assert q[1].tolist() == list(range(8, 16)) + list(range(24, 32))          # a row and its partner hd/2 on
    assert q[-1].tolist() == list(range(3 * 32 + 16, 4 * 32))                  # v: 16 rows in a run


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (8, 100, 160), (16, 33, 992), (5, 320, 96), (9, 4096, 11008),
                                   (8, 16400, 64)])      # 1025 tiles: two a block, the last block has one
def test_products_from_the_decode_copy_equal_those_from_the_matrix(M, N, K, monkeypatch):
    """The copy laid out for the few-rows kernels holds the same numbers in another order: with
    K cut over the same number of waves the products are the same sums in the same order, bit
    for bit."""
    o = ops()
    for knob in ("PLAIN_WAVES", "GATE_UP_WAVES", "QKV_ROPE_WAVES"):
        monkeypatch.setattr(o, knob, 3)
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1).to(DEV), rnd(N, K, dtype=torch.bfloat16, seed=2).to(DEV)
    wc = _decode_copy(w)
    assert wc.tiled.shape == ((N + 15) // 16, K // 32, 16, 32)
    for ydt in DTYPES:
        assert torch.equal(o.linear(x, wc, ydt), o.linear(x, w, ydt))
    into_a, into_b = rnd(M, N, seed=3).to(DEV), rnd(M, N, seed=3).to(DEV)
    nw = (1 + rnd(N, seed=4) * 0.3).to(torch.bfloat16).to(DEV)
    ra, rb = o.linear_add(x, wc, into_a, (nw, 1e-5)), o.linear_add(x, w, into_b, (nw, 1e-5))
    assert torch.equal(into_a, into_b)
    if ra is not None:
        assert torch.equal(ra.xb, rb.xb) and torch.equal(ra.ssq, rb.ssq)
        w2 = rnd(48, N, dtype=torch.bfloat16, seed=5).to(DEV)
        if N % 32 == 0:
            assert torch.equal(o.linear(ra, _decode_copy(w2)), o.linear(rb, w2))
    if K % 64 == 0:                                        # gate|up: N rows as two halves
        for F in (56, 8200):                               # 8200: 1025 tiles, two a block
            wg = rnd(2 * F, K, dtype=torch.bfloat16, seed=6, std=0.2).to(DEV)
            assert torch.equal(o.gate_up_silu(x, _decode_copy(wg, "gate_up")), o.gate_up_silu(x, wg))
    xl = rnd(17, K, dtype=torch.bfloat16, seed=7).to(DEV)     # more rows: the matrix itself is read
    assert torch.equal(o.linear(xl, wc), o.linear(xl, w))
    # a copy that follows another kernel's tiles is never read by the plain product
    if N % 2 == 0 and K % 64 == 0:
        other = _decode_copy(w, "gate_up")
        assert not torch.equal(other.tiled.view(-1)[: 16 * K], wc.tiled.view(-1)[: 16 * K]) or N <= 16
        assert torch.equal(o.linear(x, other), o.linear(x, w))


def test_products_of_many_rows_follow_the_plan_and_stay_right(monkeypatch):
    """A product of many rows runs whole or cut along its output columns as the plan's table
    says; a plan that measures times the candidates once per shape; whatever plan is taken,
    every element is the plain product."""
    o = ops()
    from inferllm_amd.kernels.plan import Plan
    M, N, K = 1100, 9000, 64
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
    fixed = Plan()
    monkeypatch.setattr(o, "_plan", fixed)
    whole = o.linear(x.to(DEV), w.to(DEV))
    assert not fixed.cuts                                  # no table entry: whole, nothing timed
    assert torch.equal(whole, torch.matmul(x.to(DEV), w.to(DEV).t()))
    fixed.cuts[(-(-M // 256), N, K)] = (4096,)
    cut = o.linear(x.to(DEV), w.to(DEV))
    close(cut, R.linear(x, w), torch.bfloat16, scale=math.sqrt(K))
    assert torch.equal(cut[:, :4096], torch.matmul(x.to(DEV), w.to(DEV)[:4096].t()))
    plan = Plan(measure=True)
    monkeypatch.setattr(o, "_plan", plan)
    got = o.linear(x.to(DEV), w.to(DEV))
    key = (-(-M // 256), N, K)
    assert key in plan.cuts and len(plan.cuts) == 1
    close(got, R.linear(x, w), torch.bfloat16, scale=math.sqrt(K))
    for cand in o._split_candidates(N):                    # every candidate gives the product
        assert all(0 < c < N for c in cand)
        close(o._run_plan(x.to(DEV), w.to(DEV), cand), R.linear(x, w), torch.bfloat16, scale=math.sqrt(K))
    big = rnd(2048, K, dtype=torch.bfloat16, seed=3)       # many rows: also as two halves
    cands = o._split_candidates(N, 2048)
    assert ("rows", 2) in cands and ("rows", 2) not in o._split_candidates(N, 1100)
    close(o._run_plan(big.to(DEV), w.to(DEV), ("rows", 2)), R.linear(big, w), torch.bfloat16, scale=math.sqrt(K))
    plan.cuts[(8, N, K)] = ("rows", 2)                     # ragged rows of that class run whole
    close(o.linear(big[:1900].to(DEV), w.to(DEV)), R.linear(big[:1900], w), torch.bfloat16, scale=math.sqrt(K))
    del plan.cuts[(8, N, K)]
    o.linear(x.to(DEV), w.to(DEV))
    assert len(plan.cuts) == 1                             # measured once
    o.linear(x[:1000].to(DEV), w.to(DEV))                  # fewer rows than planning is for
    assert len(plan.cuts) == 1
    # 65 to 255 rows: whole against filled up to 256 rows, once per shape and 32 rows
    few = x[:100].to(DEV)
    close(o.linear(few, w.to(DEV)), R.linear(x[:100], w), torch.bfloat16, scale=math.sqrt(K))
    assert plan.cuts.get(("pad", 4, N, K)) in ((), ("pad", 256)) and len(plan.cuts) == 2
    close(o._run_plan(few, w.to(DEV), ("pad", 256)), R.linear(x[:100], w), torch.bfloat16, scale=math.sqrt(K))
    into = torch.empty(100, N, dtype=torch.bfloat16, device=DEV)
    assert o._run_plan(few, w.to(DEV), ("pad", 256), into) is into
    close(into, R.linear(x[:100], w), torch.bfloat16, scale=math.sqrt(K))
    o.linear(x[:64].to(DEV), w.to(DEV))
    o.linear(x[:256].to(DEV), w.to(DEV))
    assert len(plan.cuts) == 2
    assert Plan.from_dict(plan.to_dict()) == plan


def _prepared_rows(M, K, nw_dtype, eps, seed=5):
    """Residual rows with unequal scales and a norm weight far from 1, as `linear_add(norm=)`
    leaves them (made here by adding a product of zeros), and their plain norm."""
    x = rnd(M, K, seed=seed) * torch.linspace(0.02, 3.0, M)[:, None]
    nw = (1 + rnd(K, seed=seed + 1) * 0.3).to(nw_dtype)
    want = R.add_rmsnorm(x.clone(), None, nw, eps, torch.bfloat16)
    zeros = torch.zeros(M, 8, dtype=torch.bfloat16, device=DEV)
    rows = ops().linear_add(zeros, torch.zeros(K, 8, dtype=torch.bfloat16, device=DEV),
                            x.clone().to(DEV), (nw.to(DEV), eps))
    assert rows is not None and torch.equal(rows.x.cpu(), x)
    return rows, want


@pytest.mark.parametrize("nw_dtype", DTYPES)
@pytest.mark.parametrize("ydt", DTYPES)
@pytest.mark.parametrize("M,N,K,eps", [(1, 4096, 4096, 1e-5), (8, 100, 136, 1e-6), (16, 33, 1000, 1e-2), (5, 320, 96, 1e-5)])
def test_gemm_skinny_takes_the_norm(nw_dtype, ydt, M, N, K, eps):
    """The product of rows whose norm was prepared against norm, then product."""
    rows, h = _prepared_rows(M, K, nw_dtype, eps)
    w = rnd(N, K, dtype=torch.bfloat16, seed=2)
    got = ops().linear(rows, w.to(DEV), ydt)
    # the kernel rounds x * weight to bfloat16 and scales the sums, the reference rounds the
    # normed rows: the operands differ by bfloat16 roundings whatever the output's dtype
    close(got, R.linear(h, w, ydt), torch.bfloat16, scale=math.sqrt(K))
    close(rows.rows(), h, torch.bfloat16)                  # and can still be had normalised


@pytest.mark.parametrize("M,F,K", [(1, 11008, 4096), (8, 172, 64), (16, 203, 80), (3, 33, 1000)])
def test_gate_up_silu_takes_the_norm(M, F, K):
    rows, h = _prepared_rows(M, K, torch.bfloat16, 1e-5)
    w = rnd(2 * F, K, dtype=torch.bfloat16, seed=2, std=0.2)
    got = ops().gate_up_silu(rows, w.to(DEV))
    g, u = R.linear(h, w[:F], torch.float64), R.linear(h, w[F:], torch.float64)
    want = g / (1 + torch.exp(-g)) * u
    close(got, want, torch.bfloat16, scale=max(1.0, float(want.abs().max())))
    if K % 64 == 0:
        # the same through the kernel that shares X through LDS, where the plan sends few rows to it
        o = ops()
        plan = o.current_plan()
        try:
            plan.rows_from[("gate_up", 2 * F, K)] = 1
            again = o.gate_up_silu(rows, _decode_copy(w.to(DEV), "gate_up"))
        finally:
            del plan.rows_from[("gate_up", 2 * F, K)]
        close(again, want, torch.bfloat16, scale=max(1.0, float(want.abs().max())))


@pytest.mark.parametrize("nw_dtype", [None] + DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (8, 4096, 11008), (16, 104, 136), (7, 33, 1000)])
def test_linear_add(M, N, K, nw_dtype):
    """into += x . w^T in float32, nothing but the sum is rounded; with a norm's weight also
    bfloat16(into * weight) and the rows' sums of squares in parts."""
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
    into = rnd(M, N, seed=3) * 10
    dev = into.clone().to(DEV)
    assert ops().linear_add_fits(x.to(DEV), w.to(DEV), dev)
    nw = None if nw_dtype is None else (1 + rnd(N, seed=4) * 0.3).to(nw_dtype)
    rows = ops().linear_add(x.to(DEV), w.to(DEV), dev, None if nw is None else (nw.to(DEV), 1e-5))
    want = into.double() + R.linear(x, w, torch.float64)
    torch.testing.assert_close(dev.double().cpu(), want, atol=2e-4 * math.sqrt(K), rtol=1e-5)
    if nw is None or N % 8:
        assert rows is None
    else:
        assert rows.x is dev and rows.ssq.shape == (M, (N + 15) // 16)
        close(rows.xb, want * nw.double(), torch.bfloat16, scale=float(want.abs().max()))
        torch.testing.assert_close(rows.ssq.double().sum(1).cpu(), (want ** 2).sum(1), rtol=1e-5, atol=1e-6)
    assert not ops().linear_add_fits(x.to(DEV), w.to(DEV), dev.to(torch.bfloat16))
    assert not ops().linear_add_fits(rnd(17, K, dtype=torch.bfloat16).to(DEV), w.to(DEV), torch.zeros(17, N, device=DEV))


def _plain_copy(w):
    o = ops()
    return o.Weight(w, o.tile_weight(w, o.tile_rows(w.shape[0], "plain")), "plain")


# rows in every count of 16-row tiles; N with a last tile of 4 rows, with fewer tiles than
# a block's waves, with tiles beyond a multiple of 4; K of one piece, of a partial last piece
@pytest.mark.parametrize("tiles_per_wave", [0, 1, 2])
@pytest.mark.parametrize("M,N,K,splits", [(17, 40, 96, 0), (33, 100, 224, 0), (64, 4096, 11008, 0),
                                          (50, 84, 1184, 5), (48, 20, 64, 1), (31, 72, 352, 3),
                                          (64, 36, 2048, 16), (20, 8192, 16384, 0),
                                          (1, 40, 96, 0), (7, 100, 224, 2), (16, 4096, 11008, 0),
                                          (65, 40, 96, 0), (100, 84, 1184, 4), (128, 4096, 11008, 0),
                                          (81, 36, 2048, 16), (97, 132, 352, 3), (113, 4096, 4096, 0), (128, 8192, 8192, 0)])
def test_linear_planes(M, N, K, splits, tiles_per_wave):
    """The product for up to 128 rows, K cut into ranges: the planes add up to x . w^T, and what
    `add_rmsnorm` makes of them is the residual add and norm of the product.  Beyond 64 rows one
    launch and two of 64 rows give the same bits."""
    o = ops()
    if N >= 8192 and tiles_per_wave:
        return                   # the large case is there for the library's own choice of tiles
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
    wc = _plain_copy(w.to(DEV))
    assert o.linear_planes_fits(x.to(DEV), wc)
    o._lib().illm_set_mid_tiles_per_wave(tiles_per_wave)
    try:
        planes = o.linear_planes(x.to(DEV), wc, splits)
    finally:
        o._lib().illm_set_mid_tiles_per_wave(0)
    assert planes.dtype == torch.float32 and planes.shape[1:] == (M, N)
    assert splits == 0 or planes.shape[0] == splits
    if M > 64:
        o._lib().illm_set_mid_tiles_per_wave(tiles_per_wave)
        o._lib().illm_set_mid_rows_a_launch(64)
        try:
            assert torch.equal(o.linear_planes(x.to(DEV), wc, splits), planes)
        finally:
            o._lib().illm_set_mid_tiles_per_wave(0)
            o._lib().illm_set_mid_rows_a_launch(128)
    want = R.linear(x, w, torch.float64)
    torch.testing.assert_close(planes.double().sum(0).cpu(), want, atol=2e-4 * math.sqrt(K), rtol=1e-5)
    into = rnd(M, N, seed=3) * 10
    nw = (1 + rnd(N, seed=4) * 0.3).to(torch.bfloat16)
    dev = into.clone().to(DEV)
    got = o.add_rmsnorm(dev, planes, nw.to(DEV), 1e-5, torch.bfloat16)
    ref_x = into.clone()
    close(got, R.add_rmsnorm(ref_x, want.float(), nw, 1e-5, torch.bfloat16), torch.bfloat16, scale=4.0)
    torch.testing.assert_close(dev.cpu(), ref_x, atol=2e-4 * math.sqrt(K), rtol=1e-5)


@pytest.mark.parametrize("M,N,K,splits", [(129, 64, 4096, 0), (192, 4096, 4096, 0), (193, 68, 4160, 3), (256, 132, 4096, 64),
                                          (160, 260, 11008, 0), (1, 4, 64, 1), (200, 4096, 192, 3)])
def test_linear_cut(M, N, K, splits):
    """The product of 129 to 256 rows with K cut over blocks, from the row-major matrix: the planes add up
    to x . w^T (any order of K float32 sums: K 2^-24 of the sum of magnitudes) at edges of the tiles, with
    parts of one stage and of unequal length, and repeat bit for bit."""
    o = ops()
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2)
    xd, wd = x.to(DEV), w.to(DEV)
    planes = o.linear_cut(xd, wd, splits)
    assert planes.dtype == torch.float32 and planes.shape[1:] == (M, N) and (not splits or planes.shape[0] == splits)
    want = x.double() @ w.double().t()
    room = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert bool(((planes.double().sum(0).cpu() - want).abs() <= room).all())
    assert torch.equal(o.linear_cut(xd, o.Weight(wd), splits), planes)
    fits = 129 <= M <= 256 and N <= K and K >= 4096
    assert o.linear_cut_fits(xd, wd) == fits and not o.linear_cut_fits(xd.float(), wd)
    with pytest.raises(Exception):
        o.linear_cut(xd, wd, K // 64 + 1)                      # a part without a stage


def test_linear_planes_refuses_what_it_does_not_take():
    o = ops()
    w = rnd(64, 256, dtype=torch.bfloat16).to(DEV)
    x = rnd(20, 256, dtype=torch.bfloat16).to(DEV)
    assert o.linear_planes_fits(x, _plain_copy(w))
    assert not o.linear_planes_fits(x, w)                                  # no decode copy
    assert o.linear_planes_fits(x[:16], _plain_copy(w)) and o.linear_planes_pays(x, _plain_copy(w))
    assert not o.linear_planes_fits(rnd(129, 256, dtype=torch.bfloat16).to(DEV), _plain_copy(w))
    assert not o.linear_planes_fits(x.float(), _plain_copy(w))
    wide = rnd(256, 256, dtype=torch.bfloat16).to(DEV)                      # K < 2 N: not up to 16 rows
    assert not o.linear_planes_fits(x[:16], _plain_copy(wide)) and o.linear_planes_fits(x, _plain_copy(wide))
    many = rnd(100, 256, dtype=torch.bfloat16).to(DEV)                      # from 17 rows K = N is taken
    assert o.linear_planes_fits(many, _plain_copy(wide)) and o.linear_planes_pays(many, _plain_copy(wide))
    assert not o.linear_planes_fits(many, _plain_copy(rnd(512, 256, dtype=torch.bfloat16).to(DEV)))
    gate_up = o.Weight(w, o.tile_weight(w, o.tile_rows(64, "gate_up")), "gate_up")
    assert not o.linear_planes_fits(x, gate_up)                            # another kernel's tile order
    with pytest.raises(Exception):
        o.linear_planes(x, w)
    y = torch.empty(2, 20, 64, device=DEV)
    assert o._lib().illm_gemm_mid_bf16(o._p(x), o._p(_plain_copy(w).tiled), o._p(y), 0, 20, 64, 250, 2, None) != 0
    assert o._lib().illm_gemm_mid_bf16(o._p(x), o._p(_plain_copy(w).tiled), o._p(y), 0, 129, 64, 256, 2, None) != 0
    assert o._lib().illm_gemm_mid_bf16(o._p(x), o._p(_plain_copy(w).tiled), o._p(y), 0, 20, 64, 256, 3, None) != 0


@pytest.mark.parametrize("dtype", DTYPES)
def test_attn_decode_finds_one_far_key(dtype):
    """One key among hundreds is made to stand out: the output must be its value."""
    nh, nkv, hd, page, n = 4, 2, 32, 16, 777
    pt, kc, vc, slots, seq_len = paged_case(dtype, nkv, hd, [n], page)
    qkv = rnd(1, (nh + 2 * nkv) * hd, dtype=dtype, seed=1)
    target = 5
    pg, r = R.cache_offsets(pt, int(slots[0]), target, page, 0)
    q = qkv.view(1, nh + 2 * nkv, hd)
    for kvh in range(nkv):
        kc[pg, kvh, r] = q[0, kvh * (nh // nkv)].float().mul(40).to(dtype)   # huge score for head kvh*per
    got = ops().attn_decode(qkv.to(DEV), kc.to(DEV), vc.to(DEV), pt.to(DEV), page, 0, slots.to(DEV),
                            seq_len.to(DEV), nh, nkv, hd, 1.0, 0, 4).cpu().view(nh, hd)
    for kvh in range(nkv):
        close(got[kvh * (nh // nkv)], vc[pg, kvh, r], dtype)


@pytest.mark.parametrize("B,V", [(1, 256), (3, 320), (2, 32000), (64, 411), (1, 128256), (5, 128256), (64, 32000),
                                 (9, 4099)])
def test_argmax(B, V):
    logits = rnd(B, V, seed=4)
    logits[0, V - 1] = 50.0
    if B > 1:
        logits[1, 3] = 60.0; logits[1, 200] = 60.0           # a tie: the lower id wins
    got = ops().argmax(logits.to(DEV)).cpu()
    assert got.tolist() == R.argmax(logits).tolist()
    assert got[0] == V - 1 and (B == 1 or got[1] == 3)
    # ties across the parts a long row is cut into, a NaN above everything, a row of NaN alone
    logits[0, V - 1] = 0.0
    logits[0, 5] = 70.0; logits[0, V - 2] = 70.0; logits[0, V // 2] = float("nan")
    if B > 2:
        logits[2] = float("nan")
    got = ops().argmax(logits.to(DEV)).cpu()
    assert got[0] == 5 and (B <= 2 or got[2] == 0)
    assert got.tolist()[3:] == R.argmax(logits).tolist()[3:]


def interval_ok(logits_row, token, u, temperature, top_k, top_p, penalty, last):
    """The drawn token's interval of the id-ordered CDF over the kept ids contains u (with slack)."""
    ids, p = R.kept_distribution(logits_row, temperature, top_k, top_p, penalty, last)
    pairs = sorted(zip(ids, p.tolist()))
    cum = 0.0
    for i, pi in pairs:
        if i == token:
            return cum - 1e-4 <= u <= cum + pi + 1e-4
        cum += pi
    return False


def test_the_uniform_numbers_of_the_tests_and_of_the_host_side_agree():
    """The tests state the sampler's hash themselves (kernel_refs.uniform), pinned by the
    published first outputs of splitmix64; the host side's `uniform`, which the generation loop
    would use, must be the same function."""
    from inferllm_amd.sampling.params import request_seed, uniform
    assert [R.mix64(i * 0x9E3779B97F4A7C15) for i in (1, 2, 3)] == \
        [0xE220A8397B1DCDAF, 0x6E789E6AA1B965F4, 0x06C45D188009454F]
    for seed in (0, 3, 2**63 + 5, (1 << 64) - 1):
        for c in (0, 1, 77):
            assert uniform(seed, c) == R.uniform(seed, c)
            assert 0.0 <= R.uniform(seed, c) < 1.0
    assert len({R.uniform(request_seed(9, i), c) for i in range(4) for c in range(64)}) > 250


@pytest.mark.parametrize("V,temperature,top_k,top_p,penalty", [
    (256, 0.8, 0, 1.0, 1.0), (320, 0.8, 40, 0.95, 1.1), (411, 0.1, 40, 0.95, 1.3), (1000, 1.5, 5, 1.0, 1.0),
    (32000, 1.0, 0, 0.9, 1.0), (300, 0.7, 1, 1.0, 1.0), (128256, 0.9, 50, 0.8, 1.2),
    (2000, 0.9, 1024, 0.7, 1.1), (2000, 0.9, 1025, 0.7, 1.0), (50, 1.0, 49, 0.5, 1.0), (32000, 0.1, 40, 0.95, 1.1),
    # rows too long for a thread's registers: top_p alone, with a large top_k, temperature alone
    (128256, 0.9, 0, 0.8, 1.2), (40000, 1.0, 2000, 0.6, 1.0), (33000, 0.7, 0, 0.999, 1.0), (50000, 1.3, 0, 1.0, 1.0),
    # long rows with a small top_k are cut into parts that blocks of their own take: a length that
    # no part divides, the largest top_k of that way and the first beyond it
    (70001, 0.1, 40, 0.95, 1.1), (65536, 1.0, 64, 0.5, 1.0), (65536, 1.0, 65, 0.5, 1.3), (200003, 0.8, 3, 1.0, 1.3),
    # long rows without top_k: several blocks a row and a kernel a pass
    (70001, 0.7, 0, 0.9, 1.0), (131072, 1.0, 0, 1.0, 1.1), (200003, 0.5, 0, 0.5, 1.3), (65536, 2.0, 0, 0.999, 1.0),
    (65537, 0.3, 0, 0.05, 1.0), (16384, 0.9, 0, 0.7, 1.2), (16387, 1.1, 0, 1.0, 1.0)])
def test_sample_draws_from_the_reference_distribution(V, temperature, top_k, top_p, penalty):
    uniform = R.uniform                                      # the tests' own statement of the hash
    B = 6
    logits = rnd(B, V, seed=8, std=2.0)
    logits[2] = 0.0                                            # all equal: ties everywhere
    last = torch.full((B, 8), -1, dtype=torch.int32)
    last[:, :4] = torch.tensor([1, 5, V - 1, 5], dtype=torch.int32)     # an id twice: penalised once
    seeds = torch.tensor([3, 99, 12345, -7, 2**62, 0], dtype=torch.int64)
    counters = torch.tensor([0, 1, 2, 3, 4, 5], dtype=torch.int32)
    got = ops().sample(logits.to(DEV), temperature, top_k, top_p, penalty,
                       last.to(DEV) if penalty != 1.0 else None, seeds.to(DEV), counters.to(DEV)).cpu().tolist()
    for b in range(B):
        u = uniform(int(seeds[b]) & ((1 << 64) - 1), int(counters[b]))
        assert interval_ok(logits[b], got[b], u, temperature, top_k, top_p, penalty,
                           last[b] if penalty != 1.0 else None), (b, got[b], u)
    if top_k == 1:
        assert got == torch.argmax(logits, -1).tolist() or penalty != 1.0


def test_sample_of_a_long_row_in_parts_keeps_what_one_block_would():
    """A long row with a small top_k is the work of several blocks, each with a stretch of the ids.
    Equal scores at the k-th place go to the lower ids, wherever the stretches' edges lie: of 90 equal
    scores spread over the whole row, the 40 with the lowest ids are kept, and every draw is one of them."""
    V, B, top_k = 131072, 64, 40
    logits = rnd(B, V, seed=21, std=1.0).clamp_(max=3.0)
    high = torch.arange(90) * 1451 + 7                        # up to id 129,146: in every stretch
    logits[:, high] = 9.0
    logits[1, high[:5]] = 12.0                                # row 1: five above, then 35 of the 85 equal ones
    seeds = torch.arange(B, dtype=torch.int64) * 104729 + 3
    counters = torch.arange(B, dtype=torch.int32)
    got = ops().sample(logits.to(DEV), 1.0, top_k, 1.0, 1.0, None, seeds.to(DEV), counters.to(DEV)).cpu()
    kept = set(high[:top_k].tolist())
    assert all(int(t) in kept for t in got), [int(t) for t in got if int(t) not in kept]
    assert len({int(t) for t in got}) > 20                    # and not always the same few
    for b in range(B):
        u = R.uniform(int(seeds[b]), int(counters[b]))
        assert interval_ok(logits[b], int(got[b]), u, 1.0, top_k, 1.0, 1.0, None), (b, int(got[b]), u)


@pytest.mark.parametrize("top_p", [1.0, 0.9, 0.3])
def test_sample_of_a_long_row_does_not_depend_on_its_company(top_p):
    """Rows of 16,384 ids and more without top_k are cut into more or fewer parts depending on how
    many rows there are; the masses are added as integers, so a row draws the same id alone and
    among 69 others, draw after draw."""
    V = 100003
    rows = rnd(70, V, seed=33, std=3.0)
    seeds = torch.arange(70, dtype=torch.int64) * 7919 + 5
    last = torch.randint(0, V, (70, 16), generator=torch.Generator().manual_seed(2), dtype=torch.int32)
    for counter in (0, 1, 2):
        counters = torch.full((70,), counter, dtype=torch.int32)
        together = ops().sample(rows.to(DEV), 0.8, 0, top_p, 1.2, last.to(DEV), seeds.to(DEV), counters.to(DEV)).cpu()
        for b in (0, 13, 69):
            alone = ops().sample(rows[b:b + 1].to(DEV), 0.8, 0, top_p, 1.2, last[b:b + 1].to(DEV),
                                 seeds[b:b + 1].to(DEV), counters[b:b + 1].to(DEV)).cpu()
            assert int(alone[0]) == int(together[b]), (b, counter)
        few = ops().sample(rows[:9].to(DEV), 0.8, 0, top_p, 1.2, last[:9].to(DEV), seeds[:9].to(DEV),
                           counters[:9].to(DEV)).cpu()
        assert few.tolist() == together[:9].tolist()


def test_sample_frequencies_match_probabilities():
    V, n = 7, 4000
    row = torch.tensor([2.0, 1.0, 0.5, 0.0, -1.0, 1.5, -3.0])
    logits = row.repeat(n, 1)
    seeds = torch.arange(n, dtype=torch.int64) * 7919 + 1
    counters = torch.zeros(n, dtype=torch.int32)
    got = ops().sample(logits.to(DEV), 0.9, 0, 1.0, 1.0, None, seeds.to(DEV), counters.to(DEV)).cpu()
    freq = torch.bincount(got.long(), minlength=V).double() / n
    p = torch.softmax(row.double() / 0.9, 0)
    chi2 = float((n * (freq - p) ** 2 / p).sum())
    assert chi2 < 30.0, (chi2, freq, p)           # 6 degrees of freedom: far beyond any honest draw


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hd", [32, 24])
def test_window_edge_prefill_and_decode(dtype, hd):
    """A key that stands out sits exactly at the window's edge: the query `window - 1` places
    after it still sees it, the next query does not (prefill), and likewise for a single new
    token over the cache (decode)."""
    nh, nkv, n, window, edge = 2, 2, 150, 40, 70
    qkv = rnd(n, (nh + 2 * nkv) * hd, dtype=dtype, seed=5, std=0.3)
    view = qkv.view(n, nh + 2 * nkv, hd)
    probe = rnd(hd, seed=6).to(dtype)
    view[:, 0] = probe                                   # every query of head 0 looks for the probe
    view[edge, nh] = probe.float().mul(25).to(dtype)     # and key `edge` answers it loudly
    view[edge, nh + nkv] = 7.0                           # its value is unmistakable
    cu = torch.tensor([0, n], dtype=torch.int32)
    out = ops().attn_prefill(qkv.to(DEV), cu.to(DEV), 1, n, nh, nkv, hd, 1.0, window).cpu().view(n, nh, hd).float()
    last_seeing = edge + window - 1
    assert float(out[last_seeing, 0].mean()) > 6.5       # still inside the window
    assert float(out[last_seeing + 1, 0].mean()) < 3.0   # one step further: gone
    assert float(out[edge - 1, 0].mean()) < 3.0          # and the future is hidden
    want = R.attn_prefill(qkv, cu, 1, n, nh, nkv, hd, 1.0, window)
    close(out.reshape(n, -1), want, dtype, scale=8)
    # decode: cache holds keys 0..L-1 (the last one is the new token's)
    page = 64
    ring = (window + page - 2) // page + 1
    for L, sees in ((edge + window, True), (edge + window + 1, False)):
        pt = torch.tensor([[3, 1, 0][:ring] + [2] * max(0, ring - 3)], dtype=torch.int32)[:, :ring]
        kc = torch.full((4, nkv, page, hd), float("nan"), dtype=dtype); vc = kc.clone()
        for pos in range(max(0, L - ring * page), L):    # what a ring keeps
            pg = int(pt[0, (pos // page) % ring])
            if pos // page + ring > (L - 1) // page:
                kc[pg, :, pos % page] = view[pos, nh:nh + nkv]; vc[pg, :, pos % page] = view[pos, nh + nkv:]
        q = view[L - 1:L].reshape(1, -1).contiguous()
        got = ops().attn_decode(q.to(DEV), kc.to(DEV), vc.to(DEV), pt.to(DEV), page, ring,
                                torch.zeros(1, dtype=torch.int32, device=DEV),
                                torch.tensor([L], dtype=torch.int32, device=DEV), nh, nkv, hd, 1.0, window, 2)
        mean = float(got.cpu().view(nh, hd)[0].float().mean())
        assert (mean > 6.5) == sees, (L, mean)
        close(got.cpu().view(nh, hd), out[L - 1], dtype, scale=8)


_QKV_SHAPES = [(1, 32, 32, 128, 4096), (8, 4, 2, 32, 64), (16, 6, 3, 64, 200), (3, 8, 1, 96, 72),
               (5, 3, 3, 48, 136), (2, 2, 1, 16, 40), (5, 3, 3, 48, 160), (7, 2, 2, 16, 96),
               (13, 3, 3, 48, 192), (16, 8, 2, 128, 1024)]


# with the decode copy only where one can be made (K a multiple of 32)
@pytest.mark.parametrize("M,nh,nkv,hd,K,copy", [s + (c,) for s in _QKV_SHAPES for c in (False, True)
                                                if not (c and s[4] % 32)])
@pytest.mark.parametrize("normed", [False, True])
@pytest.mark.parametrize("shared_x", [False, True])
def test_qkv_rope_store_equals_the_three_steps(M, nh, nkv, hd, K, normed, copy, shared_x, monkeypatch):
    """The fused decode kernel against (norm,) product, then rotation and cache store.
    `shared_x`: the plan sends these few rows to the kernel that shares X through LDS
    (csrc/gemm_rows.hip), which needs the decode copy and K a multiple of 64."""
    from inferllm_amd.parts.position import rotary_table
    if shared_x:
        if not copy or K % 64:
            pytest.skip("the shared-X kernel needs the decode copy and K % 64 == 0")
        monkeypatch.setitem(ops().current_plan().rows_from, ("qkv", (nh + 2 * nkv) * hd, K), 1)
    dtype, page = torch.bfloat16, 64
    table = rotary_table(777.0, hd, 300, "cpu")
    x = rnd(M, K, dtype=dtype, seed=1)
    x_dev = x.to(DEV)
    if normed:
        x_dev, x = _prepared_rows(M, K, torch.bfloat16, 1e-5)
    w = rnd((nh + 2 * nkv) * hd, K, dtype=dtype, seed=2, std=0.1)
    pos = torch.tensor([(37 * i + 5) % 290 for i in range(M)], dtype=torch.int32)
    slot = torch.randperm(M + 2, generator=torch.Generator().manual_seed(9))[:M].to(torch.int32)
    assert len(set(slot.tolist())) == M
    g = torch.Generator().manual_seed(4)
    pt = torch.randperm((M + 2) * 5, generator=g).reshape(M + 2, 5).to(torch.int32)
    kc, vc = make_cache((M + 2) * 5, nkv, page, hd, dtype)
    # reference: float64 product, rounded to bfloat16 once (as the fused kernel rounds once)
    qkv_ref = R.linear(x, w, torch.float64)
    kr, vr = kc.clone().double(), vc.clone().double()
    R.rope_store(qkv_ref, table, hd, 0, pos, slot, None, kr, vr, pt, page, 0, nh, nkv, hd)
    w_dev = _decode_copy(w.to(DEV), "qkv", nh=nh, nkv=nkv, hd=hd) if copy else w.to(DEV)
    got = ops().qkv_rope_store(x_dev, w_dev, table.to(DEV), pos.to(DEV), slot.to(DEV), kc_g := kc.to(DEV),
                               vc_g := vc.to(DEV), pt.to(DEV), page, 0, nh, nkv, hd).cpu()
    sc = math.sqrt(K) * 0.1
    close(got[:, :nh * hd], qkv_ref[:, :nh * hd], dtype, scale=sc)
    for gotc, wantc in ((kc_g.cpu(), kr), (vc_g.cpu(), vr)):
        assert torch.equal(torch.isnan(gotc), torch.isnan(wantc))        # the same rows, nothing else
        close(torch.nan_to_num(gotc), torch.nan_to_num(wantc), dtype, scale=sc)


# ---------------------------------------------------------------- products of 9 to 128 rows
# (tiles a block, parts of K)
_ROWS_SHAPES = [(None, None), (2, 1), (2, 4), (3, 2), (3, 4), (4, 1), (4, 2), (5, 2), (6, 1), (7, 1), (8, 2)]


@pytest.fixture
def rows_shape():
    """Forces the block shape of the rows kernels and gives the library's own choice back after."""
    lib = ops()._lib()
    yield lambda tb, kp: lib.illm_set_rows_shape(tb or 0, kp or 0)
    lib.illm_set_rows_shape(0, 0)


@pytest.mark.parametrize("tb,kp", _ROWS_SHAPES)
@pytest.mark.parametrize("M,N,K", [(17, 40, 128), (33, 100, 192), (64, 12288, 4096), (9, 320, 64), (1, 64, 64),
                                   (65, 411, 320), (128, 1000, 1088), (48, 32000, 256), (100, 8, 4096)])
def test_linear_rows(M, N, K, tb, kp, rows_shape):
    """The product with X shared through LDS and K cut inside the block, in every block shape,
    float32 and bfloat16 results; row counts around the tile and launch edges (16, 64)."""
    o = ops()
    rows_shape(tb, kp)
    x, w = rnd(M, K, dtype=torch.bfloat16, seed=1), rnd(N, K, dtype=torch.bfloat16, seed=2, std=0.2)
    wc = _decode_copy(w.to(DEV))
    want = R.linear(x, w, torch.float64)
    for ydt in DTYPES:
        got = o.linear_rows(x.to(DEV), wc, ydt)
        assert got.dtype == ydt
        close(got, want, ydt, scale=0.2 * math.sqrt(K))
    # a row's result does not depend on the other rows of the step: the same bits (beyond 64 rows
    # a block has half as many parts of K at most, so a forced number of parts may hold for the
    # row alone and not for the step: another order of summation)
    if not (M > 64 and kp is not None and kp > (1 if tb >= 4 else 2)):
        alone = o.linear_rows(x[M - 1:].to(DEV), wc, torch.float32)
        among = o.linear_rows(x.to(DEV), wc, torch.float32)[M - 1]
        assert torch.equal(alone[0], among)


def test_linear_rows_takes_the_norm_and_refuses_what_it_does_not_take(rows_shape):
    o = ops()
    M, N, K = 12, 200, 4096
    x_dev, x = _prepared_rows(M, K, torch.bfloat16, 1e-5)
    w = rnd(N, K, dtype=torch.bfloat16, seed=2, std=0.2)
    wc = _decode_copy(w.to(DEV))
    for tb, kp, ps in ((None, None, None), (2, 4, 2), (4, 1, 4)):
        rows_shape(tb, kp)
        close(o.linear_rows(x_dev, wc, torch.float32), R.linear(x, w, torch.float64), torch.bfloat16,
              scale=0.2 * math.sqrt(K))
    assert not o.rows_fits(rnd(129, K, dtype=torch.bfloat16).to(DEV), wc, "plain")
    assert not o.rows_fits(rnd(20, K, dtype=torch.bfloat16).to(DEV), wc, "gate_up")     # another kernel's tiles
    assert not o.rows_fits(rnd(20, K, dtype=torch.bfloat16).to(DEV), w.to(DEV), "plain")  # no copy
    assert not o.rows_fits(rnd(20, K).to(DEV), wc, "plain")                             # float32 rows
    w96 = _decode_copy(rnd(N, 96, dtype=torch.bfloat16, seed=3).to(DEV))
    assert not o.rows_fits(rnd(20, 96, dtype=torch.bfloat16).to(DEV), w96, "plain")     # K must be a multiple of 64
    with pytest.raises(o.KernelError):
        o.linear_rows(rnd(20, K).to(DEV), wc, torch.float32)


@pytest.mark.parametrize("tb,kp", _ROWS_SHAPES)
@pytest.mark.parametrize("M,F,K", [(17, 172, 64), (64, 11008, 4096), (40, 50, 192), (64, 203, 320), (33, 8, 1024),
                                   (65, 50, 192), (100, 172, 128), (128, 2056, 512), (113, 203, 320)])
def test_gate_up_silu_of_many_rows(M, F, K, tb, kp, rows_shape):
    """17 to 128 rows: the product and the SiLU-multiply in one kernel, from the gate|up tiles."""
    o = ops()
    rows_shape(tb, kp)
    x = rnd(M, K, dtype=torch.bfloat16, seed=1)
    w = rnd(2 * F, K, dtype=torch.bfloat16, seed=2, std=0.2)
    got = o.gate_up_silu(x.to(DEV), _decode_copy(w.to(DEV), "gate_up"))
    g, u = R.linear(x, w[:F], torch.float64), R.linear(x, w[F:], torch.float64)
    want = g / (1 + torch.exp(-g)) * u
    top = max(1.0, float(want.abs().max()))
    close(got, want, torch.bfloat16, scale=top)
    swapped = u / (1 + torch.exp(-u)) * g
    assert not torch.allclose(got.double().cpu(), swapped, atol=0.1 * top)
    # the product alone keeps float32 sums where the unfused path rounds gate and up to bfloat16
    # first: the fused result is the closer one
    loose = o.gate_up_silu(x.to(DEV), w.to(DEV))            # no copy: vendor GEMM, then SiLU-multiply
    close(loose, want, torch.bfloat16, scale=top)
    assert float((got.double().cpu() - want).abs().mean()) <= float((loose.double().cpu() - want).abs().mean()) * 1.05


@pytest.mark.parametrize("tb,kp", _ROWS_SHAPES)
@pytest.mark.parametrize("M,nh,nkv,hd,K", [(17, 4, 2, 32, 64), (64, 32, 32, 128, 4096), (40, 6, 3, 64, 256),
                                           (64, 8, 1, 96, 128), (33, 3, 3, 48, 192), (50, 2, 1, 16, 1024),
                                           (65, 4, 2, 32, 64), (96, 6, 3, 64, 256), (128, 48, 8, 128, 256),
                                           (113, 40, 40, 128, 128)])
def test_qkv_rope_store_of_many_rows(M, nh, nkv, hd, K, tb, kp, rows_shape):
    """17 to 128 sequences decoding together (96 for matrices of fewer than 8192 rows): the q|k|v
    product, the rotation and the cache store in one kernel against the three steps."""
    from inferllm_amd.parts.position import rotary_table
    o = ops()
    rows_shape(tb, kp)
    dtype, page = torch.bfloat16, 64
    table = rotary_table(777.0, hd, 300, "cpu")
    x = rnd(M, K, dtype=dtype, seed=1)
    w = rnd((nh + 2 * nkv) * hd, K, dtype=dtype, seed=2, std=0.1)
    pos = torch.tensor([(37 * i + 5) % 290 for i in range(M)], dtype=torch.int32)
    slot = torch.randperm(M + 2, generator=torch.Generator().manual_seed(9))[:M].to(torch.int32)
    g = torch.Generator().manual_seed(4)
    pt = torch.randperm((M + 2) * 5, generator=g).reshape(M + 2, 5).to(torch.int32)
    kc, vc = make_cache((M + 2) * 5, nkv, page, hd, dtype)
    qkv_ref = R.linear(x, w, torch.float64)
    kr, vr = kc.clone().double(), vc.clone().double()
    R.rope_store(qkv_ref, table, hd, 0, pos, slot, None, kr, vr, pt, page, 0, nh, nkv, hd)
    w_dev = _decode_copy(w.to(DEV), "qkv", nh=nh, nkv=nkv, hd=hd)
    assert o.qkv_rope_store_fits(x.to(DEV), w_dev, hd) and not o.qkv_rope_store_fits(x.to(DEV), w.to(DEV), hd)
    got = o.qkv_rope_store(x.to(DEV), w_dev, table.to(DEV), pos.to(DEV), slot.to(DEV), kc_g := kc.to(DEV),
                           vc_g := vc.to(DEV), pt.to(DEV), page, 0, nh, nkv, hd).cpu()
    sc = math.sqrt(K) * 0.1
    close(got[:, :nh * hd], qkv_ref[:, :nh * hd], dtype, scale=sc)
    for gotc, wantc in ((kc_g.cpu(), kr), (vc_g.cpu(), vr)):
        assert torch.equal(torch.isnan(gotc), torch.isnan(wantc))        # the same rows, nothing else
        close(torch.nan_to_num(gotc), torch.nan_to_num(wantc), dtype, scale=sc)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("E", [4, 1024, 1028, 2052, 4096, 4100, 8196, 90])
def test_passes_of_single_tokens_over_widths_and_taps(E, dtype):
    """The passes that ask for all they read at once: groups of four columns a thread from none left over to one
    more than a thread's share, and the widths that take the plain loops; 2 to 5 taps (compiled in up to 4)."""
    g = torch.Generator().manual_seed(E)
    o, T, V, buckets = ops(), 3, 11, 7
    # float32: sums of up to 8,196 squares and 5 taps, relative error below 1e-5; bfloat16: the result's rounding,
    # and one step more where the rounded input of the convolution falls on the other side
    tol = 1e-5 if dtype == torch.float32 else 2 ** -7

    def near(got, want, tol):
        want = want.double()
        assert float((got.double().cpu() - want).abs().max()) <= tol * max(1.0, float(want.abs().max()))
    a, pw = (torch.randn(T, E, generator=g) * 3).to(dtype), torch.randn(E, generator=g) + 1
    x, w = torch.randn(T, E, generator=g), (torch.randn(E, generator=g) + 1).to(dtype)
    slots = torch.tensor([3, 0, 2], dtype=torch.int32)
    for taps in (2, 3, 4, 5):
        cw, tail = torch.randn(E, taps, generator=g), torch.randn(4, taps - 1, E, generator=g).to(dtype)
        for post in (None, (a, pw, 1e-5, 0.3)):
            x_want, x_got, t_want, t_got = x.clone(), x.to(DEV), tail.clone(), tail.to(DEV)
            want = R.post_add_rmsnorm(x_want, o.PostNormed(*post) if post else None, w, 2e-5, dtype, None,
                                      (cw, t_want, slots))
            got = o.post_add_rmsnorm(x_got, o.PostNormed(a.to(DEV), pw.to(DEV), 1e-5, 0.3) if post else None,
                                     w.to(DEV), 2e-5, dtype, None, (cw.to(DEV), t_got, slots.to(DEV)))
            near(got, want, tol), near(x_got, x_want, 1e-5), near(t_got, t_want, tol)
        # rows of two sequences (the second's first inputs are kept ones) and single rows; taps of an odd base
        X, bias, odd = x.to(dtype), torch.randn(E, generator=g), torch.zeros(E * taps + 1)
        odd[1:] = cw.reshape(-1)
        for row_slot in (torch.tensor([1, 1, 2], dtype=torch.int32), slots):
            for cwd in (cw.to(DEV), odd.to(DEV)[1:].view(E, taps)):
                single = row_slot is slots
                t_want, t_got = tail.clone(), tail.to(DEV)
                want = R.short_conv(X, 0, E, cw, t_want, row_slot, torch.float32, bias, bias, False, update_tail=single)
                got = o.short_conv(X.to(DEV), 0, E, cwd, t_got, row_slot.to(DEV), torch.float32, bias.to(DEV),
                                   bias.to(DEV), False, update_tail=single)
                near(got, want, tol), near(t_got, t_want, tol)
    table, pairs = torch.randn(V, E, generator=g).to(dtype), torch.randn(buckets + 1, E, generator=g).to(dtype)
    places = torch.randn(5, E, generator=g)
    tokens, pos = torch.tensor([3, 10, 0], dtype=torch.int32), torch.tensor([0, 4, 2], dtype=torch.int32)
    for pr, pl in ((pairs, places), (pairs, None), (None, places), (None, None)):
        l_want, l_got = torch.tensor([1, 2, 4, 9], dtype=torch.int32), torch.tensor([1, 2, 4, 9], dtype=torch.int32).to(DEV)
        put = lambda t: t.to(DEV) if t is not None else None
        want = R.embed_pairs(tokens, pos, slots, table, 2.5, pr, buckets, 7, 3, pl, l_want, True)
        got = o.embed_pairs(put(tokens), put(pos), put(slots), put(table), 2.5, put(pr), buckets, 7, 3, put(pl), l_got, True)
        near(got, want, 1e-6)
        assert torch.equal(l_got.cpu(), l_want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh, nkv, dk, dv, weights, mix", [(2, 1, 4, 8, True, True), (16, 4, 64, 64, True, False),
                                                           (8, 2, 132, 128, False, True), (4, 4, 256, 260, True, True),
                                                           (32, 8, 128, 128, True, True), (33, 1, 128, 64, True, True),
                                                           (4, 2, 128, 128, False, False), (16, 4, 128, 128, False, True),
                                                           (3, 1, 32, 16, False, True), (2, 1, 248, 252, False, True), (2, 1, 252, 256, False, True),
                                                           (40, 8, 128, 128, False, True)])
def test_norm_mix_and_store_four_columns_a_load(nh, nkv, dk, dv, weights, mix, dtype):
    """Widths around a thread's share (1,024, 2,048 and 4,096 columns; 4,224 takes the loop by column, and below 256
    without the norm), with and without the norm and the mix of values, into a cache with a ring and into none."""
    g = torch.Generator().manual_seed(nh * dk + dv)
    o, page, pages, ring = ops(), 16, 6, 2
    # float32: one rounding a step and a sum of up to 4,224 squares; bfloat16: the result's rounding (2^-8)
    tol = 1e-5 if dtype == torch.float32 else 2 ** -8
    pos, slot = torch.tensor([40, 3, 17], dtype=torch.int32), torch.tensor([1, 0, 2], dtype=torch.int32)
    table = torch.randperm(pages, generator=g).view(3, 2).to(torch.int32)
    k_off, v_off = nh * dk + 4, nh * dk + 4 + nkv * dk
    rows = torch.randn(3, v_off + nkv * dv + 8, generator=g).to(dtype)
    first = torch.randn(3, nkv * dv + 12, generator=g).to(dtype) if mix else None
    lam = torch.tensor([0.3]) if mix else None
    qw, kw = (torch.randn(n * dk, generator=g).to(dtype) if weights else None for n in (nh, nkv))
    put = lambda t: t.to(DEV) if t is not None else None
    for cached in (True, False):
        kc = torch.randn(pages, nkv, page, dk, generator=g).to(dtype) if cached else None
        vc = torch.randn(pages, nkv, page, dv, generator=g).to(dtype) if cached else None
        r_want, r_got, kc_got, vc_got = rows.clone(), put(rows), put(kc), put(vc)
        o.qkv_norm_mix_store(r_got, k_off, v_off, put(qw), put(kw), 1e-5, put(lam), put(first), 8, put(pos), put(slot),
                             kc_got, vc_got, put(table), page, ring, nh, nkv, dk, dv)
        R.qkv_norm_mix_store(r_want, k_off, v_off, qw, kw, 1e-5, lam, first, 8, pos, slot, kc, vc, table, page, ring,
                             nh, nkv, dk, dv)
        for got, want in ((r_got, r_want), (kc_got, kc), (vc_got, vc)):
            if want is not None:
                want = want.double()
                assert float((got.double().cpu() - want).abs().max()) <= tol * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("T", [1, 4, 7, 128, 129])
@pytest.mark.parametrize("nb, cb", [(2, 4), (3, 32), (1, 36), (2, 128), (1, 1028), (2, 30)])
def test_recurrent_gates_of_few_rows(T, nb, cb):
    """Blocks of channels around the 32 outputs a block takes; rows around its 4; 129 rows and blocks below 64
    channels take the other kernel."""
    g = torch.Generator().manual_seed(T + cb)
    u = torch.randn(T, nb * cb, generator=g) * 2
    wt = torch.randn(2, nb, cb, cb, generator=g) * min(0.5, 4.0 / cb ** 0.5)
    rb, ib, lam = (torch.randn(nb * cb, generator=g) for _ in range(3))
    for got, want in zip(ops().lru_gates(*(t.to(DEV) for t in (u, wt, rb, ib, lam)), 8.0),
                         R.lru_gates(u, wt, rb, ib, lam, 8.0)):
        # sums of up to 1,028 products of size 8 in float32, through functions of slope below 8
        assert float((got.cpu().double() - want.double()).abs().max()) <= 1e-5 * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("nb, cb", [(2, 4), (3, 36), (3, 64), (2, 65), (16, 128), (1, 129), (2, 200), (2, 256), (1, 1028), (1, 3072),
                                    (1, 4096)])
def test_recurrent_gates_of_a_row_alone_and_among_others(nb, cb):
    """A row's gates are the same bits alone, among 128 rows (the most of one kernel) and among 129: blocks narrower
    and wider than a thread block, with a last slice of their inputs cut short, up to the widest that was ever taken."""
    g = torch.Generator().manual_seed(cb)
    u = (torch.randn(129, nb * cb, generator=g) * 2).to(DEV)
    maps = [t.to(DEV) for t in (torch.randn(2, nb, cb, cb, generator=g) * min(0.5, 4.0 / cb ** 0.5),
                                *(torch.randn(nb * cb, generator=g) for _ in range(3)))]
    every = ops().lru_gates(u, *maps, 8.0)
    for T in (1, 3, 4, 5, 128):
        for at in (0, 129 - T):
            for a, b in zip(ops().lru_gates(u[at:at + T].contiguous(), *maps, 8.0), every):
                assert torch.equal(a, b[at:at + T]), (T, at)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H, dk, dv", [(4, 256, 128), (1, 4, 4), (8, 132, 264), (16, 64, 64), (5, 12, 2), (4, 64, 64), (2, 64, 128),
                                       (2, 130, 64)])
def test_gated_linear_attention_rows_four_columns_a_load(H, dk, dv, dtype):
    g = torch.Generator().manual_seed(H * dk)
    for off in (0, 1):                                  # (an odd offset takes the loop by column)
        U = (torch.randn(3, 2 * H * dk + H * dv + 8, generator=g) * 2).to(dtype)
        Z, zb = (torch.randn(3, H * dk, generator=g) * 3).to(dtype), torch.randn(H * dk, generator=g)
        args = (off, off + H * dk, off + 2 * H * dk)
        want = R.gla_prepare(U, *args, Z, zb, 7.0, H, dk, dv)
        got = ops().gla_prepare(U.to(DEV), *args, Z.to(DEV), zb.to(DEV), 7.0, H, dk, dv)
        for a, b in zip(got, want):                     # (one exponential and one logarithm in float32)
            assert float((a.cpu().double() - b.double()).abs().max()) <= 1e-5 * max(1.0, float(b.abs().max()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh, nkv, dk, dv", [(4, 1, 128, 128), (6, 2, 64, 32), (5, 1, 104, 72), (2, 2, 8, 128), (3, 1, 64, 8)])
def test_capped_decode_ranges_and_rounds(nh, nkv, dk, dv, dtype):
    """Key counts around a wave's rounds (32 keys) and the ranges' tiles (64), so that ranges are empty, end in their
    first round or go past the two in flight; heads of a block that are not there; columns beyond the sizes."""
    g = torch.Generator().manual_seed(nh * dk + dv)
    lens, page = [1, 8, 31, 33, 64, 65, 97, 129, 200, 321], 16
    B, per = len(lens), 21
    table = torch.randperm(B * per, generator=g).view(B, per).to(torch.int32)
    kc, vc = torch.randn(B * per, nkv, page, dk, generator=g).to(dtype), torch.randn(B * per, nkv, page, dv, generator=g).to(dtype)
    q, slots = torch.randn(B, nh * dk, generator=g).to(dtype), torch.randperm(B, generator=g).to(torch.int32)
    seq_len, slopes = torch.tensor(lens, dtype=torch.int32), torch.rand(nh, generator=g) * 0.1
    put = lambda t: t.to(DEV)
    for window, cap in ((0, 0.0), (70, 5.0)):
        args = (nh, nkv, dk, dv, dk ** -0.5, cap, window)
        want = R.attn_cap_decode(q, kc, vc, table, page, 0, slots, seq_len, *args, 1, slopes).double()
        for nsplit in (1, 3, 16, 17):
            got = ops().attn_cap_decode(put(q), put(kc), put(vc), put(table), page, 0, put(slots), put(seq_len), *args,
                                        nsplit, put(slopes))
            # float32: the scores' and sums' rounding; bfloat16: the result's (2^-9) and the exponential's
            tol = 1e-5 if dtype == torch.float32 else 2 ** -8
            assert float((got.double().cpu() - want).abs().max()) <= tol * max(1.0, float(want.abs().max())), (window, nsplit)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dk, dv", [(128, 128), (64, 32), (40, 200)])
def test_capped_decode_of_ranges_without_keys(dk, dv, dtype, monkeypatch):
    """Ragged lengths, so that up to 32 of 33 ranges hold no key; nobody writes such a range's values and nobody may
    read them: the partial results begin as NaN.  As many ranges as the merge takes at once (16), one more and fewer."""
    g, o, page, nh, nkv = torch.Generator().manual_seed(dv), ops(), 16, 6, 2
    lens = [1, 31, 64, 65, 300, 1056]
    B, per = len(lens), 66
    table = torch.randperm(B * per, generator=g).view(B, per).to(torch.int32)
    kc, vc = (torch.randn(B * per, nkv, page, d, generator=g).to(dtype) for d in (dk, dv))
    q, slots = torch.randn(B, nh * dk, generator=g).to(dtype), torch.randperm(B, generator=g).to(torch.int32)
    seq_len, sink = torch.tensor(lens, dtype=torch.int32), torch.randn(nh, generator=g)
    put = lambda t: t.to(DEV) if t is not None else None  # noqa: E731
    args, real = (nh, nkv, dk, dv, dk ** -0.5, 0.0, 0), torch.empty
    on = [put(t) for t in (q, kc, vc, table)]
    slots_d, len_d = put(slots), put(seq_len)
    for sk in (None, sink):
        want = R.attn_cap_decode(q, kc, vc, table, page, 0, slots, seq_len, *args, 1, sink=sk).double()
        for nsplit in (2, 15, 16, 17, 33):
            with monkeypatch.context() as m:
                m.setattr(torch, "empty", lambda *a, **k: real(*a, **k).fill_(float("nan")))
                got = o.attn_cap_decode(*on, page, 0, slots_d, len_d, *args, nsplit, sink=put(sk)).double().cpu()
            assert bool(torch.isfinite(got).all()), nsplit
            tol = 1e-5 if dtype == torch.float32 else 2 ** -8     # (as for the ranges and rounds above)
            assert float((got - want).abs().max()) <= tol * max(1.0, float(want.abs().max())), nsplit


@pytest.mark.parametrize("dtype, Rk, dr", [(torch.bfloat16, r, d) for r, d in ((16, 8), (64, 32), (128, 64), (208, 64), (256, 72), (320, 64),
                                                                             (384, 192), (512, 32), (512, 64))] +
                         [(torch.float32, 30, 8), (torch.float32, 64, 32), (torch.float32, 500, 12)])
def test_latent_single_tokens_over_widths_and_ranges(dtype, Rk, dr, monkeypatch):
    """Key widths on either side of the groups of 6 and 9 steps of 32 dims, the last step whole and in part; ranges
    without keys (up to 63 of 64) whose sums nobody writes and nobody may read: the partial results begin as NaN; as few
    and as many ranges as either way of combining them takes."""
    o, g, H, dv, page = ops(), torch.Generator().manual_seed(Rk + dr), 3, 40, 64
    lens = [1, 31, 33, 64, 300, 800, 1090]
    B, per = len(lens), 18
    table = torch.randperm(B * per, generator=g).view(B, per).to(torch.int32)
    cache = torch.randn(B * per, page, Rk + dr, generator=g).to(dtype)
    mfma = dtype == torch.bfloat16
    ct = cache[:, :, :Rk].transpose(1, 2).contiguous().unsqueeze(-1) if mfma else None
    qa = (torch.randn(B, H, Rk + dr, generator=g) * 0.3).to(dtype)
    y, wuv = torch.randn(B, H + 2, generator=g).to(dtype), (torch.randn(H * dv, Rk, generator=g) * Rk ** -0.5).to(dtype)
    slot, ln = torch.randperm(B, generator=g).to(torch.int32), torch.tensor(lens, dtype=torch.int32)
    put = lambda t: t.to(DEV) if t is not None else None  # noqa: E731
    want = R.latent_attn_decode(qa, y, wuv, 2, cache, table, page, 0, slot, ln, 0, H, dr, Rk, dv, 0.2, 0, 1).double()
    args = (put(qa), put(y), put(wuv), 2, put(cache), put(table), page, 0, put(slot), put(ln), 0, H, dr, Rk, dv, 0.2, 0)
    ct, real = put(ct), torch.empty
    for nsplit in (1, 3, 8, 9, 16, 24, 25, 35, 64):
        with monkeypatch.context() as m:
            m.setattr(torch, "empty", lambda *a, **k: real(*a, **k).fill_(float("nan")))
            got = o.latent_attn_decode(*args, nsplit, ct).double().cpu()
        assert bool(torch.isfinite(got).all()), nsplit
        # bfloat16: a weight's and a result's rounding (2^-9 each, 2^-8 beside the norm's share); float32 sums of up to 1,090
        assert float((got - want).norm() / want.norm()) < (2 ** -7 if mfma else 2e-5), nsplit


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dk, dv", [(128, 128), (64, 32)])
def test_capped_decode_of_infinite_values(dk, dv, dtype):
    """An infinity in the last key's value reaches its own dim as an infinity and no other: rounds of 32 keys that are
    full, that end early, and whole rounds past the range."""
    g, o, page, nh, nkv = torch.Generator().manual_seed(dk), ops(), 16, 4, 1
    lens = [8, 31, 32, 33, 64, 96, 128]
    B, per = len(lens), 8
    table = torch.arange(B * per, dtype=torch.int32).view(B, per)
    kc, vc = (torch.randn(B * per, nkv, page, d, generator=g).to(dtype) for d in (dk, dv))
    for b, n in enumerate(lens):
        vc[table[b, (n - 1) // page], 0, (n - 1) % page, 5] = float("inf")
    q = torch.randn(B, nh * dk, generator=g).to(dtype)
    put = lambda t: t.to(DEV)  # noqa: E731
    for nsplit in (1, 2, 5):
        got = o.attn_cap_decode(put(q), put(kc), put(vc), put(table), page, 0, put(torch.arange(B, dtype=torch.int32)),
                                put(torch.tensor(lens, dtype=torch.int32)), nh, nkv, dk, dv, dk ** -0.5, 0.0, 0, nsplit)
        got = got.float().cpu().view(B, nh, dv)
        assert bool((got[:, :, 5] == float("inf")).all()), nsplit
        assert bool(torch.isfinite(got[:, :, [d for d in range(dv) if d != 5]]).all()), nsplit


@pytest.mark.parametrize("nh, nkv, dk, dv", [(8, 2, 128, 128), (5, 1, 72, 40), (3, 3, 32, 8)])
def test_capped_decode_steps_of_16_keys(nh, nkv, dk, dv):
    """bfloat16 key counts around a wave's steps (16 keys, the next one 64 further on) that end in the first, the second
    and the third of them; a head has the same bits whether a block takes four heads, two or one."""
    g, o, page = torch.Generator().manual_seed(nh + dk), ops(), 32
    lens = [15, 16, 17, 63, 79, 80, 81, 143, 145, 257]
    B, per = len(lens), 9
    table = torch.randperm(B * per, generator=g).view(B, per).to(torch.int32)
    kc, vc = (torch.randn(B * per, nkv, page, d, generator=g).to(torch.bfloat16) for d in (dk, dv))
    q, slots = torch.randn(B, nh * dk, generator=g).to(torch.bfloat16), torch.randperm(B, generator=g).to(torch.int32)
    seq_len = torch.tensor(lens, dtype=torch.int32)
    on = [t.to(DEV) for t in (q, kc, vc, table, slots, seq_len)]
    want = R.attn_cap_decode(q, kc, vc, table, page, 0, slots, seq_len, nh, nkv, dk, dv, dk ** -0.5, 0.0, 0, 1).double()
    try:
        for nsplit in (1, 2):
            got = []
            for heads in (4, 2, 1):
                o._lib().illm_set_attn_cap_heads(heads)
                got.append(o.attn_cap_decode(*on[:4], page, 0, *on[4:], nh, nkv, dk, dv, dk ** -0.5, 0.0, 0, nsplit))
            assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
            # (the result's rounding, 2^-9, and the exponential's)
            assert float((got[0].double().cpu() - want).abs().max()) <= 2 ** -8 * max(1.0, float(want.abs().max())), nsplit
    finally:
        o._lib().illm_set_attn_cap_heads(0)


@pytest.mark.parametrize("N, K, K2", [(48, 128, 128), (72, 256, 128), (2048, 128, 896), (2048, 2048, 8192), (4128, 384, 256)])
def test_sum_of_two_products_of_few_rows(N, K, K2):
    """x . w^T + x2 . w2^T in one kernel: one piece of 128 k of either product, odd numbers of them, more
    pieces than waves and fewer, rows of W beyond the last tile; a row has the same bits alone, among 8 rows (half a tile a
    block) and among 16; an infinity in one row's second operand stays in that row."""
    o = ops()
    x, x2 = (rnd(16, k, dtype=torch.bfloat16, seed=i).to(DEV) for i, k in enumerate((K, K2)))
    w, w2 = ((rnd(N, k, seed=i + 2) * 0.1).to(torch.bfloat16).to(DEV) for i, k in enumerate((K, K2)))
    a, b = (o.decode_weight(t, "plain", True) for t in (w, w2))
    want = x.double() @ w.double().t() + x2.double() @ w2.double().t()
    got = {}
    for M in (1, 7, 8, 9, 16):
        pair = o.Product(x[:M], a), o.Product(x2[:M], b)
        assert o.linear_sum_fits(*pair)
        got[M] = o.linear_sum(*pair)
        # a float32 sum of K + K2 products
        assert float((got[M].double() - want[:M]).abs().max()) <= (K + K2) * 2.0 ** -24 * float((x.abs().double() @ w.abs().double().t()
                                                                              + x2.abs().double() @ w2.abs().double().t()).max())
        assert torch.equal(got[M][:1], got[1])
    assert torch.equal(got[16][:8], got[8])
    x2[3, 5] = float("inf")
    bad = o.linear_sum(o.Product(x[:8], a), o.Product(x2[:8], b))
    rows = [0, 1, 2, 4, 5, 6, 7]
    assert torch.equal(bad[rows], got[8][rows]) and not bool(torch.isfinite(bad[3]).any())
    assert not o.linear_sum_fits(o.Product(x, w), o.Product(x2, b)) and not o.linear_sum_fits(o.Product(x[:4], a), o.Product(x2, b))


@pytest.mark.parametrize("M, F, K, shape, tiles", [
    (1, 8, 128, 3, 1), (129, 136, 256, 3, 3), (257, 264, 384, 3, 10), (300, 2184, 128, 3, 70), (700, 40, 1024, 3, 3),
    (2100, 2056, 256, 1, 187), (500, 11008, 128, 0, 172), (300, 8328, 256, 2, 198), (1281, 10256, 384, 0, 486),
    (2313, 8200, 128, 0, 650), (2050, 11016, 128, 1, 957), (520, 10888, 128, 2, 430), (1000, 11016, 256, 3, 692)])
def test_gate_up_of_many_rows_in_turns(M, F, K, shape, tiles):
    """Gate and up with their activation over tiles in turns: every shape of tiles, less than a tile and remainders along both
    sides, one stage pair of K and more, two rounds of 256 blocks and more in every shape (so that loads run on into the next
    tile), infinities that stay in their rows and columns; the same rows have the same bits in every shape of tiles (other
    numbers of rows)."""
    import ctypes
    o, lib = ops(), ops()._lib()
    found = ctypes.c_int(-1)
    assert (lib.illm_gemm_turns_tiles(M, F, ctypes.byref(found)), found.value) == (tiles, shape)
    x = rnd(M, K, dtype=torch.bfloat16, seed=1).to(DEV)
    w = (rnd(2 * F, K, seed=2) * K ** -0.5).to(torch.bfloat16).to(DEV)

    def run(rows, limit):
        y = torch.full((rows + 1, F), 7.0, dtype=torch.bfloat16, device=DEV)
        assert lib.illm_gemm_turns_gate_up(o._p(x), o._p(w), o._p(y), rows, F, K, limit, 1.702, None) == 0
        assert bool((y[rows] == 7.0).all())
        return y[:rows]
    z = x.double() @ w.double().t()
    for limit in (0.0, 1.5):
        y = run(M, limit)
        g, u = z[:, :F], z[:, F:]
        if limit:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            want = g * torch.sigmoid(1.702 * g) * (u + 1)
        else:
            want = g * torch.sigmoid(g) * u
        # the result's rounding (half of the last of 8 bits: 2^-8 of a number that begins a power of two), and float32 sums of
        # K products (of at most 4 x 4 K^-1/2 each) through a slope of up to 1.1
        scale = want.abs() * 2.0 ** -8 + (g.abs() + u.abs() + 2) * K ** 0.5 * 16 * 2.0 ** -24
        assert bool(((y.double() - want).abs() <= 1.01 * scale).all())
        for rows in (1, M // 2 + 1, M):
            assert torch.equal(run(rows, limit), y[:rows])
    y, rows = run(M, 0.0), [i for i in range(M) if i != M // 3]
    x[M // 3, 5] = float("inf")
    bad = run(M, 0.0)
    assert torch.equal(bad[rows], y[rows]) and bool(torch.isfinite(bad[rows].float()).all())
    assert lib.illm_gemm_turns_gate_up(o._p(x), o._p(w), o._p(y), M, F, K + 64, 0.0, 1.0, None) != 0


@pytest.mark.parametrize("N, K", [(8, 4), (9, 256), (1, 1024), (70, 260), (33, 1284), (8200, 2052), (24, 5120)])
def test_float32_rows_of_every_number_have_the_same_bits(N, K):
    """A row of X gives the same sums alone and among 2, 3, 4, 5, 8, 9 and 16, each of which goes to its own number of rows a
    block: no whole piece of 256 k, one, pieces for some waves only, a last piece in part, odd and even numbers a wave,
    one piece at a time and the next one ahead (8,192 rows of W and more)."""
    o = ops()
    x, w = rnd(16, K, seed=1).to(DEV), rnd(N, K, seed=2).to(DEV)
    want = x.double() @ w.double().t()
    all16 = o.gemv_rows_f32(x, w, torch.float32)
    assert float((all16.double() - want).abs().max()) <= K * 2.0 ** -24 * float((x.abs().double() @ w.abs().double().t()).max())
    for M in (1, 2, 3, 4, 5, 8, 9):
        assert torch.equal(o.gemv_rows_f32(x[:M].contiguous(), w, torch.float32), all16[:M]), M


@pytest.mark.parametrize("F,K", [(5, 4), (96, 96), (131, 1028), (4100, 516), (33, 4096)])
def test_float32_products_of_few_rows_with_what_surrounds_them(F, K):
    """The norm in front, the activation behind and the add to the residual rows in the product's kernel: a part of a
    piece of K, odd numbers of columns, one piece at a time and the next ahead, 1 to 8 rows.  Against 64 bits within the
    bound of a sum of K float32 products; the add and the activation with the bits of the separate kernels; a row's bits
    whatever the number of rows."""
    o = ops()
    x, w = (rnd(8, K, seed=1) * 3.0).to(DEV), rnd(2 * F, K, seed=2).to(DEV)
    nw, eps = (rnd(K, seed=3) + 1.0).to(DEV), 1e-5
    xn = x.double() / torch.sqrt((x.double() ** 2).mean(1, keepdim=True) + eps) * nw.double()
    want = xn @ w.double().t()
    bound = (K + 8) * 2.0 ** -24 * (xn.abs() @ w.double().abs().t())           # a sum's K roundings and those of the norm
    left = o.norm_left(x[:8 if K <= 2048 else 4], (nw, eps), torch.float32)
    n = left.shape[0]
    got, want, bound, xn = o.linear(left, w), want[:n], bound[:n], xn[:n]
    assert bool(((got.double() - want).abs() <= bound).all())
    close(left.rows(), xn.float().cpu(), torch.float32)
    sums, acts = o.linear(x, w), {lim: o.gate_up_act(x, w, lim) for lim in (0.0, 1.25)}
    assert torch.equal(acts[0.0], o.silu_mul(sums)) and torch.equal(acts[1.25], o.clamped_swish_mul(sums, 1.25))
    assert torch.equal(o.gate_up_act(left, w), o.silu_mul(got))
    base = rnd(8, 2 * F, seed=4).to(DEV)
    for M in (1, 2, 3, 4, 5, 8):
        xm, into = x[:M].contiguous(), base[:M].clone()
        assert torch.equal(o.gate_up_act(xm, w), acts[0.0][:M])
        assert o.linear_add_fits(xm, w, into) == (M <= 4 or 2 * F <= 2048)
        if not o.linear_add_fits(xm, w, into):
            continue
        after = o.linear_add(xm, w, into, (torch.ones(2 * F, device=DEV), eps), torch.float32)
        assert torch.equal(into, base[:M] + sums[:M])
        assert (after is None) == (2 * F % 4 != 0) and (after is None or after.x is into)
        part = o.norm_left(xm, (nw, eps), torch.float32)
        assert (part is None) == (M > 4 and K > 2048)
        if part is not None:
            assert torch.equal(o.linear(part, w), got[:M]) and torch.equal(o.gate_up_act(part, w), o.silu_mul(got[:M]))
    assert o.norm_left(torch.zeros(9, K, device=DEV), (nw, eps), torch.float32) is None
    assert o.norm_left(x, (nw, eps), torch.bfloat16) is None and not o.linear_add_fits(x, w, base.to(torch.bfloat16))


@pytest.mark.parametrize("M,nh,nkv,hd,K,ring", [(1, 4, 2, 24, 96, 0), (3, 3, 1, 8, 1028, 2), (8, 16, 16, 128, 256, 0),
                                                (5, 60, 1, 128, 516, 3), (4, 2, 2, 120, 4096, 0),
                                                (2, 4, 4, 64, 2048, 0)])
@pytest.mark.parametrize("normed", [False, True])
def test_float32_qkv_rope_store_equals_the_three_steps(M, nh, nkv, hd, K, ring, normed):
    """Few float32 rows: the product with rotation and store in one kernel against product, then `rope_store` (whose two
    roundings a rotated value may take in another order)."""
    from inferllm_amd.parts.position import rotary_table
    o, page = ops(), 16
    table = rotary_table(777.0, hd, 300, "cpu").to(DEV)
    x, w = rnd(M, K, seed=1).to(DEV), rnd((nh + 2 * nkv) * hd, K, seed=2, std=0.1).to(DEV)
    x = o.norm_left(x, ((rnd(K, seed=3) + 1.0).to(DEV), 1e-5), torch.float32) if normed else x
    pos = torch.tensor([(37 * i + 5) % 290 for i in range(M)], dtype=torch.int32, device=DEV)
    slot = torch.randperm(M + 2, generator=torch.Generator().manual_seed(9))[:M].to(torch.int32).to(DEV)
    pt = torch.randperm((M + 2) * 19, generator=torch.Generator().manual_seed(4)).reshape(M + 2, 19).to(torch.int32).to(DEV)
    caches = [[c.to(DEV) for c in make_cache((M + 2) * 19, nkv, page, hd, torch.float32)] for _ in range(2)]
    assert o.qkv_rope_store_fits(x, w, hd)
    got = o.qkv_rope_store(x, w, table, pos, slot, *caches[0], pt, page, ring, nh, nkv, hd)
    want = o.linear(x, w)
    size = float(want.abs().max())
    o.rope_store(want, table, hd, 0, pos, slot, None, *caches[1], pt, page, ring, nh, nkv, hd)
    near = lambda a, b: float((a - b).abs().max()) <= 2.0 ** -22 * size
    assert near(got[:, :nh * hd], want[:, :nh * hd])
    for a, b in zip(*caches):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and near(torch.nan_to_num(a), torch.nan_to_num(b))
    assert not o.qkv_rope_store_fits(x, w, hd + 4)


@pytest.mark.parametrize("V", [1, 2, 1023, 1024, 1025, 2047, 2048, 2049])
@pytest.mark.parametrize("top_k,top_p", [(0, 1.0), (0, 0.8), (1500, 0.9)])
def test_sample_of_short_rows(V, top_k, top_p):
    """Rows whose scores stay in LDS, one and two ids a thread, and the first that do not: each draw's interval of the kept
    ids' distribution holds its number, equal scores and a score of minus infinity among them."""
    B = 5
    logits = rnd(B, V, seed=8, std=2.0)
    logits[1] = 0.0
    logits[2] = (logits[2] * 2).round() / 2
    logits[3, V // 2:V - 1] = float("-inf")
    seeds, counters = torch.tensor([3, 99, 12345, -7, 2**62], dtype=torch.int64), torch.arange(B, dtype=torch.int32)
    got = ops().sample(logits.to(DEV), 0.9, top_k, top_p, 1.0, None, seeds.to(DEV), counters.to(DEV)).cpu().tolist()
    for b in range(B):
        u = R.uniform(int(seeds[b]) & ((1 << 64) - 1), b)
        assert interval_ok(logits[b], got[b], u, 0.9, top_k, top_p, 1.0, None), (b, got[b], u)


@pytest.mark.parametrize("V, top_p", [(300, 1.0), (5000, 0.9), (20000, 0.95)])
def test_draws_outlive_their_samplers(V, top_p):
    """Samplers that go as soon as their draw is under way, behind work that is not done, and pinned buffers of the same size
    that are written at once: the draws use the seeds that they were given."""
    from inferllm_amd.sampling import Sampler, SamplingParams
    logits, params = rnd(8, V, seed=3).to(DEV), SamplingParams(temperature=1.5, top_p=top_p)
    want, kept = [], []
    for i in range(8):
        kept.append(Sampler(params, DEV))
        want.append(kept[-1](logits, list(range(100 * i, 100 * i + 8)), [i] * 8))
    a = torch.randn(4096, 4096, device=DEV)
    torch.cuda.synchronize()
    for _ in range(20):
        b = a @ a
    draws, others = [], []
    for i in range(8):
        more = i % 2                       # (a seed and a counter more than there are rows)
        draws.append(Sampler(params, DEV).draw(logits, list(range(100 * i, 100 * i + 8 + more)), [i] * (8 + more)))
        others.append(torch.empty(1024, dtype=torch.int32, pin_memory=True).fill_(7))
    assert [d.tokens() for d in draws] == want and b.shape == a.shape
    with pytest.raises(Exception):
        ops().sample(logits, 1.0, 0, 1.0, 1.0, None, torch.zeros(8, dtype=torch.int64, pin_memory=True),
                     torch.zeros(8, dtype=torch.int32, device=DEV))


def test_gates_far_below_zero_in_turns():
    """g / (1 + e^-g) up is a normal number until e^-g is infinite: gates down to -88.5 by tiles in turns, and a limit's
    slope of 1.702, against 64 bits within the result's rounding (2^-8 where a power of two begins) and float32's."""
    o, lib = ops(), ops()._lib()
    M, F, K = 5, 264, 128
    gates = torch.linspace(-88.5, 40.0, F).mul(2 / K).bfloat16().mul(K / 2)      # exact sums of K / 2 equal products
    w = torch.zeros(2 * F, K)
    w[:F, ::2], w[F:, 1] = (gates / (K / 2))[:, None], 1.0
    x, w, y = torch.ones(M, K, dtype=torch.bfloat16, device=DEV), w.bfloat16().to(DEV), torch.empty(M, F, dtype=torch.bfloat16, device=DEV)
    for limit, slope, up in ((0.0, 1.0, 1.0), (50.0, 1.702, 2.0)):
        assert lib.illm_gemm_turns_gate_up(o._p(x), o._p(w), o._p(y), M, F, K, limit, 1.702, None) == 0
        z = gates.double() * torch.tensor(slope).double()
        want = gates.double() / (1 + torch.exp(-z)) * up
        want[torch.exp(-z.float()).isinf()] = 0.0
        assert float(want[0].abs()) > 1e-37 or slope > 1
        assert bool(((y.double().cpu() - want).abs() <= (2.0 ** -8 + 2e-5) * want.abs()).all())


def test_gate_up_of_many_rows_under_plans(monkeypatch):
    """One kernel by default; the product and its activation, to the bit, under a plan saved before that kernel and where its
    last round of blocks is nearly empty."""
    from inferllm_amd.kernels.plan import Plan
    o = ops()
    old = {k: v for k, v in Plan.fixed().to_dict().items() if k != "turns"}
    for M, F, K, plan, one in ((500, 8192, 512, Plan.fixed(), True), (500, 8192, 512, Plan.from_dict(old), False),
                               (520, 13824, 4096, Plan.fixed(), False)):
        x = rnd(M, K, dtype=torch.bfloat16, seed=4).to(DEV)
        w = (torch.randn(2 * F, K, device=DEV) * K ** -0.5).to(torch.bfloat16)
        monkeypatch.setattr(o, "_plan", plan)
        assert o.gate_up_turns_fits(x, w) == one
        assert torch.equal(o.gate_up_act(x, w), o.silu_mul(o.linear(x, w))) != one
