"""The rules that send a call to one kernel or another, and what the library refuses before it launches anything:
no GPU is needed for either."""
import pytest
import torch

from inferllm_amd.kernels import ops

ERR_ARG = 1
AT = 1 << 20                                               # an address that nothing reads: the call is refused


def test_the_cut_product_is_given_only_what_it_takes():
    """`linear_cut_fits` against the library's own limits: sizes near 4 GiB and views that begin off a 16-byte
    address go to the product they took before."""
    def fits(M, N, K, x_at=0, w_at=0, **kw):
        x = torch.empty(x_at + M * K, dtype=torch.bfloat16, **kw)[x_at:].view(M, K)
        w = torch.empty(w_at + N * K, dtype=torch.bfloat16, **kw)[w_at:].view(N, K)
        return ops.linear_cut_fits(x, w)

    lib = ops._lib()
    rc = lambda M, N, K, X=AT, W=AT, Y=AT: lib.illm_gemm_tiles_planes(X, W, Y, M, N, K, 1, None)  # noqa: E731
    assert fits(129, 4096, 4096) and fits(256, 4096, 4096) and not fits(128, 4096, 4096) and not fits(257, 4096, 4096)
    # more than 192 rows, too few blocks: the vendor's product
    assert fits(192, 1024, 4096) and not fits(193, 1024, 4096) and fits(193, 1536, 4096) and fits(256, 256, 4096)
    # the last K that the planes' offsets reach (N + 63 rows of W, 256 of X), and the next
    for N in (1536, 4096):
        last = (0xffffffff - 1) // (2 * (N + 63)) // 64 * 64
        assert fits(200, N, last, device="meta") and not fits(200, N, last + 64, device="meta")
        assert rc(200, N, last + 64) == ERR_ARG
    assert rc(150, 4, (0xffffffff // 512 // 64 + 1) * 64) == ERR_ARG
    assert not fits(150, 4, (0xffffffff // 512 // 64 + 1) * 64, device="meta")
    for off in (1, 4):                                     # 2 and 8 bytes off
        assert not fits(129, 2048, 4096, x_at=off) and not fits(129, 2048, 4096, w_at=off)
    for off in (2, 4, 8):
        assert rc(129, 64, 4096, X=AT + off) == rc(129, 64, 4096, W=AT + off) == rc(129, 64, 4096, Y=AT + off) == ERR_ARG
    # rows that are columns of wider ones are copied first
    wide = torch.empty(129, 4104, dtype=torch.bfloat16)[:, 1:4097]
    assert ops.linear_cut_fits(wide, torch.empty(2048, 4096, dtype=torch.bfloat16))


def test_the_experts_tiles_of_128_pairs_refuse_other_addresses():
    """Rows and matrices go straight into LDS 16 bytes a lane: what does not lie on 16 bytes is refused (the caller
    groups such pairs for the kernels of 16 to 64)."""
    call = lambda rows=128, X=AT, W=AT, Y=AT: ops._lib().illm_moe_rows_mfma(  # noqa: E731
        X, 1, W, 0, rows, AT, AT, 1, Y, 64, 64, 0, 0.0, None, None)
    for off in (2, 8):
        assert call(X=AT + off) == call(W=AT + off) == call(Y=AT + off) == ERR_ARG


def test_the_experts_tiles_of_128_pairs_are_taken_where_they_pay():
    """Stacks that leave compute units idle, or whose matrices are small, keep the smaller tiles up to 12 pairs an expert, of
    few experts up to 24 (experts, F, E -> the fewest pairs an expert in tiles of 128, measured to be no slower from there on)."""
    rows = lambda NE, F, E, p: ops._moe_tiling(torch.bfloat16, E, F, int(p * NE), NE)[1]  # noqa: E731
    for NE, F, E, first in ((64, 1408, 2048, 6), (32, 4096, 2048, 6), (8, 14336, 4096, 6), (24, 1536, 1536, 12), (128, 768, 2048, 6),
                            (256, 256, 1024, 6), (16, 512, 512, 12), (4, 1024, 1024, 24), (8, 2048, 1024, 12), (16, 2048, 2048, 12),
                            (2, 4096, 4096, 24), (32, 2048, 4096, 3), (8, 8192, 4096, 6), (64, 1024, 1024, 6)):
        for p in (1, 1.5, 2, 3, 4, 6, 8, 12, 16, 24, 64, 500):
            assert (rows(NE, F, E, p) == 128) == (p >= first), (NE, F, E, p)


def test_float32_rows_in_pieces_that_the_product_in_parts_takes():
    """Any number of rows, on and beyond what the library takes in one call (4 GiB of scratch, 65,535 tiles): pieces
    that hold every row once, each with no more scratch than the limit says, and no row refused that another product
    had taken."""
    lib = ops._lib()
    for K in (512, 2048, 4096, 11008, 1 << 18):
        for M in (1, 127, 128, 129, 2048, 4064, 4065, 65536, (1 << 20) - 128, 1 << 20, (1 << 20) + 1, 3000000):
            pieces = ops._f32_split_pieces(M, K)
            assert [r for r, _ in pieces] == [0] + [r + n for r, n in pieces][:-1] and sum(n for _, n in pieces) == M
            for r, n in pieces:
                rows = lib.illm_gemm_f32_split_rows(n)
                assert r % 128 == 0 and n <= rows < n + 128 and rows // 16 <= 65535
                assert rows * K * 6 <= max(ops.F32_SPLIT_SCRATCH, 128 * 6 * K) <= 0xffffffff
    x, w = torch.empty((1 << 20) + 1, 512, device="meta"), torch.empty(16384, 512, device="meta")
    assert ops.gemm_f32_split_fits(x, w) and ops.gemm_f32_split_pays(x, w)
    # planes and their scratch are bounded too
    for M, N, K in ((4096, 1024, 11008), (16384, 1024, 2048), (2048, 4096, 11008), (300, 1024, 1 << 18)):
        if lib.illm_gemm_f32_split_planes(M, N, K):
            planes = -(-K // 32 // lib.illm_gemm_f32_split_per(M, N, K))
            assert planes * M * N * 4 <= 1 << 27 and 6 * M * K <= ops.F32_SPLIT_SCRATCH


def test_a_slot_is_zeroed_on_its_tensors_device(monkeypatch):
    """A new sequence's state is cleared on the tensors' own card and its stream, whichever card is the current one."""
    seen, current = [], ["another"]

    class on:
        def __init__(self, device):
            self.device = device

        def __enter__(self):
            self.before, current[0] = current[0], self.device

        def __exit__(self, *exc):
            current[0] = self.before

    class library:
        @staticmethod
        def illm_zero_pieces(at, size, n, stream):
            seen.append((list(at), list(size), n, stream))
            return 0
    monkeypatch.setattr(torch.cuda, "device", on)
    monkeypatch.setattr(ops, "_gpu", lambda *t: None)
    monkeypatch.setattr(ops, "_lib", lambda: library)
    monkeypatch.setattr(ops, "_stream", lambda: ("stream of", current[0]))
    a, b = torch.zeros(4, 3, dtype=torch.float32), torch.zeros(4, 5, 2, dtype=torch.bfloat16)
    ops.zero_slot([a, b], 2)
    assert seen == [([a[2].data_ptr(), b[2].data_ptr()], [12, 20], 2, ("stream of", a.device))] and current == ["another"]


def test_the_cut_product_refuses_float32_rows_with_another_matrix(monkeypatch):
    """float32 rows with a bfloat16 matrix, or one of another width, are refused before anything reads them as float32."""
    monkeypatch.setattr(ops, "_gpu", lambda *t: None)
    monkeypatch.setattr(ops, "_f32_split", lambda x, w, dtype, S: torch.zeros((x.shape[0], w.shape[0]) if S == 1
                                                                             else (S or 4, x.shape[0], w.shape[0])))
    x = torch.zeros(140, 2048)
    for w in (torch.zeros(1024, 2048, dtype=torch.bfloat16), torch.zeros(1024, 1024)):
        with pytest.raises(ops.KernelError):
            ops.linear_cut(x, w)
    for splits, planes in ((0, 4), (1, 1), (3, 3)):
        assert ops.linear_cut(x, torch.zeros(1024, 2048), splits).shape == (planes, 140, 1024)


def test_a_draw_keeps_the_numbers_that_its_kernel_reads(monkeypatch):
    """Seeds and counters in pinned memory are there until the kernel that reads them has run, also where the sampler and
    the draw are gone before: here a buffer is let go of once the event behind its kernel has passed, and no sooner."""
    import gc
    import weakref

    import numpy as np

    from inferllm_amd.sampling import Sampler, SamplingParams
    events = []

    class event:
        def __init__(self):
            self.passed = False
            events.append(self)

        def query(self):
            return self.passed

    class library:
        @staticmethod
        def illm_sample(*a):
            return 0
    monkeypatch.setattr(torch.cuda, "Event", event)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.Tensor, "is_pinned", lambda t: True)
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda t: True))
    monkeypatch.setattr(ops, "record", lambda e: None)
    monkeypatch.setattr(ops, "_gpu", lambda *t: None)
    monkeypatch.setattr(ops, "_lib", lambda: library)
    monkeypatch.setattr(ops, "_stream", lambda: None)
    refs = []
    for i in range(3):
        sampler, numbers = Sampler(SamplingParams(temperature=0.8), "cuda:0"), np.zeros(1024, np.int32)
        sampler._stages = [torch.from_numpy(numbers)] * 4
        sampler._back = [torch.empty(2, dtype=torch.int32)] * 4
        refs.append(weakref.ref(numbers))
        sampler.draw(torch.zeros(2, 8), [1, 2], [0, 0])
        del sampler, numbers
        gc.collect()
        assert [r() is not None for r in refs] == ([True], [True, True], [False, True, True])[i]
        events[0].passed = i == 1
    events[1].passed = events[2].passed = True
    ops.keep_until(event(), torch.zeros(1))
    gc.collect()
    assert [r() for r in refs] == [None] * 3
    ops._kept.clear()


def test_float32_products_of_few_rows_refuse_what_is_not_there():
    """The product with what surrounds it and the one with rotation and store: a null operand, an empty table, sizes that
    they do not take, or heads whose rows pass the numbers' range, are refused before anything is launched."""
    lib = ops._lib()
    fused = dict(X=AT, W=AT, Y=AT, M=4, N=64, K=64, norm_w=AT, eps=1e-5, epi=0, limit=0.0, alpha=1.0, stream=None)
    qkv = dict(X=AT, W=AT, Y=AT, M=4, K=64, norm_w=AT, eps=1e-5, cos_sin=AT, max_pos=32, row_pos=AT, row_slot=AT, kcache=AT,
               vcache=AT, page_table=AT, table_stride=2, page_size=16, ring=0, nh=2, nkv=1, hd=64, stream=None)
    for entry, good, bad in (
            (lib.illm_gemv_rows_f32_fused, fused, dict(X=None, W=None, Y=None, M=9, N=0, K=66, epi=3)),
            (lib.illm_gemv_qkv_f32, qkv, dict(X=None, W=None, Y=None, M=9, K=66, cos_sin=None, max_pos=0, row_pos=None,
                                              row_slot=None, kcache=None, vcache=None, page_table=None, table_stride=0,
                                              page_size=0, nh=1 << 25, nkv=0, hd=60))):
        for name, value in bad.items():
            assert entry(*dict(good, **{name: value}).values()) == ERR_ARG, name


def test_a_pinned_plan_keeps_the_gate_and_up_products_that_it_was_made_with():
    """A plan saved before gate and up of many rows had a kernel of their own says nothing of it and keeps the products;
    so do the matrices that a plan made by hand has cuts for.  What is saved now comes back as it was."""
    import json

    from inferllm_amd.kernels.plan import FIXED_CUTS, Plan
    shape, cut = (22016, 4096), {(8, 22016, 4096): (8192,)}
    old = Plan.fixed().to_dict()
    old["cuts"].append([[8, 22016, 4096], [8192]])
    del old["turns"]
    old = Plan.from_dict(json.loads(json.dumps(old)))
    assert old.cuts[8, 22016, 4096] == (8192,) and all(old.keeps_products(M, *shape) for M in (256, 1000, 2048))
    for plan in (Plan.fixed(), Plan.fixed(measure=True), Plan(), Plan(measure=True), Plan(cuts=FIXED_CUTS), Plan(cuts=cut, turns=True)):
        assert plan.turns is True and not any(plan.keeps_products(M, *shape) for M in (256, 1000, 2048))
    own = Plan(cuts={**FIXED_CUTS, **cut})
    assert [own.keeps_products(M, *shape) for M in (1792, 1793, 2048, 2049)] == [False, True, True, False]
    measured = Plan(measure=True)
    measured.cuts.update(cut)                          # (timed for another matrix of that shape)
    for plan in (old, own, measured, Plan.fixed()):
        again = Plan.from_dict(json.loads(json.dumps(plan.to_dict())))
        assert again == plan and [again.keeps_products(M, *shape) for M in (1000, 2048)] == [plan.keeps_products(M, *shape)
                                                                                              for M in (1000, 2048)]
    assert old != Plan.from_dict(dict(old.to_dict(), turns=True))


@pytest.mark.parametrize("F, K, one_kernel, two", [
    (11008, 4096, (256, 500, 768, 1000, 2048, 2112, 2305, 2816, 2881, 9061), (255, 2113, 2200, 2304, 2817, 2880)),
    (14336, 4096, (256, 512, 577, 1000, 9061), (513, 576)), (13824, 5120, (500, 640, 2048), (528, 576)),
    (6144, 3072, (384, 1296, 1344, 2048), (256, 383)), (8192, 4096, (288, 500, 2905), (256, 287)),
    (2816, 2048, (838, 2048), (500, 837)), (1024, 1024, (2304, 9061), (1000, 2303))])
def test_gate_up_and_activation_are_one_kernel_where_that_is_the_faster_way(F, K, one_kernel, two):
    """Rows and outputs enough, and no last round that is nearly empty: both sides of every line."""
    assert all(ops.turns_pays(M, F, K) for M in one_kernel) and not any(ops.turns_pays(M, F, K) for M in two)


def test_tuning_times_a_product_that_has_the_shape_of_gate_and_up():
    """Two matrices of one shape, one of them gate and up: the other's ways are those that are timed, whichever comes first."""
    from inferllm_amd.kernels import tune
    a, b = torch.zeros(64, 32, dtype=torch.bfloat16), torch.zeros(64, 32, dtype=torch.bfloat16)

    class part:
        def __init__(self, *listed):
            self.tunables = lambda: listed

    for parts in ([part(("gate_up", a, {})), part(("plain", b, {}))], [part(("plain", b, {}), ("gate_up", a, {}))]):
        model = type("model", (), {"every_part": staticmethod(lambda: parts)})
        (kind, w), = tune.matrices(type("engine", (), {"model": model})).values()
        assert kind == "plain" and w is b
