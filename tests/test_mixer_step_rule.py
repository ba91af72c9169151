"""Up to how many heads of rows single tokens go through a mixer in one kernel (csrc/mixer_steps.hip)."""
import pytest
import torch

import plain_dotorax as P
from dotorax_tiny import _gla, single, weights64, write_model
from tiny import random_ids

from inferllm_amd.kernels import ops


# (kind, dk, dv, rank of the decays), heads of rows measured faster in one kernel, and slower
@pytest.mark.parametrize("call, faster, slower", [
    (("memory", 32, 32, 0), 512, 1024), (("memory", 32, 64, 0), 1024, 4096), (("memory", 128, 128, 0), 8192, None),
    (("gated_linear", 32, 64, 16), 1024, 4096), (("gated_linear", 64, 128, 16), 4096, 8192), (("gated_linear", 64, 64, 32), 1024, 4096),
    (("gated_linear", 64, 128, 64), 512, 1024), (("gated_linear", 128, 128, 128), None, 16), (("gated_linear", 64, 128, 256), None, 16),
    (("state_space", 16, 128, 0), 256, 512), (("state_space", 64, 64, 0), 512, 1024), (("state_space", 128, 64, 0), 4096, 8192),
    (("state_space", 128, 128, 0), 8192, None)])
def test_both_sides_of_the_line(call, faster, slower):
    most = ops.mixer_step_heads(*call)
    assert (faster is None or faster <= most) and (slower is None or most < slower)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [3, 70])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_decays_of_a_high_rank_have_a_product_of_their_own(tmp_path, n, dtype):
    """Steps of single tokens that the one kernel leaves out, up to 64 rows and above."""
    import inferllm_amd as I
    config = single("gla", _gla(3, 16, 24, 5.0, 96))
    assert ops.mixer_step_heads("gated_linear", 16, 24, 96) == 0
    d = write_model(tmp_path, config, seed=8, dtype=getattr(torch, dtype))
    w = weights64(d)
    reqs = [random_ids(4 + i % 9, config["vocab"], 90 + i) for i in range(n)]
    eng = I.Engine.from_pretrained(d, dtype=dtype, device="cuda:0", max_batch=n, max_seq_len=128, decode_copies=dtype == "bfloat16")
    slots, errs = [eng.alloc_slot() for _ in reqs], []
    eng.step([I.StepEntry(s, r[:-2], []) for s, r in zip(slots, reqs)])
    for t in (2, 1):
        out = eng.step([I.StepEntry(s, [r[-t]], [0]) for s, r in zip(slots, reqs)]).double().cpu()
        for o, r in zip(out, reqs):
            want = P.forward(config, w, r)
            errs.append(float((o - want[-t]).abs().max() / want.abs().max()))
    # the designs' own budgets: float32 3e-5 of the largest logit; bfloat16 4e-2 for all rows but a few, the median half of it
    if dtype == "float32":
        assert max(errs) < 3e-5
    else:
        assert sum(not e < 4e-2 for e in errs) <= max(1, len(errs) // 20) and sorted(errs)[len(errs) // 2] < 2e-2
