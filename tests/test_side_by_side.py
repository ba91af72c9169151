"""Mixers side by side in either order through the step function on the CPU, with the GPU kernels replaced by their plain torch
stand-ins (tests/kernel_refs.py)."""
import pytest
import torch

import kernel_refs
import plain_dotorax as P
from dotorax_tiny import MIXED, weights64, write_model
from tiny import random_ids

import inferllm_amd as I
from inferllm_amd.cache import CacheManager
from inferllm_amd.engine import DecoderModel, StepEntry, StepRunner
from inferllm_amd.weights.loader import stored_shapes


@pytest.mark.parametrize("swapped", [False, True])
def test_attention_on_either_side_of_a_recurrent_unit(tmp_path, monkeypatch, swapped):
    """Only on the left do attention's columns begin a matrix stacked with the recurrent unit's; on the right each has its own."""
    kernel_refs.patch(monkeypatch)
    d = write_model(tmp_path, MIXED, seed=2)
    w = weights64(d)
    spec = I.load_config(d).with_tensor_shapes(stored_shapes(d)).to_spec()
    pairs = [l.mixer.params for l in spec.layers if l.mixer.kind == "side_by_side"]
    for p in pairs:
        if swapped:
            p["left"], p["right"] = p["right"], p["left"]
            p["left_scale"], p["right_scale"] = p["right_scale"], p["left_scale"]
    model = DecoderModel(spec)
    model.load({k: v.to(torch.float32) for k, v in w.items() if k in model.wants()})
    stacked = [l.mixer.w_in is not None for l in model.layers if hasattr(l.mixer, "right_column")]
    cache = CacheManager(model.kv_lines(), model.state_lines(), max_tokens=512, max_slots=2, max_seq_len=256,
                         dtype=torch.float32, device="cpu", poison_freed=True)
    r = StepRunner(model, cache, torch.float32, torch.device("cpu"), use_graphs=False)
    ids = random_ids(60, MIXED["vocab"], 7)
    want, s = P.forward(MIXED, w, ids), cache.alloc_slot()
    got = torch.cat([r.step([StepEntry(s, ids[a:b], list(range(b - a)))]) for a, b in ((0, 50), (50, 58), (58, 59), (59, 60))])
    assert (got.double() - want).abs().max() < 1e-4
    assert stacked == [not swapped] * len(pairs) and pairs
