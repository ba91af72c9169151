"""What this library is timed on: passes through `Engine.step` and `Sampler.draw` as a serving
program drives them, from a tiny float32 model whose steps cost little but their launches to
prompts of nine thousand tokens.

A case names a model shape, a kind of pass, the sequences and their lengths:

  "decode"    `steps` steps of one token for every sequence of a batch whose contexts are in the
              cache already; the tokens come from the seed (a replay), every step's logits are
              handed to the sampler and its tokens are read one step later, as the generation loop
              does; the steps are then taken back, so that a pass can be repeated
  "prompts"   whole prompts in one step, the first token chosen for each
  "generate"  both: the prompts, then `steps` steps of one token

Weights are random, drawn from the seed here, so that `exact` can draw the same ones, and rounded
to the engine's type: matrices N(0, 0.02), norm weights 1 + N(0, 0.01) as the library's own rule has
them; in the LLaMA shapes the embedding is N(0, 1) and the matrices that write the residual stream
are divided by sqrt(2 layers), as deep decoders are initialised (with 0.02 everywhere the rounding
of bfloat16 activations grows to 5 % of a logit through 32 layers, which would hide a fault).
LLaMA shapes have all their layers; the other designs have the four layers that the benchmark gives
them.
"""
import hashlib
import math

import torch

LLAMA2_7B = {"architectures": ["LlamaForCausalLM"], "hidden_size": 4096, "intermediate_size": 11008,
             "num_hidden_layers": 32, "num_attention_heads": 32, "num_key_value_heads": 32, "head_dim": 128,
             "vocab_size": 32000, "rms_norm_eps": 1e-5, "rope_theta": 10000.0,
             "max_position_embeddings": 4096, "tie_word_embeddings": False, "bos_token_id": 1, "eos_token_id": 2}
LLAMA3_8B = dict(LLAMA2_7B, intermediate_size=14336, num_key_value_heads=8, vocab_size=128256,
                 rope_theta=500000.0, max_position_embeddings=8192)
TINY = dict(LLAMA2_7B, hidden_size=96, intermediate_size=256, num_hidden_layers=3, num_attention_heads=4,
            num_key_value_heads=2, head_dim=24, vocab_size=320, rope_theta=500000.0,
            max_position_embeddings=256, eos_token_id=[2, 3])


def _rabapel(width=2048, heads=16, ff=8192):
    """Latent attention; a dense feed-forward and 6 of 64 routed experts in turn."""
    mixer = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5,
             "rot": {"base": 10000.0, "dims": 64,
                     "scaling": {"factor": 40.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
    moe = {"kind": "moe", "expert": {"ff": 1408}, "router": {"experts": 64, "identity": 0, "top": 6},
           "shared": {"ff": 2816}}
    return {"architecture": "Rabapel", "vocab": 32000, "width": width, "norm": {"eps": 1e-6},
            "embedding": {"scale": 1.0}, "max_positions": 8192,
            "layers": [{"type": "latent_attention", "mixer": dict(mixer),
                        "mlp": dict(moe) if i % 2 else {"kind": "dense", "ff": ff}} for i in range(4)]}


def _sabipel(width=2048, heads=16, kv_heads=4):
    """State-space, chunked attention, matrix memory, chunked attention; dense feed-forwards."""
    ssm = {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}
    mem = {"heads": heads, "dim": 128, "vdim": 128, "gate_cap": 15.0}
    att = {"heads": heads, "kv_heads": kv_heads, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
           "mask": {"size": 1024}, "v_mix": True}
    kinds = [("mamba2", ssm), ("attention", att), ("mlstm", mem), ("attention", att)]
    return {"architecture": "Sabipel", "vocab": 32000, "width": width, "max_positions": 8192, "norm": {"eps": 1e-6},
            "embedding": {"scale": 1.0, "bigram": {"buckets": 65521, "mul_prev": 37, "mul_cur": 11}},
            "layers": [{"type": k, "mixer": dict(m), "mlp": {"kind": "dense", "ff": 4 * width}} for k, m in kinds]}


def _dotorax(width=2048, heads=16, kv_heads=4):
    """Rotated attention, gated linear attention, a window with pooled blocks beside a recurrent
    unit, attention on the first layer's keys; gated feed-forwards behind a short convolution."""
    att = {"heads": heads, "kv_heads": kv_heads, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
           "rot": {"base": 10000.0, "dims": 64}}
    gla = {"heads": heads, "dim": 64, "vdim": 128, "tau": 16.0, "rank": 16}
    par = {"left": dict(att, mask={"size": 1024, "pool": 8}),
           "right": {"width": width, "blocks": 16, "conv": 4}, "left_scale": 1.0, "right_scale": 1.0}
    mlp = {"kind": "dense", "ff": 8 * width // 3 // 256 * 256, "limit": 7.0}
    kinds = [("attention", att), ("gla", gla), ("parallel", par), ("attention", dict(att, kv_from=0))]
    return {"architecture": "Dotorax", "vocab": 32000, "width": width, "max_positions": 8192,
            "norm": {"eps": 1e-6}, "residual_mult": 0.5, "canon": {"taps": 3},
            "layers": [{"type": k, "mixer": dict(m), "mlp": dict(mlp)} for k, m in kinds]}


MODELS = {"tiny": TINY, "llama2-7b": LLAMA2_7B, "llama3-8b": LLAMA3_8B,
          "rabapel": _rabapel(), "sabipel": _sabipel(), "dotorax": _dotorax()}


def _case(model, kind, batch, shortest, longest, steps=0, dtype="bfloat16", temperature=0.0, top_k=0, top_p=1.0,
          repeat_penalty=1.0, **more):
    return dict(more, model=model, dtype=dtype, kind=kind, batch=batch, shortest=shortest, longest=longest,
                steps=steps, temperature=temperature, top_k=top_k, top_p=top_p, repeat_penalty=repeat_penalty)


def listed():
    return [
        # a first try of the library, or a test suite: a model whose steps are launches and nothing
        # else; the small ragged batch at temperature 0.8
        _case("tiny", "generate", 3, 2, 11, 6, "float32", temperature=0.8, name="tiny_f32_generate_b3"),
        # one user at a chat prompt, with the command line's usual sampling
        _case("llama2-7b", "decode", 1, 512, 512, 4, temperature=0.1, top_k=40, top_p=0.95, repeat_penalty=1.1,
              name="7b_decode_b1_chat"),
        # a handful of users, greedy
        _case("llama2-7b", "decode", 8, 512, 512, 4, name="7b_decode_b8"),
        # a full batch, greedy
        _case("llama2-7b", "decode", 64, 512, 512, 4, name="7b_decode_b64"),
        # a server's live sequences, of very different lengths, grouped heads, a wide vocabulary
        _case("llama3-8b", "decode", 16, 64, 4096, 4, temperature=0.8, top_p=0.95, name="8b_decode_b16_ragged"),
        # the first token of a short question
        _case("llama2-7b", "prompts", 1, 160, 160, name="7b_prompt_160"),
        # the first token of a long prompt
        _case("llama2-7b", "prompts", 1, 2048, 2048, name="7b_prompt_2048"),
        # a batch of prompts that arrived together, ragged, 9,061 tokens
        _case("llama3-8b", "prompts", 8, 64, 4096, name="8b_prompts_b8_ragged"),
        # the true 32-bit path: short prompts and the first answer tokens
        _case("llama2-7b", "generate", 4, 17, 129, 4, "float32", name="7b_f32_generate_b4"),
        # another design each: latent attention with routed experts, state-space and matrix-memory
        # layers, gated linear attention and a recurrent unit; a ragged batch from prompts to answers
        _case("rabapel", "generate", 8, 61, 1024, 16, name="rabapel_generate_b8"),
        _case("sabipel", "generate", 8, 61, 1024, 16, name="sabipel_generate_b8"),
        _case("dotorax", "generate", 8, 61, 1024, 16, name="dotorax_generate_b8"),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    sampling = rng.choice([{}, {}, {"temperature": 0.8, "top_p": 0.95}, {"temperature": 0.7},
                           {"temperature": 0.1, "top_k": 40, "top_p": 0.95, "repeat_penalty": 1.1}])
    what = rng.choice(["tiny", "decode", "decode", "decode", "short", "long", "long", "f32", "other", "other"])
    if what == "tiny":
        longest = _log(rng, 4, 128)
        return _case("tiny", "generate", _log(rng, 1, 8), rng.randint(1, longest), longest, rng.randint(2, 12),
                     "float32", **sampling)
    llama = rng.choice(["llama2-7b", "llama3-8b"])
    if what == "decode":
        batch = _log(rng, 1, 64)
        longest = _log(rng, 100, 4000 if batch <= 16 else 600)
        return _case(llama, "decode", batch, rng.choice([longest, _log(rng, 32, longest)]), longest, 4, **sampling)
    if what == "short":
        return _case(llama, "prompts", 1, *[_log(rng, 5, 300)] * 2, **sampling)
    if what == "long":
        batch = _log(rng, 1, 8)
        longest = _log(rng, 300, 4000)
        shortest = rng.choice([longest if longest * batch <= 9000 else 9000 // batch, _log(rng, 32, min(longest, 128))])
        return _case(llama, "prompts", batch, min(shortest, longest), longest, **sampling)
    if what == "f32":
        longest = _log(rng, 17, 150)
        return _case("llama2-7b", "generate", _log(rng, 1, 8), rng.randint(9, longest), longest, 4, "float32", **sampling)
    longest = _log(rng, 100, 1500)
    return _case(rng.choice(["rabapel", "sabipel", "dotorax"]), "generate", _log(rng, 1, 16), _log(rng, 17, longest),
                 longest, rng.randint(4, 16), **sampling)


# ---------------------------------------------------------------- inputs
def _lengths(case):
    """The sequences' context lengths: from the longest to the shortest in equal factors."""
    b, lo, hi = case["batch"], case["shortest"], case["longest"]
    if b == 1:
        return [hi]
    return [int(round(hi * (lo / hi) ** (i / (b - 1)))) for i in range(b)]


def _tokens(case, seed):
    """(contexts, the token every sequence is given in every step)."""
    cfg = MODELS[case["model"]]
    vocab = cfg.get("vocab_size") or cfg["vocab"]
    g = torch.Generator().manual_seed(seed * 2 + 1)
    ids = lambda n: torch.randint(0, vocab, (n,), generator=g).tolist()  # noqa: E731
    return [ids(n) for n in _lengths(case)], [ids(case["batch"]) for _ in range(case["steps"])]


def _weight(seed, name, shape, ones, dtype, layers=0):
    """One tensor of the model: a function of the seed, its name and, in a LLaMA shape, the number
    of layers."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int.from_bytes(hashlib.sha256(f"{seed} {name}".encode()).digest()[:7], "little"))
    t = torch.randn(tuple(shape), generator=g, dtype=torch.float32, device="cuda")
    if ones:
        return t.mul_(0.01).add_(1.0).to(dtype)
    if layers and "embed" not in name:
        t.mul_((2 * layers) ** -0.5 if "o_proj" in name or "down_proj" in name else 1.0)
    return t.mul_(1.0 if layers and "embed" in name else 0.02).to(dtype)


def prepare(case, seed):
    from inferllm_amd import Engine, StepEntry
    from inferllm_amd.config.registry import config_from_dict
    from inferllm_amd.engine.model import expected_tensors
    from inferllm_amd.sampling import Sampler, SamplingParams
    config = config_from_dict(MODELS[case["model"]])
    dtype = getattr(torch, case["dtype"])
    weights = {n: _weight(seed, n, w.shape, w.init == "ones_normal", dtype, MODELS[case["model"]].get("num_hidden_layers", 0))
               for n, w in expected_tensors(config.to_spec()).items() if not w.optional}
    contexts, fed = _tokens(case, seed)
    room = sum((len(c) + case["steps"] + 63) // 64 * 64 for c in contexts)
    eng = Engine(config, weights, case["dtype"], max_batch=case["batch"], max_tokens=room)
    params = SamplingParams(temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"],
                            repeat_penalty=case["repeat_penalty"], seed=seed)
    state = {"case": case, "eng": eng, "contexts": contexts, "fed": fed, "sampler": Sampler(params, eng.device),
             "seeds": [seed * 1000 + i for i in range(case["batch"])]}
    if case["steps"]:
        eng.warm_up([case["batch"]], longest=case["longest"] + case["steps"])
    if case["kind"] == "decode":
        state["slots"] = [eng.alloc_slot() for _ in contexts]
        part, n = [], 0
        for s, c in zip(state["slots"], contexts):            # contexts in steps of bounded size
            if n + len(c) > 16384:
                eng.step(part)
                part, n = [], 0
            part.append(StepEntry(s, c))
            n += len(c)
        eng.step(part)
    elif sum(len(c) for c in contexts) <= 256:
        # a program that has answered before has captured the graphs of short prompts
        for _ in range(2):
            run(state)
    return state


def run(state):
    from inferllm_amd import StepEntry
    case, eng, sampler, contexts = state["case"], state["eng"], state["sampler"], state["contexts"]
    out, drawn, unread = [], [], None
    slots = state.get("slots")
    histories = [list(c) for c in contexts]
    plan = [[[t] for t in f] for f in state["fed"]]
    if slots is None:
        slots = [eng.alloc_slot() for _ in contexts]
        plan.insert(0, contexts)
    for k, tokens in enumerate(plan):
        logits = eng.step([StepEntry(s, t, [len(t) - 1]) for s, t in zip(slots, tokens)])
        if k or case["kind"] == "decode":
            for h, t in zip(histories, tokens):
                h.extend(t)
        choice = sampler.draw(logits, state["seeds"], [k] * len(slots), histories)
        if unread is not None:
            drawn.append(unread.tokens())
        unread = choice
        out.append(logits)
    drawn.append(unread.tokens())
    if case["kind"] == "decode":
        for s in slots:
            eng.cache.rewind(s, case["steps"])
    else:
        for s in slots:
            eng.free_slot(s)
    # chosen tokens are whole numbers: in bfloat16 two near logits may change places in another
    # correct implementation, so there the logits they were chosen from stand for them
    return {"logits": out, "tokens": torch.tensor(drawn)} if case["dtype"] == "float32" else {"logits": out}


# ---------------------------------------------------------------- what a pass cannot do without
def _counts(cfg, batch_rows):
    """(weights that every step reads, weights of the embedding's rows a token, multiply-adds a
    token outside attention and recurrences, [(cache values a token, score and value columns a
    pair of tokens, most keys seen, state values a sequence)] per layer, head weights) for steps
    of `batch_rows` tokens."""
    if "hidden_size" in cfg:
        E, F, L = cfg["hidden_size"], cfg["intermediate_size"], cfg["num_hidden_layers"]
        nh, nkv, hd = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        w = L * ((nh + 2 * nkv) * hd * E + nh * hd * E + 3 * E * F)
        return w, E, w, [(2 * nkv * hd, 2 * nh * hd, 1 << 30, 0)] * L, cfg["vocab_size"] * E
    E = cfg["width"]
    read = mul = 0
    per = []
    for layer in cfg["layers"]:
        m, mlp, kind = layer["mixer"], layer["mlp"], layer["type"]
        if kind == "latent_attention":
            H, dq, R = m["heads"], m["dim"] + m["rot_dim"], m["kv_rank"]
            w = E * (H * dq + R + m["rot_dim"] + H) + R * H * (m["dim"] + m["vdim"]) + H * m["vdim"] * E
            per.append((R + m["rot_dim"], H * (dq + m["vdim"]), 1 << 30, 0))
        elif kind == "mamba2":
            inner, gn = m["heads"] * m["vdim"], m["groups"] * m["state"]
            w = E * (2 * inner + 2 * gn + m["heads"]) + inner * E
            per.append((0, 0, 0, m["heads"] * m["state"] * m["vdim"]))
        elif kind in ("mlstm", "gla"):
            H, dk, dv = m["heads"], m["dim"], m["vdim"]
            w = E * (2 * H * dk + 2 * H * dv) + H * dv * E + (
                2 * E * H if kind == "mlstm" else m["rank"] * (E + H * dk))
            per.append((0, 0, 0, H * dk * dv))
        else:
            a = m["left"] if kind == "parallel" else m
            H, G, dk, dv = a["heads"], a["kv_heads"], a["dim"], a["vdim"]
            own = 0 if "kv_from" in a else G * (dk + dv)
            w = E * (H * dk + own) + H * dv * E
            w += E * H * dv if "v_mix" in a else E * H if kind == "attention" else 0
            state = 0
            if kind == "parallel":
                C, nb = m["right"]["width"], m["right"]["blocks"]
                w, state = w + 3 * E * C + 2 * C * (C // nb), C
            mask = a.get("mask") or {}
            per.append((G * (dk + dv), H * (dk + dv), mask.get("size", 1 << 30), state))
        if mlp["kind"] == "moe":
            n, top, ff, sh = mlp["router"]["experts"], mlp["router"]["top"], mlp["expert"]["ff"], mlp["shared"]["ff"]
            read += w + E * n + 3 * E * (sh + ff * n * (1.0 - (1.0 - top / n) ** batch_rows))
            mul += w + E * n + 3 * E * (sh + top * ff)
        else:
            ffw = (3 if "limit" in mlp else 2) * E * mlp["ff"]
            read, mul = read + w + ffw, mul + w + ffw
    return read, E * (3 if cfg["architecture"] == "Sabipel" else 2 if cfg["architecture"] == "Dotorax" else 1), mul, per, cfg["vocab"] * E


def work(case):
    """Each step reads every weight it needs and its sequences' cache once; prompts read the
    weights once and write their cache rows."""
    cfg, esz = MODELS[case["model"]], 2 if case["dtype"] == "bfloat16" else 4
    lens, B = _lengths(case), case["batch"]
    total_bytes = total_flops = 0.0
    if case["kind"] != "decode":
        T = sum(lens)
        read, emb, mul, per, head = _counts(cfg, T)
        total_bytes += (read + head + T * (emb + sum(p[0] for p in per))) * esz
        total_flops += 2.0 * T * mul + 2.0 * B * head
        for kv, cols, most, st in per:
            pairs = sum(n * (n + 1) / 2 if n <= most else most * (most + 1) / 2 + (n - most) * most for n in lens)
            total_flops += 2.0 * cols * pairs + 2.0 * 2 * st * T
            total_bytes += B * st * 4
        total_bytes += B * 4 * (cfg.get("vocab_size") or cfg["vocab"])
    for k in range(case["steps"]):
        read, emb, mul, per, head = _counts(cfg, B)
        total_bytes += (read + head + B * emb) * esz + B * 4 * (cfg.get("vocab_size") or cfg["vocab"])
        total_flops += 2.0 * B * (mul + head)
        for kv, cols, most, st in per:
            seen = sum(min(n + k + 1, most) for n in lens)
            total_bytes += seen * kv * esz + B * st * 4 * 2
            total_flops += 2.0 * cols * seen + 2.0 * 2 * st * B
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    """About four times what the outputs are off the same in 64 bits."""
    if case["dtype"] == "float32":
        return {"rel": 2e-5}                          # 1e-7 (tiny) to 4e-6
    # 0.005 to 0.007 (LLaMA shapes, Rabapel, Sabipel), 0.013 (Dotorax); another order of the sums
    # moves as many bfloat16 roundings
    return {"rel": 0.03 if case["model"] in ("rabapel", "sabipel", "dotorax") else 0.025}


# ---------------------------------------------------------------- the same in 64 bits, plainly
class _Weights:
    """The case's weights in 64 bits, drawn when asked for."""

    def __init__(self, case, seed, keep):
        self.seed, self.dtype, self.kept = seed, getattr(torch, case["dtype"]), {} if keep else None
        self.layers = MODELS[case["model"]].get("num_hidden_layers", 0)

    def __call__(self, name, *shape, ones=False):
        if self.kept is not None and name in self.kept:
            return self.kept[name]
        t = _weight(self.seed, name, shape, ones, self.dtype, self.layers).double()
        if self.kept is not None:
            self.kept[name] = t
        return t


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _softplus(x):
    return torch.nn.functional.softplus(x, threshold=40)


def _turn(x, base, dims, halves, scaling=None):
    """Rotate the first `dims` of the heads x [T, heads, d] by position: pairs half apart, or neighbours."""
    half = dims // 2
    i = torch.arange(half, dtype=torch.float64, device=x.device)
    f, gain = float(base) ** (-2.0 * i / dims), 1.0
    if scaling:
        at = lambda turns: dims * math.log(scaling["original"] / (2 * math.pi * turns)) / (2 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(at(scaling["fast"])), 0), min(math.ceil(at(scaling["slow"])), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f, gain = f / scaling["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(scaling["factor"]) + 1.0
    a = torch.arange(x.shape[0], dtype=torch.float64, device=x.device)[:, None] * f[None]
    c, s = (torch.cos(a) * gain)[:, None], (torch.sin(a) * gain)[:, None]
    out = x.clone()
    first, second = (slice(0, half), slice(half, dims)) if halves else (slice(0, dims, 2), slice(1, dims, 2))
    out[..., first], out[..., second] = x[..., first] * c - x[..., second] * s, x[..., second] * c + x[..., first] * s
    return out


def _attend(q, k, v, see, scale=1.0, bias=None, more=None):
    """q [T, H, dk], k and v [T, G, d], see [T, T]; `scale` a number or one a head; `bias(head)`
    added to the scores; `more` = (keys, values, seen) share the softmax."""
    T, H, _ = q.shape
    rep, out = H // k.shape[1], []
    for h in range(H):
        g = h // rep
        sc = scale[h] if torch.is_tensor(scale) else scale
        s = q[:, h] @ k[:, g].T * sc
        if bias is not None:
            s = s + bias(h)
        s, val = s.masked_fill(~see, -math.inf), v[:, g]
        if more is not None:
            s = torch.cat([s, (q[:, h] @ more[0][:, g].T * sc).masked_fill(~more[2], -math.inf)], 1)
            val = torch.cat([val, more[1][:, g]], 0)
        out.append(torch.softmax(s, 1) @ val)
    return torch.stack(out, 1)


def _causal(T, dev):
    i = torch.arange(T, device=dev)
    return i[:, None] - i[None, :]


def _exact_llama(cfg, W, seqs):
    """Hidden rows after the last norm, of all sequences one after the other; the head's matrix."""
    E, F, H, G, d = (cfg[k] for k in ("hidden_size", "intermediate_size", "num_attention_heads", "num_key_value_heads", "head_dim"))
    eps, V, lens = cfg["rms_norm_eps"], cfg["vocab_size"], [len(s) for s in seqs]
    x = W("model.embed_tokens.weight", V, E)[torch.tensor([t for s in seqs for t in s], device="cuda")]
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = _rms(x, eps) * W(p + "input_layernorm.weight", E, ones=True)
        q, k, v = ((h @ W(p + f"self_attn.{n}_proj.weight", m * d, E).T).view(-1, m, d) for n, m in (("q", H), ("k", G), ("v", G)))
        parts, at = [], 0
        for n in lens:
            s = slice(at, at + n)
            parts.append(_attend(_turn(q[s], cfg["rope_theta"], d, True), _turn(k[s], cfg["rope_theta"], d, True), v[s],
                                 _causal(n, x.device) >= 0, d ** -0.5).reshape(n, H * d))
            at += n
        x = x + torch.cat(parts) @ W(p + "self_attn.o_proj.weight", E, H * d).T
        h = _rms(x, eps) * W(p + "post_attention_layernorm.weight", E, ones=True)
        u = _silu(h @ W(p + "mlp.gate_proj.weight", F, E).T) * (h @ W(p + "mlp.up_proj.weight", F, E).T)
        x = x + u @ W(p + "mlp.down_proj.weight", E, F).T
    return _rms(x, eps) * W("model.norm.weight", E, ones=True), W("lm_head.weight", V, E)


def _exact_rabapel(cfg, W, ids):
    E, eps = cfg["width"], cfg["norm"]["eps"]
    x = W("embed", cfg["vocab"], E)[ids] * cfg["embedding"]["scale"]
    see, T = _causal(len(ids), x.device) >= 0, len(ids)
    for i, layer in enumerate(cfg["layers"]):
        m, f, p = layer["mixer"], layer["mlp"], f"l{i}.mix."
        H, dn, dr, dv, R, rot = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], m["rot"]
        h = _rms(x, eps) * W(f"l{i}.norm1", E, ones=True)
        q = (h @ W(p + "q", H * (dn + dr), E).T).view(T, H, dn + dr)
        down = h @ W(p + "dkv", R + dr, E).T
        c = _rms(down[:, :R], eps) * W(p + "dkv.norm", R, ones=True)
        kr = _turn(down[:, None, R:], rot["base"], rot["dims"], False, rot["scaling"]).expand(T, H, dr)
        k = torch.cat([(c @ W(p + "uk", H * dn, R).T).view(T, H, dn), kr], -1)
        q = torch.cat([q[..., :dn], _turn(q[..., dn:], rot["base"], rot["dims"], False, rot["scaling"])], -1)
        o = _attend(q, k, (c @ W(p + "uv", H * dv, R).T).view(T, H, dv), see, m["scale"])
        o = (o * torch.sigmoid(h @ W(p + "g", H, E).T)[..., None]).reshape(T, H * dv) @ W(p + "o", E, H * dv).T
        p = f"l{i}.mlp."
        if f["kind"] == "dense":
            y = torch.relu(h @ W(p + "up", f["ff"], E).T) ** 2 @ W(p + "down", E, f["ff"]).T
        else:
            gated = lambda r, q, n: (_silu(r @ W(q + "gate", n, E).T) * (r @ W(q + "up", n, E).T)) @ W(q + "down", E, n).T  # noqa: E731
            n = f["router"]["experts"]
            s = torch.softmax(h @ W(p + "router", n, E).T, -1)
            chosen = torch.topk(s + W(p + "correction", n), f["router"]["top"], -1).indices
            y = torch.sigmoid(h @ W(p + "shared.sg", 1, E).T) * gated(h, p + "shared.", f["shared"]["ff"])
            for e in range(n):
                rows = (chosen == e).any(1).nonzero()[:, 0]
                y[rows] += s[rows, e, None] * gated(h[rows], f"{p}e{e}.", f["expert"]["ff"])
        x = x + o + y
    return _rms(x, eps) * W("final.norm", E, ones=True), W("embed", cfg["vocab"], E)


def _conv(x, w, b=None):
    taps, y = w.shape[1], torch.zeros_like(x) if b is None else b.expand_as(x).clone()
    for j in range(taps):
        back = taps - 1 - j
        y[back:] += w[:, j] * x[:len(x) - back]
    return y


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _exact_sabipel(cfg, W, ids):
    E, eps, T = cfg["width"], cfg["norm"]["eps"], len(ids)
    big = cfg["embedding"]["bigram"]
    pair = torch.cat([torch.full_like(ids[:1], big["buckets"]), (ids[:-1] * big["mul_prev"] + ids[1:] * big["mul_cur"]) % big["buckets"]])
    x = (W("embed", cfg["vocab"], E)[ids] * cfg["embedding"]["scale"] + W("bigram", big["buckets"] + 1, E)[pair]
         + W("pos", cfg["max_positions"], E)[:T])
    first = None
    for i, layer in enumerate(cfg["layers"]):
        m, p, kind = layer["mixer"], f"l{i}.mix.", layer["type"]
        h = _rms(x, eps) * W(f"l{i}.norm1", E, ones=True)
        H, dv = m["heads"], m["vdim"]
        if kind == "mamba2":
            N, G, inner = m["state"], m["groups"], H * dv
            u = h @ W(p + "in", 2 * inner + 2 * G * N + H, E).T
            c = inner + 2 * G * N
            xbc = _silu(_conv(u[:, inner:inner + c], W(p + "conv", c, m["conv"]), W(p + "conv.b", c)))
            xs, B, C = (xbc[:, :inner].view(T, H, dv), *(xbc[:, inner + j * G * N:inner + (j + 1) * G * N].view(T, G, N)
                                                        .repeat_interleave(H // G, 1) for j in (0, 1)))
            dt = _softplus(u[:, inner + c:] + W(p + "dt_bias", H))
            keep = torch.exp(-torch.exp(W(p + "A_log", H)) * dt)
            S, ys = torch.zeros(H, N, dv, dtype=x.dtype, device=x.device), []
            Bd = B * dt[..., None]
            for t in range(T):
                S = torch.baddbmm(S * keep[t, :, None, None], Bd[t, :, :, None], xs[t, :, None])
                ys.append(torch.bmm(C[t, :, None], S)[:, 0])
            y = (torch.stack(ys) + W(p + "D", H, ones=True)[:, None] * xs).reshape(T, inner) * _silu(u[:, :inner])
            y = _rms(y.view(T, m["norm_groups"], -1), eps).reshape(T, inner)
            a = (y * W(p + "norm", inner, ones=True)) @ W(p + "o", E, inner).T
        elif kind == "mlstm":
            dk, cap = m["dim"], m["gate_cap"]
            q, k = ((h @ W(p + n, H * dk, E).T).view(T, H, dk) for n in "qk")
            q, v = q * dk ** -0.5, (h @ W(p + "v", H * dv, E).T).view(T, H, dv)
            ig, fg = (cap * torch.tanh((h @ W(p + n, H, E).T + W(p + n + ".b", H)) / cap) for n in "if")
            fg = -_softplus(-fg)
            S, n, mx, ys = torch.zeros(H, dk, dv, dtype=x.dtype, device=x.device), 0.0, torch.zeros_like(ig[0]), []
            for t in range(T):
                new = torch.maximum(fg[t] + mx, ig[t])
                keep, take = torch.exp(fg[t] + mx - new), torch.exp(ig[t] - new)
                S = torch.baddbmm(S * keep[:, None, None], (k[t] * take[:, None])[:, :, None], v[t][:, None])
                n, mx = n * keep[:, None] + take[:, None] * k[t], new
                ys.append(torch.bmm(q[t][:, None], S)[:, 0]
                          / (torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-new)) + 1e-6)[:, None])
            y = _rms(torch.stack(ys), eps).reshape(T, H * dv) * W(p + "norm", H * dv, ones=True)
            a = (y * torch.sigmoid(h @ W(p + "g", H * dv, E).T)) @ W(p + "o", E, H * dv).T
        else:
            G, dk, size = m["kv_heads"], m["dim"], m["mask"]["size"]
            q = (_rms(h @ W(p + "q", H * dk, E).T, eps) * W(p + "q.norm", H * dk, ones=True)).view(T, H, dk)
            k = (_rms(h @ W(p + "k", G * dk, E).T, eps) * W(p + "k.norm", G * dk, ones=True)).view(T, G, dk)
            v = h @ W(p + "v", G * dv, E).T
            if first is None:
                first = v
            else:
                lam = W(p + "vmix")
                v = (1 - lam) * v + lam * first
            dist, pos = _causal(T, x.device), torch.arange(T, device=x.device) // size
            o = _attend(q, k, v.view(T, G, dv), (dist >= 0) & (pos[:, None] == pos[None]), m["scale"],
                        bias=lambda hh: -2.0 ** (-8.0 * (hh + 1) / H) * dist)
            a = (o.reshape(T, H * dv) * torch.sigmoid(h @ W(p + "g", H * dv, E).T)) @ W(p + "o", E, H * dv).T
        ff = layer["mlp"]["ff"]
        h = _rms(x, eps) * W(f"l{i}.norm2", E, ones=True)
        x = x + a + _gelu(h @ W(f"l{i}.mlp.up", ff, E).T) @ W(f"l{i}.mlp.down", E, ff).T
    return _rms(x, eps) * W("final.norm", E, ones=True), W("embed", cfg["vocab"], E)


def _exact_dotorax(cfg, W, ids):
    E, eps, T, mult = cfg["width"], cfg["norm"]["eps"], len(ids), cfg["residual_mult"]
    norm = lambda r, name: _rms(r, eps) * (1 + W(name, E))  # noqa: E731
    x = W("embed", cfg["vocab"], E)[ids] + W("pos", cfg["max_positions"], E)[:T]
    dist, kept = _causal(T, x.device), None

    def heads(h, p, a, n, d):
        return (h @ W(p, n * d, E).T).view(T, n, d)

    for i, layer in enumerate(cfg["layers"]):
        m, p, kind = layer["mixer"], f"l{i}.mix.", layer["type"]
        h = norm(x, f"l{i}.norm1")
        h = h + _conv(h, W(f"l{i}.canon1", E, 3))
        if kind == "gla":
            H, dk, dv = m["heads"], m["dim"], m["vdim"]
            q, k, v = heads(h, p + "q", m, H, dk) * dk ** -0.5, heads(h, p + "k", m, H, dk), heads(h, p + "v", m, H, dv)
            z = (h @ W(p + "a1", m["rank"], E).T) @ W(p + "a2", H * dk, m["rank"]).T + W(p + "a2.b", H * dk)
            al = torch.exp(-_softplus(-z) / m["tau"]).view(T, H, dk)
            S, ys = torch.zeros(H, dk, dv, dtype=x.dtype, device=x.device), []
            for t in range(T):
                S = torch.baddbmm(S * al[t][..., None], k[t][..., None], v[t][:, None])
                ys.append(torch.bmm(q[t][:, None], S)[:, 0])
            y = _rms(torch.stack(ys), eps) * W(p + "norm", dv, ones=True)
            a = (y.reshape(T, H * dv) * _silu(h @ W(p + "g", H * dv, E).T)) @ W(p + "o", E, H * dv).T
        else:
            l, c = (m["left"], p + "left.") if kind == "parallel" else (m, p)
            H, G, dk, dv, rot = l["heads"], l["kv_heads"], l["dim"], l["vdim"], l["rot"]
            turn = lambda r: _turn(r, rot["base"], rot["dims"], kind == "attention")  # noqa: E731
            q = turn(heads(h, c + "q", l, H, dk))
            k, v = kept if "kv_from" in l else (turn(heads(h, c + "k", l, G, dk)), heads(h, c + "v", l, G, dv))
            if kind == "attention":
                kept = kept or (k, v)
                o = _attend(q, k, v, dist >= 0, l["scale"]) * torch.sigmoid(h @ W(p + "g", H, E).T)[..., None]
                a = o.reshape(T, H * dv) @ W(p + "o", E, H * dv).T
            else:
                q, k, size, P = _rms(q, eps), _rms(k, eps), l["mask"]["size"], l["mask"]["pool"]
                nb = T // P
                pool = lambda r: r[:nb * P].view(nb, P, *r.shape[1:]).mean(1)  # noqa: E731
                last = torch.arange(nb, device=x.device) * P + P - 1
                seen = last[None] <= torch.arange(T, device=x.device)[:, None] - size
                o = _attend(q, k, v, (dist >= 0) & (dist < size), l["scale"] * W(c + "temp", H, ones=True), more=(pool(k), pool(v), seen))
                a = l_out = o.reshape(T, H * dv) @ W(c + "o", E, H * dv).T
                r, c = m["right"], p + "right."
                C, n = r["width"], r["blocks"]
                y = _gelu(h @ W(c + "y", C, E).T + W(c + "y.b", C))
                u = _conv(h @ W(c + "x", C, E).T + W(c + "x.b", C), W(c + "conv", C, r["conv"]), W(c + "conv.b", C))
                gate = lambda g: torch.sigmoid(torch.bmm(u.view(T, n, -1).transpose(0, 1).contiguous(),  # noqa: E731
                                                         W(c + g, n, C // n, C // n).transpose(1, 2).contiguous()).transpose(0, 1)
                                               + W(c + g + ".b", n, C // n)).reshape(T, C)
                al = torch.exp(-8.0 * gate("ra") * _softplus(W(c + "lam", C)))
                add = torch.sqrt(1 - al * al) * gate("ri") * u
                S, ys = torch.zeros_like(al[0]), []
                for t in range(T):
                    S = al[t] * S + add[t]
                    ys.append(S)
                a = m["left_scale"] * l_out + m["right_scale"] * ((torch.stack(ys) * y) @ W(c + "o", E, C).T)
        x = x + mult * norm(a, f"l{i}.norm1b")
        ff, lim, p = layer["mlp"]["ff"], layer["mlp"]["limit"], f"l{i}.mlp."
        h = norm(x, f"l{i}.norm2")
        h = h + _conv(h, W(f"l{i}.canon2", E, 3))
        g, u = (h @ W(p + "gate", ff, E).T).clamp(max=lim), (h @ W(p + "up", ff, E).T).clamp(-lim, lim)
        x = x + mult * norm((g * torch.sigmoid(1.702 * g) * (u + 1)) @ W(p + "down", E, ff).T, f"l{i}.norm2b")
    return norm(x, "final.norm"), W("head", cfg["vocab"], E)


@torch.no_grad()
def exact(case, seed):
    cfg = MODELS[case["model"]]
    contexts, fed = _tokens(case, seed)
    seqs = [c + [f[i] for f in fed] for i, c in enumerate(contexts)]
    first = 0 if case["kind"] == "decode" else -1      # the step of the first logits, behind the context
    steps = range(first, case["steps"])
    if "hidden_size" in cfg:
        if sum(len(s) for s in seqs) > 20000:
            return None                               # over about 20 seconds in 64 bits
        rows, head = _exact_llama(cfg, _Weights(case, seed, False), seqs)
        at, wanted = 0, []
        for c, s in zip(contexts, seqs):
            wanted.append([at + len(c) + k for k in steps])
            at += len(s)
        logits = [rows[[w[j] for w in wanted]] @ head.T for j in range(len(steps))]
    else:
        W = _Weights(case, seed, True)
        plain = {"rabapel": _exact_rabapel, "sabipel": _exact_sabipel, "dotorax": _exact_dotorax}[case["model"]]
        per = []
        for c, s in zip(contexts, seqs):
            rows, head = plain(cfg, W, torch.tensor(s, device="cuda"))
            per.append(rows[[len(c) + k for k in steps]] @ head.T)
        logits = [torch.stack([p[j] for p in per]) for j in range(len(steps))]
    return {"logits": logits, "tokens": None} if case["dtype"] == "float32" else {"logits": logits}
