"""Cases for timing the engine: what a program that uses it has it do, at the sizes it is used at.

A pass is a short stretch of serving, driven through ``Engine.step`` with given tokens as the replay tool does
(``torchllms_amd/engine/replay.py``), so that two implementations see the same inputs at every step whatever their
rounding: some requests are in the cache already (``held`` tokens each), some arrive (``arrive``, with prompts of
``prompt`` tokens cut into portions under ``budget`` tokens a step, beside the running requests' tokens), and then all
decode together for ``steps`` steps.  ``ragged`` lengths are spread evenly from an eighth of the stated length up to
it.  ``sample`` adds the sampler behind every step: tokens drawn at that temperature (0: greedy) and read by the
host, as a program that streams them does.

Results are the logits of every step (and the drawn tokens).  ``exact`` computes the same logits in 64 bits from
the checkpoint tensors with plain torch; it shares no code with the engine.
"""

from __future__ import annotations

import hashlib
import math
import random
from typing import Dict, List

import torch

VOCAB = 128256  # of the Llama 3 shapes

# layer sizes: Llama-3.2-1B and Llama-3.1-8B, and a tiny configuration for the smallest calls
SHAPES = {
    "8b": dict(width=4096, heads=32, kv_heads=8, dim=128, ff=14336, vocab=VOCAB, layers=32, tied=False, eps=1e-5, factor=8.0, original=8192),
    "1b": dict(width=2048, heads=32, kv_heads=8, dim=64, ff=8192, vocab=VOCAB, layers=16, tied=True, eps=1e-5, factor=32.0, original=8192),
    "tiny": dict(width=256, heads=8, kv_heads=1, dim=32, ff=688, vocab=512, layers=3, tied=False, eps=1e-6, factor=8.0, original=64),
}
ROPE_BASE = 500000.0


def _case(name, family, shape, layers, dtype="bfloat16", held=0, running=0, arrive=0, prompt=0, budget=8192, steps=0, ragged=False, sample=-1.0):
    case = dict(name=name, family=family, shape=shape, layers=layers, dtype=dtype, held=held, running=running, arrive=arrive,
                prompt=prompt, budget=budget, steps=steps, ragged=ragged, sample=sample)
    if name is None:
        del case["name"]
    return case


def listed() -> List[dict]:
    return [
        # the smallest calls: four short prompts in 32-bit through a tiny model, in small portions, then decode; all launches and host work
        _case("tiny_f32_generate", "llama", "tiny", 3, dtype="float32", arrive=4, prompt=100, budget=48, steps=12, ragged=True, sample=0.7),
        # one user at a chat prompt of 2,000 tokens: a token at a time, bound by reading the weights and by launches
        _case("llama1b_decode_1", "llama", "1b", 16, held=2001, running=1, steps=16),
        # a small server at long contexts: the headline's batch 8 at context 8,192
        _case("llama8b_decode_8_long", "llama", "8b", 32, held=8152, running=8, steps=8),
        # a busy server: 64 requests of very different lengths, every token drawn and streamed
        _case("llama1b_serve_64", "llama", "1b", 16, held=3000, running=64, steps=6, ragged=True, sample=0.7),
        # a busy server with the larger model
        _case("llama8b_decode_64", "llama", "8b", 32, held=1000, running=64, steps=4, ragged=True),
        # a long prompt to its first token
        _case("llama8b_prefill_2048", "llama", "8b", 32, arrive=1, prompt=2048),
        # continuous batching: odd prompts come in by portions beside 13 requests that go on decoding
        _case("llama8b_mixed", "llama", "8b", 16, held=900, running=13, arrive=3, prompt=1777, budget=1024, steps=3, ragged=True),
        # the 32-bit path: a prompt and greedy tokens behind it
        _case("llama1b_f32", "llama", "1b", 16, dtype="float32", arrive=2, prompt=500, steps=4, ragged=True, sample=0.0),
        # selective scan, delta rule and chunked attention: one long prompt, then its answer
        _case("taluvik_8b_prompt", "taluvik", "8b", 8, arrive=1, prompt=2048, steps=8),
        # matrix memory, delta rule by channel, routed experts: eight requests of different lengths
        _case("kepevik_8b_batch", "kepevik", "8b", 8, arrive=8, prompt=400, steps=12, ragged=True),
        # windowed attention beside retention, looped layers, routed experts: many short requests
        _case("rifizen_1b_short", "rifizen", "1b", 8, arrive=24, prompt=90, steps=12, ragged=True),
        # state-space layers, attention through a latent, routed experts: a long prompt in portions
        _case("mesolix_8b_long", "mesolix", "8b", 8, arrive=1, prompt=3999, budget=2048, steps=8),
    ]


def _between(rng: random.Random, low: float, high: float) -> int:
    """A whole number between the two, spread over their logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random) -> dict:
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["tiny", "decode", "decode", "serve", "prefill", "mixed", "f32", "taluvik", "kepevik", "rifizen", "mesolix"])
    if kind == "tiny":
        return _case(None, "llama", "tiny", 3, dtype="float32", arrive=_between(rng, 1, 8), prompt=_between(rng, 5, 200), budget=rng.randint(16, 96),
                     steps=rng.randint(4, 16), ragged=rng.random() < 0.5, sample=rng.choice([0.0, 0.7]))
    if kind in ("decode", "serve"):
        shape = rng.choice(["1b", "8b"])
        running = _between(rng, 1, 64)
        held = _between(rng, 100, min(8000, 64000 // running))
        sample = rng.choice([0.0, 0.7]) if kind == "serve" else -1.0
        return _case(None, "llama", shape, 16, held=held, running=running, steps=rng.randint(4, 8), ragged=rng.random() < 0.5, sample=sample)
    if kind == "prefill":
        return _case(None, "llama", rng.choice(["1b", "8b"]), 16, arrive=_between(rng, 1, 4), prompt=_between(rng, 30, 1024))
    if kind == "mixed":
        return _case(None, "llama", rng.choice(["1b", "8b"]), 16, held=_between(rng, 100, 2000), running=_between(rng, 2, 24), arrive=rng.randint(1, 3),
                     prompt=_between(rng, 50, 1500), budget=rng.randint(256, 1500), steps=rng.randint(2, 4), ragged=True)
    if kind == "f32":
        return _case(None, "llama", "1b", 16, dtype="float32", arrive=rng.randint(1, 4), prompt=_between(rng, 8, 400), steps=rng.randint(2, 4),
                     ragged=True, sample=rng.choice([0.0, 0.7]))
    arrive = _between(rng, 1, 24)
    return _case(None, kind, rng.choice(["1b", "8b"]), 8, arrive=arrive, prompt=_between(rng, 20, 3000 // arrive), budget=rng.choice([1024, 2048, 8192]),
                 steps=rng.randint(4, 10), ragged=rng.random() < 0.5)


# ----------------------------------------------------------------------------- model descriptions
def config_of(case: dict) -> dict:
    """What config.json of the case's model holds."""
    s = SHAPES[case["shape"]]
    D, H, G, d, ff, n = s["width"], s["heads"], s["kv_heads"], s["dim"], s["ff"], case["layers"]
    if case["family"] == "llama":
        return dict(architectures=["LlamaForCausalLM"], hidden_size=D, num_hidden_layers=n, num_attention_heads=H, num_key_value_heads=G, head_dim=d,
                    intermediate_size=ff, vocab_size=s["vocab"], rms_norm_eps=s["eps"], rope_theta=ROPE_BASE, max_position_embeddings=131072,
                    tie_word_embeddings=s["tied"], rope_scaling=dict(rope_type="llama3", factor=s["factor"], low_freq_factor=1.0,
                                                                     high_freq_factor=4.0, original_max_position_embeddings=s["original"]))
    moe = {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 8, "top": 2}}
    if case["family"] == "taluvik":
        mixers = {
            "attention": {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "scale": d ** -0.5, "softcap": 30.0, "mask": {"size": 8192},
                          "rot": {"dims": d, "base": ROPE_BASE, "scaling": {"factor": s["factor"], "low": 1.0, "high": 4.0, "original": s["original"]}}},
            "delta": {"heads": H, "kv_heads": H // 2, "dim": d, "vdim": d, "conv": 4},
            "mamba1": {"inner": 2 * D, "state": 16, "dt_rank": D // 16, "conv": 4},
        }
        turn = ["mamba1", "attention", "delta", "mamba1"]
        return {"architecture": "Taluvik", "vocab": s["vocab"], "width": D, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-5}, "residual_mult": 1.0,
                "layers": [{"type": turn[i % 4], "mixer": mixers[turn[i % 4]], "mlp": {"kind": "dense", "ff": ff}} for i in range(n)]}
    if case["family"] == "kepevik":
        memory = {"heads": H, "dim": d, "vdim": d, "gate_cap": 15.0}
        pair = {"left": {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "scale": d ** -0.5, "rot": {"dims": d // 2, "base": ROPE_BASE}},
                "right": {"heads": H, "kv_heads": H // 2, "dim": d, "vdim": d, "conv": 4, "decay_rank": 64, "gate_rank": 64},
                "left_scale": 0.6, "right_scale": 0.5}
        moe = {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 8, "top": 2, "identity": 1}, "shared": {"ff": ff // 4}}
        return {"architecture": "Kepevik", "vocab": s["vocab"], "width": D, "embedding": {"scale": 50.0}, "norm": {"eps": 1e-6},
                "layers": [{"type": "mlstm" if i % 2 == 0 else "parallel", "mixer": memory if i % 2 == 0 else pair,
                            "mlp": {"kind": "dense", "ff": ff} if i == 0 else moe} for i in range(n)]}
    if case["family"] == "rifizen":
        h2 = H // 2
        pair = {"left": {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "scale": d ** -0.5, "softcap": 30.0, "mask": {"size": 4096}},
                "right": {"heads": h2, "dim": d, "vdim": d, "decay": [1.0 - 2.0 ** (-5.0 - 7.0 * h / h2) for h in range(h2)],
                          "rot": {"dims": d, "base": ROPE_BASE}}}
        return {"architecture": "Rifizen", "vocab": s["vocab"], "width": D, "norm": {"eps": 1e-6},
                "layers": [{"type": "parallel", "mixer": pair, "mlp": {"kind": "dense", "ff": ff} if i == 0 else moe} for i in range(n - 2)],
                "loop": {"start": (n - 2) // 2, "stop": (n - 2) // 2 + 2, "times": 2}}
    assert case["family"] == "mesolix"
    mixers = {
        "mamba2": {"heads": 2 * D // 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8},
        "attention": {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "scale": d ** -0.5, "bias_max": 1024, "mask": {"size": 4096}},
        "latent_attention": {"heads": H, "dim": d, "vdim": d, "q_rank": 3 * D // 8, "kv_rank": 256, "scale": d ** -0.5},
    }
    turn = ["mamba2", "attention", "mamba2", "latent_attention"]
    moe = dict(moe, shared={"ff": ff // 4})
    layers = [{"type": turn[i % 4], "mixer": mixers[turn[i % 4]], "mlp": {"kind": "dense", "ff": ff, "limit": 7.0} if i == 0 else moe} for i in range(n)]
    layers[n // 4 * 4 - 1]["weights_of"] = 3
    return {"architecture": "Mesolix", "vocab": s["vocab"], "width": D, "max_positions": 8192, "norm": {"eps": 1e-6}, "layers": layers}


def shapes_of(case: dict) -> Dict[str, tuple]:
    """Checkpoint name -> shape of every tensor of the case's model."""
    c, family = config_of(case), case["family"]
    if family == "llama":
        D, H, G, d, F, V = (c[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim", "intermediate_size", "vocab_size"))
        out = {"model.embed_tokens.weight": (V, D), "model.norm.weight": (D,)}
        if not c["tie_word_embeddings"]:
            out["lm_head.weight"] = (V, D)
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            out.update({p + "self_attn.q_proj.weight": (H * d, D), p + "self_attn.k_proj.weight": (G * d, D), p + "self_attn.v_proj.weight": (G * d, D),
                        p + "self_attn.o_proj.weight": (D, H * d), p + "mlp.gate_proj.weight": (F, D), p + "mlp.up_proj.weight": (F, D),
                        p + "mlp.down_proj.weight": (D, F), p + "input_layernorm.weight": (D,), p + "post_attention_layernorm.weight": (D,)})
        return out
    D, V = c["width"], c["vocab"]
    out = {"embed": (V, D), "final.norm": (D,)}
    if family != "kepevik":
        out["head"] = (V, D)
    if family == "taluvik":
        out["final.norm.b"] = (D,)
    if family == "mesolix":
        out["pos"] = (c["max_positions"], D)
    if family == "rifizen":
        out["loop.step"] = (c["loop"]["times"], D)

    def gated(p, F):
        out.update({p + "gate": (F, D), p + "up": (F, D), p + "down": (D, F)})

    def attention(p, m, value=True):
        out.update({p + "q": (m["heads"] * m["dim"], D), p + "k": (m["kv_heads"] * m["dim"], D), p + "o": (D, m["heads"] * m["vdim"])})
        if value:
            out[p + "v"] = (m["kv_heads"] * m["vdim"], D)

    def delta(p, m):
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        for t, n in (("q", G * d), ("k", G * d), ("v", H * dv)):
            out.update({p + t: (n, D), p + t + ".conv": (n, m["conv"])})
        out.update({p + "b": (H, D), p + "A_log": (H,), p + "norm": (dv,), p + "o": (D, H * dv)})

    for i, layer in enumerate(c["layers"]):
        if layer.get("weights_of") is not None:
            continue
        L, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
        p = L + "mix."
        if family == "taluvik":
            out.update({L + "norm1": (D,), L + "norm1.b": (D,)})
            gated(L + "mlp.", mlp["ff"])
            if layer["type"] == "attention":
                attention(p, m)
                out[p + "sink"] = (m["heads"],)
            elif layer["type"] == "delta":
                delta(p, m)
                out.update({p + "a": (m["heads"], D), p + "dt_bias": (m["heads"],), p + "g": (m["heads"] * m["vdim"], D)})
            else:
                I, N, R = m["inner"], m["state"], m["dt_rank"]
                out.update({p + "in": (2 * I, D), p + "conv": (I, m["conv"]), p + "conv.b": (I,), p + "x": (R + 2 * N, I), p + "dt": (I, R),
                            p + "dt.b": (I,), p + "A_log": (I, N), p + "D": (I,), p + "o": (D, I)})
            continue
        if family in ("kepevik", "rifizen"):
            out.update({L + n: (D,) for n in ("norm1", "norm1b", "norm2", "norm2b")})
        if family == "kepevik":
            out.update({L + "ls1": (D,), L + "ls2": (D,)})
            if layer["type"] == "mlstm":
                H, d, dv = m["heads"], m["dim"], m["vdim"]
                out.update({p + "q": (H * d, D), p + "k": (H * d, D), p + "v": (H * dv, D), p + "g": (H * dv, D), p + "o": (D, H * dv),
                            p + "i": (H, D), p + "i.b": (H,), p + "f": (H, D), p + "f.b": (H,), p + "norm": (H * dv,)})
            else:
                r = m["right"]
                attention(p + "left.", m["left"], value=False)
                delta(p + "right.", r)
                out.update({p + "right.a1": (r["decay_rank"], D), p + "right.a2": (r["heads"] * r["dim"], r["decay_rank"]),
                            p + "right.dt_bias": (r["heads"] * r["dim"],), p + "right.g1": (r["gate_rank"], D),
                            p + "right.g2": (r["heads"] * r["vdim"], r["gate_rank"])})
            if mlp["kind"] == "dense":
                F = mlp["ff"]
                out.update({L + "mlp.up": (F, D), L + "mlp.up.b": (F,), L + "mlp.down": (D, F), L + "mlp.down.b": (D,)})
        if family == "rifizen":
            r = m["right"]
            attention(p + "left.", m["left"])
            out.update({p + "right." + t: (r["heads"] * r["dim"], D) for t in "qkvg"})
            out.update({p + "right.o": (D, r["heads"] * r["vdim"]), p + "left.out": (D,), p + "right.out": (D,)})
            if mlp["kind"] == "dense":
                out.update({L + "mlp.up": (mlp["ff"], D), L + "mlp.down": (D, mlp["ff"])})
        if family == "mesolix":
            out.update({L + "norm1": (D,), L + "norm2": (D,)})
            if layer["type"] == "mamba2":
                H, inner, conv = m["heads"], m["heads"] * m["vdim"], m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"]
                out.update({p + "in": (inner + conv + H, D), p + "conv": (conv, m["conv"]), p + "conv.b": (conv,), p + "dt_bias": (H,),
                            p + "A_log": (H,), p + "D": (H,), p + "norm": (inner,), p + "o": (D, inner)})
            elif layer["type"] == "attention":
                attention(p, m)
                out.update({p + "g": (m["heads"] * m["vdim"], D), p + "rel": (32, m["heads"])})
            else:
                H, d, dv, R, Q = m["heads"], m["dim"], m["vdim"], m["kv_rank"], m["q_rank"]
                out.update({p + "dq": (Q, D), p + "dq.norm": (Q,), p + "uq": (H * d, Q), p + "dkv": (R, D), p + "dkv.norm": (R,), p + "uk": (H * d, R),
                            p + "uv": (H * dv, R), p + "sink": (H,), p + "g": (H * dv, D), p + "o": (D, H * dv)})
            if mlp["kind"] == "dense":
                gated(L + "mlp.", mlp["ff"])
        if mlp["kind"] == "moe":
            experts = mlp["router"]["experts"] + mlp["router"].get("identity", 0)
            out[L + "mlp.router"] = (experts, D)
            for e in range(mlp["router"]["experts"]):
                gated(f"{L}mlp.e{e}.", mlp["expert"]["ff"])
            if mlp.get("shared"):
                gated(L + "mlp.shared.", mlp["shared"]["ff"])
            if family == "kepevik":
                out.update({L + "mlp.correction": (experts,), L + "mlp.shared.sg": (1, D)})
            if family == "rifizen":
                out[L + "mlp.router.b"] = (experts,)
    return out


def tensor_of(name: str, shape: tuple, seed: int, family: str, dtype: torch.dtype) -> torch.Tensor:
    """A checkpoint tensor drawn from (seed, name) in 32-bit and cast: matrices N(0, 0.02); embeddings of the order of one
    and branches whose last matrix (or last norm) is smaller, so that a layer adds to the stream what a trained layer does and
    rounding is not blown up from layer to layer; the parameters of recurrences in the ranges that such layers are
    initialised with and trained around (steps of 0.001 to 0.1 and rates of 1 to 16 and so memories of a few to a thousand
    tokens, forget gates well open); routers that are sure of nearly all their choices, so
    that rounding seldom sends a token to another expert."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int.from_bytes(hashlib.sha256(f"{seed}/{name}".encode()).digest()[:7], "little"))
    t = torch.empty(shape, dtype=torch.float32, device="cuda")
    leaf = name.rsplit("mix.", 1)[-1].rsplit("mlp.", 1)[-1].split("left.")[-1].split("right.")[-1]
    if leaf in ("dt_bias", "dt.b"):
        t.uniform_(math.log(0.001), math.log(0.1), generator=gen)
        t = t.exp().expm1().log()  # softplus of it is the step
    elif leaf == "A_log":
        t.uniform_(1.0, 16.0, generator=gen)
        t = t.log()
    elif leaf == "f.b":
        t.uniform_(3.0, 6.0, generator=gen)
    elif leaf.endswith("conv"):
        t.normal_(0.0, 0.5, generator=gen)
    elif leaf in ("a2", "g2", "dt"):
        t.normal_(0.0, 0.1, generator=gen)
    elif leaf == "router":
        t.normal_(0.0, (4.0 if family == "mesolix" else 40.0) * shape[1] ** -0.5, generator=gen)
    elif leaf in ("sink", "rel", "router.b"):
        t.normal_(0.0, 0.5, generator=gen)
    elif name.endswith((".ls1", ".ls2")):
        t.uniform_(0.1, 0.3, generator=gen)
    elif family == "rifizen" and name.endswith(("norm1b", "norm2b")):
        t.uniform_(0.1, 0.3, generator=gen)
    elif leaf.endswith(".b") or leaf == "correction" or name.endswith("norm1.b"):
        t.normal_(0.0, 0.02, generator=gen)
    elif len(shape) == 1:  # norms, and the direct path of a scan: around one, or around zero where one is added
        t.normal_(0.0, 0.1, generator=gen)
        around_zero = family in ("kepevik", "mesolix") and "mix." not in name
        t = t if around_zero else t + 1.0
    elif name.endswith((".o", ".down", "o_proj.weight", "down_proj.weight")):
        t.normal_(0.0, 0.004, generator=gen)
    elif name == "embed" and family != "kepevik" or name == "model.embed_tokens.weight" and shape[1] > 2048:
        t.normal_(0.0, 1.0, generator=gen)
    else:  # an embedding that is the head's matrix too is small, and scaled where the design scales it
        t.normal_(0.0, 0.02, generator=gen)
    return t.to(dtype)


# ----------------------------------------------------------------------------- a pass
def _lengths(count: int, longest: int, ragged: bool) -> List[int]:
    if not ragged or count < 2:
        return [longest] * count
    low = max(longest // 8, 1)
    return [low + (longest - low) * i // (count - 1) for i in range(count)]


def plan(case: dict, seed: int) -> dict:
    """The requests' tokens and the pass's steps: ``held`` (request -> tokens in the cache before the pass), ``arrive``
    (requests that come), ``steps`` (lists of (request, first token, tokens, wanted places))."""
    rng = random.Random(seed * 1000003 + 17)
    vocab = SHAPES[case["shape"]]["vocab"]
    held = {f"h{i}": n for i, n in enumerate(_lengths(case["running"], case["held"], case["ragged"]))}
    prompts = {f"a{i}": n for i, n in enumerate(_lengths(case["arrive"], case["prompt"], case["ragged"]))}
    done = dict(held)
    done.update({r: 0 for r in prompts})
    steps = []
    while any(done[r] < n for r, n in prompts.items()):
        going = [r for r in done if r in held or done[r] >= prompts[r]]
        step = [(r, done[r], 1, [0]) for r in going]
        room = case["budget"] - len(step)
        for r, n in prompts.items():
            take = min(n - done[r], room)
            if take > 0:
                step.append((r, done[r], take, [take - 1] if done[r] + take == n else []))
                room -= take
        steps.append(step)
        for r, _, n, _ in step:
            done[r] += n
    for _ in range(case["steps"]):
        steps.append([(r, done[r], 1, [0]) for r in done])
        for r in done:
            done[r] += 1
    tokens = {r: [rng.randrange(vocab) for _ in range(n)] for r, n in done.items()}
    return {"held": held, "arrive": list(prompts), "steps": steps, "tokens": tokens}


def prepare(case: dict, seed: int) -> dict:
    from torchllms_amd.config import get_architecture
    from torchllms_amd.engine import Engine, StepEntry
    from torchllms_amd.sampling import Sampler, SamplingParams

    p = plan(case, seed)
    raw = config_of(case)
    arch = get_architecture(raw.get("architecture") or raw["architectures"][0])
    config = arch.config_from_dict(raw)
    rules = arch.weight_rules(config)
    dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    tensors = {}
    for name, shape in shapes_of(case).items():
        rule, own = next((r, m[0]) for r, m in ((r, r.match_external(name)) for r in rules) if m is not None)
        t = tensor_of(name, shape, seed, case["family"], dtype)
        tensors[own] = (rule.load(t) if rule.load is not None else t).contiguous()
    longest = max(len(t) for t in p["tokens"].values())
    pages = sum(-(-len(t) // 16) + 1 for t in p["tokens"].values())
    engine = Engine(arch, config, tensors, dtype, page_size=16, num_pages=pages, max_seqs=len(p["tokens"]), max_model_len=longest)
    tensors.clear()
    torch.cuda.empty_cache()
    entry = lambda r, first, n, want: StepEntry(r, p["tokens"][r][first : first + n], list(want))  # noqa: E731
    for r in p["held"]:
        engine.admit(r)
    done, batch, size = {r: 0 for r in p["held"]}, [], 0
    for r, n in p["held"].items():  # the requests that run already, prompts in portions of at most 8,192 tokens a step
        batch.append(entry(r, 0, n, []))
        size += n
        if size + n > 8192 or r == list(p["held"])[-1]:
            engine.step(batch)
            batch, size = [], 0
    steps, params, counters = [], [], []
    for i, step in enumerate(p["steps"]):
        steps.append([entry(*e) for e in step])
        rows = [e[0] for e in step for _ in e[3]]
        params.append([SamplingParams(temperature=max(case["sample"], 0.0), seed=seed + int(r[1:])) for r in rows])
        counters.append([i] * len(rows))
    torch.cuda.synchronize()
    return {"engine": engine, "held": p["held"], "arrive": p["arrive"], "steps": steps, "params": params, "counters": counters,
            "sampler": Sampler() if case["sample"] >= 0 else None}


def run(state: dict):
    engine, sampler = state["engine"], state["sampler"]
    for r, n in state["held"].items():
        if engine.num_tokens(r) != n:
            engine.cache.truncate(r, n)  # back to where the pass begins
    for r in state["arrive"]:
        engine.admit(r)
    logits, tokens = [], []
    for entries, params, counters in zip(state["steps"], state["params"], state["counters"]):
        out = engine.step(entries)
        if not params:
            continue
        logits.append(out)
        if sampler is not None:
            tokens.append(sampler(out, params, counters))
    for r in state["arrive"]:
        engine.free(r)
    result = {"logits": logits}
    if sampler is not None:
        result["tokens"] = torch.tensor([t for row in tokens for t in row], dtype=torch.int64)
    return result


# ----------------------------------------------------------------------------- what a pass cannot do without
def _mixers(case: dict):
    """Per layer run: (heads, key channels, value channels, cached channels a token, window) of an attention, or the
    elements of a recurrent state."""
    s, n = SHAPES[case["shape"]], case["layers"]
    D, H, G, d = s["width"], s["heads"], s["kv_heads"], s["dim"]
    grouped = lambda window: (H, d, d, 2 * G * d, window)  # noqa: E731
    if case["family"] == "llama":
        return [[grouped(1 << 30)]] * n
    kinds = {"taluvik": [[2 * D * 16], [grouped(8192)], [H * d * d], [2 * D * 16]],
             "kepevik": [[H * d * d], [grouped(1 << 30), H * d * d]],
             "rifizen": [[grouped(4096), H // 2 * d * d]],
             "mesolix": [[2 * D * 128], [grouped(4096)], [2 * D * 128], [(H, 256, 256, 256, 1 << 30)]]}[case["family"]]
    return [kinds[i % len(kinds)] for i in range(n)]


def work(case: dict) -> dict:
    """Every step reads the weights that its tokens use and the keys, values and states that they see, and writes its logits
    and cache rows; a token multiplies every weight it uses once."""
    size = 4 if case["dtype"] == "float32" else 2
    c, shapes, steps = config_of(case), shapes_of(case), plan(case, 0)["steps"]
    vocab = SHAPES[case["shape"]]["vocab"]
    head = vocab * SHAPES[case["shape"]]["width"]
    dense = expert = 0
    for name, shape in shapes.items():
        if name in ("embed", "pos", "head", "model.embed_tokens.weight", "lm_head.weight"):
            continue
        if ".mlp.e" in name:
            expert += math.prod(shape)
        else:
            dense += math.prod(shape)
    if case["family"] == "rifizen":  # two of the layers run twice
        per = (dense - SHAPES[case["shape"]]["width"] * SHAPES[case["shape"]]["ff"] * 2) / (case["layers"] - 2)
        dense, expert = dense + 2 * per, expert * (case["layers"] - 1) / (case["layers"] - 3)
    if case["family"] == "mesolix":  # the last layer uses another's mixer and feed-forward
        dense, expert = dense * case["layers"] / (case["layers"] - 1), expert * (case["layers"] - 1) / (case["layers"] - 2)
    routed = next((layer["mlp"]["router"] for layer in c.get("layers", []) if layer["mlp"]["kind"] == "moe"), {"experts": 1, "top": 0})
    total_bytes = total_flops = 0.0
    for step in steps:
        tokens, wanted = sum(n for _, _, n, _ in step), sum(len(w) for _, _, _, w in step)
        used = min(tokens * routed["top"], routed["experts"]) / routed["experts"]
        total_bytes += size * (dense + expert * used + (head if wanted else 0)) + 4 * wanted * vocab
        total_flops += 2 * tokens * (dense + expert * routed["top"] / routed["experts"]) + 2 * wanted * head
        for mixers in _mixers(case):
            for m in mixers:
                if not isinstance(m, tuple):
                    total_bytes += 4 * m * len(step) * 2
                    total_flops += 6 * m * tokens
                    continue
                heads, dk, dv, cached, window = m
                for _, first, n, _ in step:
                    total_bytes += size * cached * (min(first + n, window + n) + n)
                    pairs = sum(min(window, p + 1) for p in (first, first + n - 1)) * n / 2
                    total_flops += 2 * heads * (dk + dv) * pairs
    return {"bytes": float(total_bytes), "flops": float(total_flops)}


def tolerance(case: dict):
    """Two to four times the distance from ``exact`` that was measured (32-bit: 2e-7 to 6e-6; bfloat16: 0.006 to 0.03), and the
    share of drawn tokens that nearly tie.  Behind routed experts whose sum is normed a row whose router nearly ties moves by a
    tenth to a quarter of itself when rounding sends it to another expert: up to 0.09 for a step of one or two rows."""
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4, "differ": 0.01}
    if case["family"] in ("kepevik", "rifizen"):
        return {"rel": 2e-1, "max": 2.0, "differ": 0.15}
    return {"rel": 6e-2, "max": 0.5, "differ": 0.15}


# ----------------------------------------------------------------------------- the same in 64 bits
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _softplus(x):
    return torch.clamp(x, min=0.0) + torch.log1p(torch.exp(-x.abs()))


def _frequencies(dims, base, scaling=None):
    out = []
    for i in range(dims // 2):
        f = base ** (-2.0 * i / dims)
        if scaling:
            turns = scaling["original"] * f / (2.0 * math.pi)
            blend = min(max((turns - scaling["low"]) / (scaling["high"] - scaling["low"]), 0.0), 1.0)
            f = f * blend + f / scaling["factor"] * (1.0 - blend)
        out.append(f)
    return torch.tensor(out, dtype=torch.float64, device="cuda")


def _rotate(x, freqs):
    """x [B, S, heads, d]: channel i turns with channel i + half of the rotated ones."""
    half = freqs.numel()
    angle = torch.arange(x.shape[1], dtype=torch.float64, device="cuda")[:, None] * freqs
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]
    a, b = x[..., :half], x[..., half : 2 * half]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., 2 * half :]], dim=-1)


def _attend(q, k, v, scale, window=1 << 30, chunk=None, cap=None, bias=None, sink=None):
    """q [B, S, H, d] over k, v [B, S, G, .], causal; ``bias`` [H, S] by distance; ``sink`` [H] joins the denominator."""
    B, S, H, _ = q.shape
    rep = H // k.shape[2]
    out = torch.empty(B, S, H, v.shape[-1], dtype=q.dtype, device=q.device)
    pos = torch.arange(S, device=q.device)
    for b in range(B):
        kb, vb = k[b].repeat_interleave(rep, 1).permute(1, 2, 0).contiguous(), v[b].repeat_interleave(rep, 1).permute(1, 0, 2).contiguous()
        for i in range(0, S, 512):
            rows = pos[i : i + 512]
            s = torch.matmul(q[b, i : i + 512].permute(1, 0, 2).contiguous(), kb) * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            far = rows[:, None] - pos[None, :]
            if bias is not None:
                s = s + bias[:, far.clamp(min=0)]
            seen = (far >= 0) & (far < window)
            if chunk:
                seen &= (pos[None, :] // chunk) == (rows[:, None] // chunk)
            s = s.masked_fill(~seen, float("-inf"))
            top = s.amax(-1, keepdim=True)
            if sink is not None:
                top = torch.maximum(top, sink[:, None, None])
            e = torch.exp(s - top)
            total = e.sum(-1, keepdim=True)
            if sink is not None:
                total = total + torch.exp(sink[:, None, None] - top)
            out[b, i : i + 512] = torch.matmul(e / total, vb).permute(1, 0, 2)
    return out


def _conv(x, taps, bias=None):
    K, S = taps.shape[1], x.shape[1]
    padded = torch.cat([x.new_zeros(x.shape[0], K - 1, x.shape[2]), x], dim=1)
    y = sum(padded[:, j : j + S] * taps[:, j] for j in range(K))
    return y if bias is None else y + bias


def _recur(S, state, decay, write, read):
    """``state <- decay(t) * state; state <- write(t, state); out_t = read(t, state)`` for t < S."""
    out = []
    for t in range(S):
        state = write(t, state * decay(t))
        out.append(read(t, state))
    return torch.stack(out, dim=1)


class _Model:
    """The case's model in 64 bits over padded sequences [B, S]; tensors are drawn anew when they are used."""

    def __init__(self, case, seed):
        self.case, self.seed, self.config, self.shapes = case, seed, config_of(case), shapes_of(case)
        self.dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16

    def w(self, name):
        return tensor_of(name, self.shapes[name], self.seed, self.case["family"], self.dtype).double()

    def mm(self, x, name):
        return x @ self.w(name).T

    def logits(self, tokens, wanted):
        """``wanted``: (sequence, position) pairs -> rows of logits."""
        c, family = self.config, self.case["family"]
        at = torch.tensor(wanted, device="cuda").T
        if family == "llama":
            x = self.llama(tokens)
            x = _rms(x[at[0], at[1]], c["rms_norm_eps"]) * self.w("model.norm.weight")
            return self.mm(x, "model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight")
        eps = c["norm"]["eps"]
        x = self.w("embed")[tokens] * c.get("embedding", {"scale": 1.0})["scale"]
        if family == "mesolix":
            x = x + self.w("pos")[: tokens.shape[1]]
        order = [(i, None) for i in range(len(c["layers"]))]
        if "loop" in c:
            loop = c["loop"]
            again = [(i, t if i == loop["start"] else None) for t in range(loop["times"]) for i in range(loop["start"], loop["stop"])]
            order = order[: loop["start"]] + again + order[loop["stop"] :]
        for i, turn in order:
            if turn is not None:
                x = x + self.w("loop.step")[turn]
            layer = c["layers"][i]
            x = getattr(self, family)(x, f"l{layer.get('weights_of', i)}.", layer, eps)
        x = x[at[0], at[1]]
        if family == "taluvik":
            return self.mm(self.layer_norm(x, "final.norm", eps), "head")
        x = _rms(x, eps) * (self.w("final.norm") + (0.0 if family == "rifizen" else 1.0))
        return self.mm(x, "embed" if family == "kepevik" else "head")

    def llama(self, tokens):
        c = self.config
        H, G, d, eps = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["rms_norm_eps"]
        r = c["rope_scaling"]
        freqs = _frequencies(d, c["rope_theta"], dict(factor=r["factor"], low=r["low_freq_factor"], high=r["high_freq_factor"],
                                                      original=r["original_max_position_embeddings"]))
        x = self.w("model.embed_tokens.weight")[tokens]
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = _rms(x, eps) * self.w(p + "input_layernorm.weight")
            q, k, v = (self.mm(h, f"{p}self_attn.{t}_proj.weight").unflatten(-1, (-1, d)) for t in "qkv")
            o = _attend(_rotate(q, freqs), _rotate(k, freqs), v, d ** -0.5).flatten(2)
            x = x + self.mm(o, p + "self_attn.o_proj.weight")
            h = _rms(x, eps) * self.w(p + "post_attention_layernorm.weight")
            x = x + self.mm(_silu(self.mm(h, p + "mlp.gate_proj.weight")) * self.mm(h, p + "mlp.up_proj.weight"), p + "mlp.down_proj.weight")
        return x

    def layer_norm(self, x, name, eps):
        x = x - x.mean(-1, keepdim=True)
        return _rms(x, eps) * self.w(name) + self.w(name + ".b")

    def heads(self, h, name, d):
        return self.mm(h, name).unflatten(-1, (-1, d))

    def gated(self, h, p):
        return self.mm(_silu(self.mm(h, p + "gate")) * self.mm(h, p + "up"), p + "down")

    def mixture(self, h, p, mlp, family):
        """Routed experts: the rows that chose an expert go through it."""
        rows = h.flatten(0, 1)
        experts, top = mlp["router"]["experts"], mlp["router"]["top"]
        z = self.mm(rows, p + "router")
        if family == "kepevik":
            s = torch.softmax(z, -1)
            ids = (s + self.w(p + "correction")).topk(top, -1).indices
            weights = s.gather(1, ids)
        elif family == "rifizen":
            best = (z + self.w(p + "router.b")).topk(top, -1)
            ids, weights = best.indices, torch.softmax(best.values, -1)
        else:
            best = torch.sigmoid(z).topk(top, -1)
            ids, weights = best.indices, best.values
        out = torch.zeros_like(rows)
        for e in range(experts + mlp["router"].get("identity", 0)):
            row, place = (ids == e).nonzero(as_tuple=True)
            g, r = weights[row, place][:, None], rows[row]
            if e >= experts:
                y = g * r
            elif family == "mesolix":  # the weight is on what the expert reads
                y = self.gated(g * r, f"{p}e{e}.")
            else:
                y = g * self.gated(r, f"{p}e{e}.")
            out.index_add_(0, row, y)
        if mlp.get("shared"):
            y = self.gated(rows, p + "shared.")
            out = out + (torch.sigmoid(self.mm(rows, p + "shared.sg")) * y if family == "kepevik" else y)
        return out.view_as(h)

    def delta_rule(self, h, p, m, decay):
        """The gated delta rule; ``decay`` [B, S, H, 1 or d]."""
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (_silu(_conv(self.mm(h, p + t), self.w(p + t + ".conv"))).unflatten(-1, (-1, n)) for t, n in (("q", d), ("k", d), ("v", dv)))
        q, k = (u / torch.sqrt((u * u).sum(-1, keepdim=True) + 1e-6) for u in (q, k))
        q, k = (q * d ** -0.5).repeat_interleave(H // G, 2), k.repeat_interleave(H // G, 2)
        beta = torch.sigmoid(self.mm(h, p + "b"))

        def write(t, state):
            u = beta[:, t, :, None] * (v[:, t] - torch.matmul(k[:, t, :, None, :], state)[..., 0, :])
            return state + k[:, t, :, :, None] * u[..., None, :]

        return _recur(h.shape[1], h.new_zeros(h.shape[0], H, d, dv), lambda t: decay[:, t, :, :, None], write,
                      lambda t, state: torch.matmul(q[:, t, :, None, :], state)[..., 0, :])

    def taluvik(self, x, L, layer, eps):
        h, p, m = self.layer_norm(x, L + "norm1", eps), L + "mix.", layer["mixer"]
        if layer["type"] == "attention":
            freqs = _frequencies(m["rot"]["dims"], m["rot"]["base"], m["rot"]["scaling"])
            q, k = (_rms(_rotate(self.heads(h, p + t, m["dim"]), freqs), eps) for t in "qk")
            y = _attend(q, k, self.heads(h, p + "v", m["vdim"]), m["scale"], chunk=m["mask"]["size"], cap=m["softcap"], sink=self.w(p + "sink"))
            y = self.mm(y.flatten(2), p + "o")
        elif layer["type"] == "delta":
            decay = torch.exp(-torch.exp(self.w(p + "A_log")) * _softplus(self.mm(h, p + "a") + self.w(p + "dt_bias")))
            y = _rms(self.delta_rule(h, p, m, decay[..., None]), eps) * self.w(p + "norm") * _silu(self.heads(h, p + "g", m["vdim"]))
            y = self.mm(y.flatten(2), p + "o")
        else:
            I, N, R = m["inner"], m["state"], m["dt_rank"]
            u, z = self.mm(h, p + "in").split(I, -1)
            u = _silu(_conv(u, self.w(p + "conv"), self.w(p + "conv.b")))
            dt, Bm, Cm = self.mm(u, p + "x").split([R, N, N], -1)
            dt = _softplus(self.mm(dt, p + "dt") + self.w(p + "dt.b"))
            A = -torch.exp(self.w(p + "A_log"))
            y = _recur(h.shape[1], h.new_zeros(h.shape[0], I, N), lambda t: torch.exp(dt[:, t, :, None] * A),
                       lambda t, s: s + (dt[:, t] * u[:, t])[..., None] * Bm[:, t, None, :], lambda t, s: (s * Cm[:, t, None, :]).sum(-1))
            y = self.mm((y + self.w(p + "D") * u) * _silu(z), p + "o")
        g, up = self.mm(h, L + "mlp.gate"), self.mm(h, L + "mlp.up")
        g = 0.5 * g * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3)))
        return x + y + self.mm(g * up, L + "mlp.down")

    def kepevik(self, x, L, layer, eps):
        norm = lambda u, name: _rms(u, eps) * (1.0 + self.w(L + name))  # noqa: E731
        h, p, m = norm(x, "norm1"), L + "mix.", layer["mixer"]
        if layer["type"] == "mlstm":
            d, cap = m["dim"], m["gate_cap"]
            q, k, v = (self.heads(h, p + t, d) for t in "qkv")
            gi, gf = (cap * torch.tanh((self.mm(h, p + t) + self.w(p + t + ".b")) / cap) for t in "if")
            gf = -_softplus(-gf)
            v = torch.cat([v, torch.ones_like(v[..., :1])], -1)  # the normaliser is one more value
            top, tops = torch.zeros_like(gf[:, 0]), []
            for t in range(h.shape[1]):
                tops.append(torch.maximum(gf[:, t] + top, gi[:, t]))
                top = tops[-1]
            tops = torch.stack(tops, 1)
            before = torch.cat([torch.zeros_like(tops[:, :1]), tops[:, :-1]], 1)
            keep, take = torch.exp(gf + before - tops), torch.exp(gi - tops)
            o = _recur(h.shape[1], h.new_zeros(h.shape[0], m["heads"], d, m["vdim"] + 1), lambda t: keep[:, t, :, None, None],
                       lambda t, s: s + (take[:, t, :, None] * k[:, t])[..., None] * v[:, t, :, None, :],
                       lambda t, s: torch.matmul(q[:, t, :, None, :] * d ** -0.5, s)[..., 0, :])
            o = o[..., :-1] / (torch.maximum(o[..., -1].abs(), torch.exp(-tops)) + 1e-6)[..., None]
            y = self.mm(_rms(o, eps).flatten(2) * self.w(p + "norm") * torch.sigmoid(self.mm(h, p + "g")), p + "o")
        else:
            a, r = m["left"], m["right"]
            freqs = _frequencies(a["rot"]["dims"], a["rot"]["base"])
            q, k = self.heads(h, p + "left.q", a["dim"]), self.heads(h, p + "left.k", a["dim"])
            left = self.mm(_attend(_rotate(q, freqs), _rotate(k, freqs), k, a["scale"]).flatten(2), p + "left.o")
            rp = p + "right."
            step = _softplus(self.mm(self.mm(h, rp + "a1"), rp + "a2") + self.w(rp + "dt_bias")).unflatten(-1, (-1, r["dim"]))
            o = self.delta_rule(h, rp, r, torch.exp(-torch.exp(self.w(rp + "A_log"))[:, None] * step))
            gate = torch.sigmoid(self.mm(self.mm(h, rp + "g1"), rp + "g2")).unflatten(-1, (-1, r["vdim"]))
            right = self.mm((_rms(o, eps) * self.w(rp + "norm") * gate).flatten(2), rp + "o")
            y = m["left_scale"] * left + m["right_scale"] * right
        x = x + norm(y, "norm1b") * self.w(L + "ls1")
        h, q = norm(x, "norm2"), L + "mlp."
        if layer["mlp"]["kind"] == "dense":
            u = self.mm(h, q + "up") + self.w(q + "up.b")
            y = self.mm(0.5 * u * (1.0 + torch.erf(u / math.sqrt(2.0))), q + "down") + self.w(q + "down.b")
        else:
            y = self.mixture(h, q, layer["mlp"], "kepevik")
        return x + norm(y, "norm2b") * self.w(L + "ls2")

    def rifizen(self, x, L, layer, eps):
        norm = lambda u, name: _rms(u, eps) * self.w(L + name)  # noqa: E731
        h, p, a, r = norm(x, "norm1"), L + "mix.", layer["mixer"]["left"], layer["mixer"]["right"]
        H, S = a["heads"], h.shape[1]
        q, k = (_rms(self.heads(h, p + "left." + t, a["dim"]), eps) for t in "qk")
        slope = torch.tensor([2.0 ** (-8.0 * (i + 1) / H) for i in range(H)], dtype=torch.float64, device="cuda")
        bias = -slope[:, None] * torch.arange(S, dtype=torch.float64, device="cuda")
        y = _attend(q, k, self.heads(h, p + "left.v", a["vdim"]), a["scale"], window=a["mask"]["size"], cap=a["softcap"], bias=bias)
        left = norm(self.mm(y.flatten(2), p + "left.o"), "mix.left.out")
        freqs = _frequencies(r["rot"]["dims"], r["rot"]["base"])
        q, k = (_rotate(self.heads(h, p + "right." + t, r["dim"]), freqs) for t in "qk")
        v, k = self.heads(h, p + "right.v", r["vdim"]), k * r["dim"] ** -0.5
        decay = torch.tensor(r["decay"], dtype=torch.float64, device="cuda")[:, None, None]
        o = _recur(S, h.new_zeros(h.shape[0], r["heads"], r["dim"], r["vdim"]), lambda t: decay,
                   lambda t, s: s + k[:, t, :, :, None] * v[:, t, :, None, :], lambda t, s: torch.matmul(q[:, t, :, None, :], s)[..., 0, :])
        right = norm(self.mm(_rms(o, eps).flatten(2) * _silu(self.mm(h, p + "right.g")), p + "right.o"), "mix.right.out")
        x = x + norm(0.5 * (left + right), "norm1b")
        h = norm(x, "norm2")
        if layer["mlp"]["kind"] == "dense":
            y = self.mm(torch.relu(self.mm(h, L + "mlp.up")) ** 2, L + "mlp.down")
        else:
            y = self.mixture(h, L + "mlp.", layer["mlp"], "rifizen")
        return x + norm(y, "norm2b")

    def mesolix(self, x, L, layer, eps):
        norm = lambda u, name: _rms(u, eps) * (1.0 + self.w(L + name))  # noqa: E731
        h, p, m = norm(x, "norm1"), L + "mix.", layer["mixer"]
        S = h.shape[1]
        if layer["type"] == "mamba2":
            H, dv, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            z, u, dt = self.mm(h, p + "in").split([H * dv, H * dv + 2 * G * N, H], -1)
            u = _silu(_conv(u, self.w(p + "conv"), self.w(p + "conv.b")))
            u, Bm, Cm = u.split([H * dv, G * N, G * N], -1)
            u = u.unflatten(-1, (H, dv))
            Bm, Cm = (t.unflatten(-1, (G, N)).repeat_interleave(H // G, 2) for t in (Bm, Cm))
            dt = _softplus(dt + self.w(p + "dt_bias"))
            keep = torch.exp(-torch.exp(self.w(p + "A_log")) * dt)
            y = _recur(S, h.new_zeros(h.shape[0], H, N, dv), lambda t: keep[:, t, :, None, None],
                       lambda t, s: s + (dt[:, t, :, None] * Bm[:, t])[..., None] * u[:, t, :, None, :],
                       lambda t, s: torch.matmul(Cm[:, t, :, None, :], s)[..., 0, :])
            y = (y + self.w(p + "D")[:, None] * u).flatten(2) * _silu(z)
            y = _rms(y.unflatten(-1, (m["norm_groups"], -1)), eps).flatten(2) * self.w(p + "norm")
        elif layer["type"] == "attention":
            rel = self.w(p + "rel")
            half, steps, most = rel.shape[0] // 2, rel.shape[0] - rel.shape[0] // 2, m["bias_max"]
            row = []
            for n in range(S):  # a row a distance, then by the logarithm, its floor taken in whole numbers
                t = 0
                if n >= half:
                    while half + t + 1 < rel.shape[0] and most ** (t + 1) * half ** steps <= n ** steps * half ** (t + 1):
                        t += 1
                row.append(n if n < half else half + t)
            q, k, v = (self.heads(h, p + t, m["dim"]) for t in "qkv")
            y = _attend(q, k, v, m["scale"], window=m["mask"]["size"], bias=rel[torch.tensor(row, device="cuda")].T.contiguous())
            y = y.flatten(2) * torch.sigmoid(self.mm(h, p + "g"))
        else:
            cq = _rms(self.mm(h, p + "dq"), eps) * self.w(p + "dq.norm")
            latent = _rms(self.mm(h, p + "dkv"), eps) * self.w(p + "dkv.norm")
            y = _attend(self.heads(cq, p + "uq", m["dim"]), self.heads(latent, p + "uk", m["dim"]), self.heads(latent, p + "uv", m["vdim"]),
                        m["scale"], sink=self.w(p + "sink"))
            y = y.flatten(2) * torch.sigmoid(self.mm(h, p + "g"))
        x = x + self.mm(y, p + "o")
        h = norm(x, "norm2")
        if layer["mlp"]["kind"] == "dense":
            limit = layer["mlp"]["limit"]
            g, u = torch.clamp(self.mm(h, L + "mlp.gate"), max=limit), torch.clamp(self.mm(h, L + "mlp.up"), -limit, limit)
            return x + self.mm(g * torch.sigmoid(1.702 * g) * (u + 1.0), L + "mlp.down")
        return x + self.mixture(h, L + "mlp.", layer["mlp"], "mesolix")


@torch.no_grad()
def exact(case: dict, seed: int):
    """The logits that ``run`` returns, from 64-bit sequences without a cache; the drawn tokens have no such value."""
    p = plan(case, seed)
    rids = list(p["tokens"])
    longest = max(len(t) for t in p["tokens"].values())
    weights = sum(math.prod(s) for n, s in shapes_of(case).items() if ".mlp.e" not in n)
    if 2.0 * weights * longest * len(rids) > 5e14:
        return None
    tokens = torch.zeros(len(rids), longest, dtype=torch.long)
    for i, r in enumerate(rids):
        tokens[i, : len(p["tokens"][r])] = torch.tensor(p["tokens"][r])
    wanted, sizes = [], []
    for step in p["steps"]:
        rows = [(rids.index(r), first + w) for r, first, _, want in step for w in want]
        if rows:
            wanted += rows
            sizes.append(len(rows))
    logits = _Model(case, seed).logits(tokens.cuda(), wanted)
    result = {"logits": list(logits.split(sizes))}
    if case["sample"] >= 0:
        result["tokens"] = None
    return result
