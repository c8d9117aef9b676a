"""Generation work that a user of this library has it do: prompt steps and decode steps of the step function, over the seven
designs, both activation types, and sizes from one short prompt to thousands of tokens.

A case is a batch of sequences of unequal lengths (spread evenly from ``shortest`` to ``longest``, in a mixed order):

* ``kind`` "turn": what a request costs.  The sequences are opened, their prompts run in one step, ``new`` tokens a sequence
  are decoded, and the sequences are closed.
* ``kind`` "decode": what a running conversation costs.  The prompts are in the cache beforehand; a pass decodes ``new``
  tokens a sequence and takes the cache back to where it was, as a reply that is asked for again does.

The tokens that follow a prompt are given (as a replayed trace gives them) and lie on the device, where the generation loop has
them.  What comes back is the logits of the last place of every prompt and of every decoded token, which depend on all that the
prompt step left in the cache and in the sequences' states.  Weights are random, of the sizes that ``bench.py`` measures
at and with fewer layers; the small tensors (decays, taps, gates' biases) have the values that trained models have.
"""
from __future__ import annotations

import math
import zlib

import numpy as np
import torch

from turboquant_cpp_amd.engine.model import model_from_config
from turboquant_cpp_amd.engine.step import Engine

DEVICE = "cuda:0"
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}

# ------------------------------------------------------------------------------------------------ configurations

# Qwen1.5-MoE-A2.7B and Qwen2-57B-A14B layer sizes
_A27B = {
    "architectures": ["Qwen2MoeForCausalLM"], "model_type": "qwen2_moe", "vocab_size": 151936, "hidden_size": 2048,
    "num_attention_heads": 16, "num_key_value_heads": 16, "intermediate_size": 5632, "moe_intermediate_size": 1408,
    "shared_expert_intermediate_size": 5632, "num_experts": 60, "num_experts_per_tok": 4, "norm_topk_prob": False,
    "decoder_sparse_step": 1, "mlp_only_layers": [], "rope_theta": 1000000.0, "rms_norm_eps": 1e-6,
    "use_sliding_window": False, "sliding_window": 32768, "tie_word_embeddings": False, "torch_dtype": "bfloat16",
}
QWEN = {
    "a27b": _A27B,
    "a14b": dict(_A27B, hidden_size=3584, num_attention_heads=28, num_key_value_heads=4, intermediate_size=18944,
                 moe_intermediate_size=2560, shared_expert_intermediate_size=20480, num_experts=64, num_experts_per_tok=8,
                 sliding_window=131072),
}
# width, heads, kv heads, head size, experts, groups, kept groups, experts per token, expert width, dense width, latent
SIZES = {
    "small": dict(width=1024, heads=8, kv_heads=2, dim=128, experts=32, groups=4, keep=2, top=4, ff=768, vocab=32000,
                  dense_ff=2816, kv_rank=256),
    "medium": dict(width=2048, heads=16, kv_heads=4, dim=128, experts=64, groups=8, keep=2, top=4, ff=1408, vocab=32000,
                   dense_ff=5632, kv_rank=512),
    "large": dict(width=4096, heads=32, kv_heads=8, dim=128, experts=32, groups=4, keep=1, top=2, ff=4096, vocab=32000,
                  dense_ff=11008, kv_rank=512),
}


def _qwen2moe(z, layers, positions):
    return dict(z, num_hidden_layers=layers, max_window_layers=layers, max_position_embeddings=positions)


def _felepel(z, layers, positions):
    """Delta rule, attention, attention, ...; routed experts chosen within groups in every layer."""
    moe = {"kind": "moe", "expert": {"ff": z["ff"]},
           "router": {"experts": z["experts"], "top": z["top"], "groups": {"count": z["groups"], "keep": z["keep"]}}}
    delta = {"type": "channel_delta", "mlp": moe,
             "mixer": {"heads": z["heads"], "kv_heads": z["heads"], "dim": z["dim"], "vdim": z["dim"], "conv": 4,
                       "decay_rank": 64, "gate_rank": 64}}
    attn = {"type": "attention", "mlp": moe,
            "mixer": {"heads": z["heads"], "kv_heads": z["kv_heads"], "dim": z["dim"], "vdim": z["dim"],
                      "scale": z["dim"] ** -0.5, "softcap": 50.0, "mask": {"size": 1024}}}
    return {"architecture": "Felepel", "vocab": z["vocab"], "width": z["width"], "max_positions": positions,
            "norm": {"eps": 1e-5}, "layers": [dict(attn if i % 3 else delta) for i in range(layers)]}


def _taminex(z, layers, positions):
    """Delta rule, attention, latent attention, latent attention on the same latents; feed-forwards of two matrices."""
    H, G, D = z["heads"], z["kv_heads"], z["dim"]
    latent = {"heads": H, "dim": D, "vdim": D, "kv_rank": z["kv_rank"], "scale": D ** -0.5}
    kinds = [("delta", {"heads": H, "kv_heads": H, "dim": D, "vdim": D, "conv": 4}),
             ("attention", {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "rot": {"dims": D // 2, "base": 1e6}}),
             ("latent_attention", latent), ("latent_attention", latent)]
    out = []
    for i in range(layers):
        kind, mixer = kinds[i % 4]
        out.append({"type": kind, "mixer": dict(mixer, kv_from=i - 1) if i % 4 == 3 else dict(mixer),
                    "mlp": {"kind": "dense", "ff": z["dense_ff"] * 3 // 2}})
    return {"architecture": "Taminex", "vocab": z["vocab"], "width": z["width"], "norm": {"eps": 1e-5}, "logit_scale": 1.0,
            "logit_softcap": 40.0, "layers": out}


def _beronex(z, layers, positions):
    """Latent attention, lightning attention, windowed attention, attention on that layer's keys and values; dense
    feed-forwards and routed experts in turn."""
    H, G, D = z["heads"], z["kv_heads"], z["dim"]
    dense = {"kind": "dense", "ff": z["dense_ff"]}
    moe = {"kind": "moe", "router": {"experts": z["experts"], "top": z["top"]}, "expert": {"ff": z["ff"], "limit": 7.0}}
    yarn = {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}
    attn = {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "mask": {"size": 1024},
            "rot": {"dims": D, "base": 1e6, "scaling": yarn}}
    kinds = [("latent_attention", {"heads": H, "dim": D, "rot_dim": D // 2, "vdim": D, "kv_rank": min(z["kv_rank"], 512 - D // 2),
                                   "q_rank": 3 * z["kv_rank"] // 2, "scale": (D + D // 2) ** -0.5,
                                   "rot": {"dims": D // 2, "base": 1e4, "scaling": yarn}}, dense),
             ("lightning", {"heads": H, "dim": D, "vdim": D, "decay": [1.0 - 2.0 ** (-5.0 - 4.0 * h / H) for h in range(H)]}, moe),
             ("attention", attn, dense), ("attention", attn, moe)]
    out = []
    for i in range(layers):
        kind, mixer, mlp = kinds[i % 4]
        out.append({"type": kind, "mixer": dict(mixer, kv_from=i - 1) if i % 4 == 3 else dict(mixer), "mlp": mlp})
    return {"architecture": "Beronex", "vocab": z["vocab"], "width": z["width"], "norm": {"eps": 1e-5},
            "embedding": {"scale": 1.0}, "layers": out}


def _bosalix(z, layers, positions):
    """Windowed latent attention twice, sigmoid attention with kept first positions twice; experts of two matrices, some of
    them the identity."""
    H, G, D = z["heads"], z["kv_heads"], z["dim"]
    moe = {"kind": "moe", "router": {"experts": z["experts"], "identity": z["experts"] // 4, "top": z["top"]},
           "expert": {"ff": z["ff"] * 3 // 2}}
    kinds = [("latent_attention", {"heads": H, "dim": D, "rot_dim": D // 2, "vdim": D, "kv_rank": min(z["kv_rank"], 512 - D // 2),
                                   "q_rank": 3 * z["kv_rank"] // 2, "scale": (D + D // 2) ** -0.5, "mask": {"size": 1024},
                                   "rot": {"dims": D // 2, "base": 1e4}}),
             ("attention", {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "v_mix": True,
                            "mask": {"size": 1024, "keep_first": 4},
                            "rot": {"dims": D // 2, "base": 1e6,
                                    "scaling": {"factor": 8.0, "original": 4096, "low": 1.0, "high": 4.0}}})]
    return {"architecture": "Bosalix", "vocab": z["vocab"], "width": z["width"], "norm": {"eps": 1e-5}, "residual_mult": 0.5,
            "embedding": {"scale": 1.0},
            "layers": [{"type": kinds[i % 4 // 2][0], "mixer": dict(kinds[i % 4 // 2][1]), "mlp": moe} for i in range(layers)]}


def _gokezen(z, layers, positions):
    """Windowed attention and a matrix memory side by side in every layer; dense feed-forwards and routed experts with a
    shared one in turn; all but the first and the last layer are a loop of one pass."""
    H, G, D = z["heads"], z["kv_heads"], z["dim"]
    mixer = {"left": {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "mask": {"size": 1024}},
             "right": {"heads": H // 2, "dim": D, "vdim": D, "gate_cap": 15.0}, "left_scale": 1.0, "right_scale": 0.5}
    dense = {"kind": "dense", "ff": z["dense_ff"]}
    moe = {"kind": "moe", "expert": {"ff": z["ff"], "limit": 7.0}, "shared": {"ff": z["ff"], "limit": 7.0},
           "router": {"experts": z["experts"], "top": z["top"], "scale": 2.5, "groups": {"count": z["groups"], "keep": z["keep"]}}}
    return {"architecture": "Gokezen", "vocab": z["vocab"], "width": z["width"], "max_positions": positions,
            "norm": {"eps": 1e-5}, "loop": {"start": 1, "stop": layers - 1, "times": 1},
            "layers": [{"type": "parallel", "mixer": mixer, "mlp": moe if i % 2 else dense} for i in range(layers)]}


def _pumozen(z, layers, positions):
    """Attention whose values are its keys, differential attention, Mamba-2, differential attention on that layer's keys and
    values; dense clamped pairs and routed experts with a gated shared one in turn; a vector per token and layer."""
    H, G, D, W = z["heads"], z["kv_heads"], z["dim"], z["width"]
    dense = {"kind": "dense", "ff": z["dense_ff"], "limit": 7.0}
    moe = {"kind": "moe", "expert": {"ff": z["ff"], "limit": 7.0}, "shared": {"ff": z["ff"], "limit": 7.0},
           "router": {"experts": z["experts"], "top": z["top"], "scale": 1.5}}
    diff = {"heads": H, "kv_heads": G, "dim": D // 2, "vdim": D, "scale": (D // 2) ** -0.5, "diff": 0.6,
            "q_temp": {"coef": 0.1, "every": 1024}}
    kinds = [("attention", {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "rot": {"dims": D, "base": 1e4}}, dense),
             ("attention_2", diff, moe),
             ("mamba2", {"heads": 4 * W // D, "vdim": D // 2, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}, dense),
             ("attention_2", diff, moe)]
    out = []
    for i in range(layers):
        kind, mixer, mlp = kinds[i % 4]
        out.append({"type": kind, "mixer": dict(mixer, kv_from=i - 2) if i % 4 == 3 else dict(mixer), "mlp": mlp})
    return {"architecture": "Pumozen", "vocab": z["vocab"], "width": W, "norm": {"eps": 1e-5}, "token_side": {"dim": W // 16},
            "layers": out}


DESIGNS = {"qwen2moe": _qwen2moe, "felepel": _felepel, "taminex": _taminex, "beronex": _beronex, "bosalix": _bosalix,
           "gokezen": _gokezen, "pumozen": _pumozen}


def _config(case):
    z = (QWEN if case["design"] == "qwen2moe" else SIZES)[case["sizes"]]
    return DESIGNS[case["design"]](z, case["layers"], -(-(case["longest"] + case["new"] + 1) // 64) * 64)


# ------------------------------------------------------------------------------------------------ cases


def _case(name, design, sizes, layers, dtype, kind, sequences, shortest, longest, new):
    return {"name": name, "design": design, "sizes": sizes, "layers": layers, "dtype": dtype, "kind": kind,
            "sequences": sequences, "shortest": shortest, "longest": longest, "new": new}


def listed():
    bf16, f32 = "bfloat16", "float32"
    return [
        # one user's reply: the smallest step, a token of one conversation at a time
        _case("qwen_decode_one", "qwen2moe", "a27b", 8, bf16, "decode", 1, 2011, 2011, 1),
        # the headline: eight long conversations
        _case("qwen_decode_8_long", "qwen2moe", "a27b", 8, bf16, "decode", 8, 8167, 8167, 1),
        # a short question: every expert's matrices are read for a few rows each
        _case("qwen_question", "qwen2moe", "a27b", 8, bf16, "turn", 1, 97, 97, 0),
        # a document's prompt
        _case("qwen_prompt", "qwen2moe", "a27b", 8, bf16, "turn", 1, 2048, 2048, 0),
        # a full batch of unequal prompts at the larger model's sizes
        _case("qwen_large_prompts", "qwen2moe", "a14b", 3, bf16, "turn", 8, 512, 2788, 0),
        # a batch of unequal requests in true 32-bit, prompts and the first tokens behind them
        _case("qwen_requests_32bit", "qwen2moe", "a27b", 3, f32, "turn", 16, 1, 2048, 4),
        # a document's prompt and its first tokens: the delta rule with a decay per channel, chunked attention
        _case("felepel_prompt", "felepel", "medium", 4, bf16, "turn", 1, 2048, 2048, 2),
        # four unequal requests: the delta rule with a decay per head, latent attention
        _case("taminex_requests", "taminex", "medium", 4, bf16, "turn", 4, 129, 1500, 4),
        # a short chat turn, mostly decode steps of one sequence: lightning, latent and windowed attention
        _case("beronex_chat", "beronex", "medium", 4, bf16, "turn", 1, 97, 97, 16),
        # a prompt longer than the window and than one cut of a step: sigmoid and latent attention
        _case("bosalix_long_prompt", "bosalix", "medium", 4, bf16, "turn", 1, 3001, 3001, 4),
        # eight short unequal requests and their replies: attention and a matrix memory side by side
        _case("gokezen_requests", "gokezen", "medium", 4, bf16, "turn", 8, 33, 401, 8),
        # a document's prompt and its first tokens: differential attention, Mamba-2
        _case("pumozen_prompt", "pumozen", "medium", 4, bf16, "turn", 1, 1999, 1999, 4),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    design = rng.choice(["qwen2moe"] * 4 + [d for d in DESIGNS if d != "qwen2moe"])
    dtype = "float32" if rng.random() < 0.2 else "bfloat16"
    if design == "qwen2moe":
        sizes = "a14b" if dtype == "bfloat16" and rng.random() < 0.25 else "a27b"
        layers = 3 if sizes == "a14b" or dtype == "float32" else 8
        kind = rng.choice(["turn", "decode"])
    else:
        sizes = rng.choice(["small", "medium", "large"] if dtype == "bfloat16" else ["small", "medium"])
        layers, kind = 4, "turn"
    sequences = _log_uniform(rng, 1, 64)
    most = 32768 if kind == "decode" else 8192 if dtype == "bfloat16" else 4096
    longest = _log_uniform(rng, 2, min(8192 if kind == "decode" else 4096, most // sequences))
    shortest = rng.randint(1, longest) if sequences > 1 else longest
    new = rng.randint(1, 4) if kind == "decode" else rng.randint(0, 16)
    case = _case("", design, sizes, layers, dtype, kind, sequences, shortest, longest, new)
    del case["name"]
    return case


def _lengths(case):
    n, lo, hi = case["sequences"], case["shortest"], case["longest"]
    even = [hi if n == 1 else lo + (hi - lo) * i // (n - 1) for i in range(n)]
    stride = next(s for s in (7, 11, 13, 17) if math.gcd(s, n) == 1)      # a mixed order, the same each time
    return [even[i * stride % n] for i in range(n)]


def _tokens(case, seed):
    """The prompts, and the tokens that follow them [new, sequences]."""
    vocab = _config(case).get("vocab_size") or _config(case)["vocab"]
    rng = np.random.default_rng([seed, 1])
    return [rng.integers(0, vocab, n).tolist() for n in _lengths(case)], rng.integers(0, vocab, (case["new"], case["sequences"]))


# ------------------------------------------------------------------------------------------------ weights

# (mean, deviation) of the small tensors, by the last parts of their names; every other tensor is N(0, 0.02)
_SMALL = {
    "conv": (0.0, 0.4), "conv.b": (0.0, 0.1),            # taps of the short convolutions
    "A_log": (0.0, 0.5), "dt_bias": (-3.0, 0.5), "D": (1.0, 0.1),      # decays of about 0.95 a token
    "i.b": (0.0, 0.2), "f.b": (3.0, 0.5),                # gates that mostly keep
    "r1": (0.5, 0.05), "r2": (0.1, 0.01), "sink": (0.0, 0.5), "pb": (-6.0, 0.2), "vmix": (0.5, 0.0), "shift": (0.5, 0.1),
    "router": (0.0, 0.08), "gate.weight": (0.0, 0.08),   # routers that are sure of their choice: the last chosen weighs little
    "correction": (0.0, 0.002), "lq1": (0.0, 0.1), "lk1": (0.0, 0.1), "lq2": (0.0, 0.1), "lk2": (0.0, 0.1),
}


class _Weights:
    """A checkpoint in memory whose tensors are drawn when they are read, each from the seed and its name."""

    class _Entry:
        def __init__(self, shape, dtype):
            self.shape, self.dtype = shape, dtype

    def __init__(self, case, seed, table=()):
        self.design, self.dtype, self.seed = case["design"], DTYPES[case["dtype"]], seed
        stored = {"bfloat16": "BF16", "float32": "F32"}[case["dtype"]]
        self.shapes = {n: tuple(s) for n, (s, _role) in dict(table).items()}
        self.entries = {n: self._Entry(s, stored) for n, s in self.shapes.items()}

    def _values(self, name):
        last = name.split(".")
        for key in (".".join(last[-2:]), last[-1]):
            if key in _SMALL:
                return _SMALL[key]
        if last[-1] in ("norm1", "norm2", "norm1b", "norm2b", "norm") or name.endswith("norm.weight"):
            # a norm behind a feed-forward lets a part of it into the stream
            mean = 0.3 if last[-1] == "norm2b" or (last[-1] == "norm2" and self.design in ("taminex", "bosalix", "pumozen")) else 1.0
            stored_less_one = self.design == "bosalix" and name.count(".") == 1
            return mean - 1.0 if stored_less_one else mean, 0.1
        if self.design == "gokezen" and last[-1] == "down" and last[-2][:1] == "e":
            return 0.0, 0.005                               # nothing norms its experts' outputs
        return 0.0, 0.02

    def draw(self, name, shape):
        gen = torch.Generator(DEVICE).manual_seed((self.seed * 1_000_003 + zlib.crc32(name.encode())) & (2 ** 62 - 1))
        mean, std = self._values(name)
        return torch.empty(shape, dtype=torch.float32, device=DEVICE).normal_(mean, std, generator=gen).to(self.dtype) \
            if std else torch.full(shape, mean, dtype=self.dtype, device=DEVICE)

    def read(self, name):
        return self.draw(name, self.shapes[name])

    def __call__(self, name, *shape):
        return self.draw(name, shape).double()


# ------------------------------------------------------------------------------------------------ a pass


def prepare(case, seed):
    model = model_from_config(_config(case), case["dtype"])
    model.load(_Weights(case, seed, model.tensor_table()), DEVICE)
    prompts, follow = _tokens(case, seed)
    room = sum(-(-(len(p) + case["new"] + 1) // 64) * 64 for p in prompts)
    engine = Engine(model, max_tokens=room, page_size=64, max_slots=len(prompts))
    state = {"engine": engine, "prompts": prompts, "follow": torch.from_numpy(follow).to(torch.int32).to(DEVICE),
             "slots": None, "lengths": [len(p) for p in prompts]}
    if case["kind"] == "decode":
        state["slots"] = engine.open(len(prompts))
        for slot, prompt in zip(state["slots"], prompts):
            engine.step([slot], [prompt])
    for _ in range(2 if case["new"] else 1):      # a program that serves has captured its decode steps
        run(state)
    torch.cuda.synchronize()
    return state


def run(state):
    engine, follow, out = state["engine"], state["follow"], []
    slots = state["slots"] if state["slots"] is not None else engine.open(len(state["prompts"]))
    if state["slots"] is None:
        out.append(engine.step(slots, state["prompts"]))
    for i in range(follow.shape[0]):
        logits = engine.step_from_device(slots, follow[i])
        # the next step of the same shape may write its logits over these
        out.append(logits if i + 1 == follow.shape[0] else logits.clone())
    if state["slots"] is None:
        engine.close(slots)
    else:
        for slot, n in zip(slots, state["lengths"]):
            engine.cache.truncate(slot, n)
    return out


# ------------------------------------------------------------------------------------------------ what a pass needs


def _mixers(case, cfg):
    """Per layer: (key-query pairs' flops, window or chunk, bytes of a cached position, flops a token and bytes of state a
    sequence of a recurrence); a layer has one or both kinds."""
    elem = 2 if case["dtype"] == "bfloat16" else 4
    if case["design"] == "qwen2moe":
        hd = cfg["hidden_size"] // cfg["num_attention_heads"]
        return [(4 * cfg["num_attention_heads"] * hd, None, 2 * cfg["num_key_value_heads"] * hd * elem, 0, 0)] * case["layers"]

    def attention(m):
        H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m.get("vdim", m["dim"])
        return 2 * H * (D + V), (m.get("mask") or {}).get("size"), G * (D + V) * elem

    def recurrence(m, keys):
        return 6 * m["heads"] * keys * m["vdim"], 2 * 4 * m["heads"] * keys * m["vdim"]

    out = []
    for layer in cfg["layers"]:
        t, m = layer["type"], layer["mixer"]
        if t == "parallel":
            out.append(attention(m["left"]) + recurrence(m["right"], m["right"]["dim"]))
        elif t == "latent_attention":
            R = m.get("rot_dim", 0)
            out.append((2 * m["heads"] * (m["dim"] + R + m["vdim"]), (m.get("mask") or {}).get("size"), (m["kv_rank"] + R) * elem, 0, 0))
        elif t == "attention_2":
            out.append((2 * m["heads"] * 2 * (m["dim"] + m["vdim"]), None, m["kv_heads"] * (2 * m["dim"] + m["vdim"]) * elem, 0, 0))
        elif t == "attention":
            out.append(attention(m) + (0, 0))
        else:
            out.append((0, None, 0) + recurrence(m, m["state"] if t == "mamba2" else m["dim"]))
    return out


def work(case):
    cfg = _config(case)
    elem = 2 if case["dtype"] == "bfloat16" else 4
    H = cfg.get("hidden_size") or cfg["width"]
    V = cfg.get("vocab_size") or cfg["vocab"]
    tied = case["design"] in ("taminex", "gokezen", "pumozen")
    dense, head, experts = 0, V * H if tied else 0, {}
    for name, (shape, role) in model_from_config(cfg, case["dtype"]).tensor_table().items():
        n = int(np.prod(shape)) if len(shape) else 1
        parts = name.split(".")
        where = next((i for i, p in enumerate(parts) if p == "experts" or (p[:1] == "e" and p[1:].isdigit())), None)
        if where is not None:
            experts.setdefault(".".join(parts[:where]), [0, set()])
            experts[".".join(parts[:where])][0] += n
            experts[".".join(parts[:where])][1].add(".".join(parts[:where + 2]) if parts[where] == "experts" else parts[where])
        elif name in ("head", "lm_head.weight"):
            head = n
        elif role != "table":
            dense += n
    first = cfg["layers"][-1]["mlp"].get("router", {}) if "layers" in cfg else {}
    top = cfg["num_experts_per_tok"] if "num_experts_per_tok" in cfg else first.get("top", 0)
    dealt = first.get("identity", 0)      # identity experts have no weights and take their share of the choices
    lens = _lengths(case)
    mixers = _mixers(case, cfg)
    total_bytes = total_flops = 0.0

    def step(tokens, wanted, spans):
        """tokens run, rows of logits, and per sequence (first position, tokens)."""
        nonlocal total_bytes, total_flops
        b = (dense + head) * elem + wanted * V * 4 + tokens * H * elem
        f = 2.0 * tokens * dense + 2.0 * wanted * head
        for numel, names in experts.values():
            E = len(names)
            used = E * (1.0 - (1.0 - top / (E + dealt)) ** tokens)
            b += numel / E * used * elem
            f += 2.0 * tokens * top * E / (E + dealt) * numel / E
        for pair_flops, window, row_bytes, token_flops, state_bytes in mixers:
            for start, n in spans:
                reach = start + n if window is None else min(start + n, window)
                pairs = n * (start + (n + 1) / 2.0) if window is None or start + n <= window else \
                    sum(min(p + 1, window) for p in range(start, start + n))
                f += pair_flops * pairs + token_flops * n
                b += row_bytes * (min(start, reach) + n) + state_bytes
        total_bytes += b
        total_flops += f

    if case["kind"] == "turn":
        step(sum(lens), len(lens), [(0, n) for n in lens])
    for i in range(case["new"]):
        step(len(lens), len(lens), [(n + i, 1) for n in lens])
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    # bfloat16: rounding of activations to 8 bits, and a token whose last chosen expert is nearly level with the next may take
    # the other one; float32: sums in another order (four times what the 32-bit path is off 64 bits)
    return {"rel": 0.03, "max": 0.5} if case["dtype"] == "bfloat16" else {"rel": 4e-5, "max": 1e-3}


# ------------------------------------------------------------------------------------------------ the same in 64 bits


def _rms(y, eps, weight=None):
    y = y / torch.sqrt((y * y).mean(-1, keepdim=True) + eps)
    return y if weight is None else y * weight


def _unit(y):
    return y / torch.sqrt((y * y).sum(-1, keepdim=True) + 1e-6)


def _layer_norm(y, weight, bias, eps):
    c = y - y.mean(-1, keepdim=True)
    return c / torch.sqrt((c * c).mean(-1, keepdim=True) + eps) * weight + bias


_silu = torch.nn.functional.silu
_softplus = torch.nn.functional.softplus


def _gelu_tanh(z):
    return torch.nn.functional.gelu(z, approximate="tanh")


def _frequencies(rot):
    dims, base, s = rot["dims"], rot["base"], rot.get("scaling")
    f = base ** (-2.0 * np.arange(dims // 2) / dims)
    if s is None:
        return f, 1.0
    if "fast" in s:      # YaRN
        lo, hi = (dims * math.log(s["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(base)) for t in (s["fast"], s["slow"]))
        lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), dims - 1)
        ramp = np.clip((np.arange(dims // 2) - lo) / max(hi - lo, 0.001), 0.0, 1.0)
        return f / s["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(s["factor"]) + 1.0
    length = 2.0 * math.pi / f      # stretched by wavelength
    t = np.clip((s["original"] / length - s["low"]) / (s["high"] - s["low"]), 0.0, 1.0)
    return (1.0 - t) * f / s["factor"] + t * f, 1.0


def _rotate(x, pos, rot, layout):
    """x [T, heads, n]; pair i is (2 i, 2 i + 1) ("pairs") or (i, i + dims / 2) ("halves")."""
    n = rot["dims"] // 2
    f, factor = _frequencies(rot)
    a = pos[:, None] * torch.from_numpy(f).to(x.device)
    cos, sin = (torch.cos(a) * factor)[:, None], (torch.sin(a) * factor)[:, None]
    u, v = (x[..., 0:2 * n:2], x[..., 1:2 * n:2]) if layout == "pairs" else (x[..., :n], x[..., n:2 * n])
    out = x.clone()
    if layout == "pairs":
        out[..., 0:2 * n:2], out[..., 1:2 * n:2] = u * cos - v * sin, v * cos + u * sin
    else:
        out[..., :n], out[..., n:2 * n] = u * cos - v * sin, v * cos + u * sin
    return out


class _Exact:
    """A whole model in 64 bits over packed sequences: the matrices run on all tokens, mixers sequence by sequence."""

    def __init__(self, case, seed):
        self.case, self.cfg, self.w = case, _config(case), _Weights(case, seed)
        prompts, follow = _tokens(case, seed)
        self.seqs = [p + follow[:, i].tolist() for i, p in enumerate(prompts)]
        ends = np.cumsum([len(s) for s in self.seqs]).tolist()
        self.spans = list(zip([0] + ends[:-1], ends))
        self.tokens = torch.tensor([t for s in self.seqs for t in s], device=DEVICE)
        self.pos = torch.cat([torch.arange(len(s), device=DEVICE, dtype=torch.float64) for s in self.seqs])
        first = [[a + len(p) - 1 for (a, _), p in zip(self.spans, prompts)]] if case["kind"] == "turn" else []
        self.rows = first + [[a + len(p) + i for (a, _), p in zip(self.spans, prompts)] for i in range(case["new"])]
        self.H = self.cfg.get("hidden_size") or self.cfg["width"]
        self.V = self.cfg.get("vocab_size") or self.cfg["vocab"]
        self.kept = {}

    def lin(self, h, name, out, bias=None):
        y = h @ self.w(name, out, h.shape[-1]).T
        return y if bias is None else y + self.w(bias, out)

    def attend(self, q, k, v, scale, window=None, chunk=None, keep_first=0, cap=None, far=None, sink=None, weights="softmax"):
        """q [T, H, D], k [T, G, D], v [T, G, V] -> [T, H, V]; ``far``: (r1, r2) a head; ``sink`` [H] joins the denominator;
        ``weights`` "sigmoid" with ``sink`` as the bias of its scores."""
        H, G = q.shape[1], k.shape[1]
        out = torch.empty((q.shape[0], H, v.shape[2]), dtype=torch.float64, device=q.device)
        for a, b in self.spans:
            kk = k[a:b].permute(1, 2, 0).repeat_interleave(H // G, 0).contiguous()
            vv = v[a:b].permute(1, 0, 2).repeat_interleave(H // G, 0).contiguous()
            j = torch.arange(b - a, device=q.device)
            for lo in range(a, b, 512):
                hi = min(b, lo + 512)
                i = torch.arange(lo - a, hi - a, device=q.device)[:, None]
                s = q[lo:hi].permute(1, 0, 2).contiguous() @ kk * scale
                if cap is not None:
                    s = cap * torch.tanh(s / cap)
                if far is not None:
                    s = s - far[0][:, None, None] * torch.log1p(far[1][:, None, None] * (i - j).clamp(min=0))
                see = j <= i
                if window is not None:
                    see = see & ((i - j < window) | (j < keep_first))
                if chunk is not None:
                    see = see & (i // chunk == j // chunk)
                if weights == "sigmoid":
                    p = torch.where(see, torch.sigmoid(s + sink[:, None, None]), 0.0)
                else:
                    s = torch.where(see, s, -math.inf)
                    top = s.amax(-1, keepdim=True)
                    if sink is not None:
                        top = torch.maximum(top, sink[:, None, None])
                    p = torch.exp(s - top)
                    p = p / (p.sum(-1, keepdim=True) + (0.0 if sink is None else torch.exp(sink[:, None, None] - top)))
                out[lo:hi] = (p @ vv).permute(1, 0, 2)
        return out

    def conv(self, x, taps, bias=None):
        out = torch.zeros_like(x)
        K = taps.shape[1]
        for a, b in self.spans:
            full = torch.cat([torch.zeros((K - 1, x.shape[1]), dtype=x.dtype, device=x.device), x[a:b]])
            out[a:b] = sum(full[j:j + b - a] * taps[:, j] for j in range(K))
        return out if bias is None else out + bias

    def delta(self, q, k, v, beta, decay):
        """S <- decay S; u = beta (v - S^T k); S <- S + k u^T; o = S^T q; decay [T, H, D] or [T, H, 1]."""
        o = torch.empty_like(v)
        for a, b in self.spans:
            S = torch.zeros((q.shape[1], q.shape[2], v.shape[2]), dtype=torch.float64, device=q.device)
            for t in range(a, b):
                S *= decay[t][:, :, None]
                u = beta[t][:, None] * (v[t] - (k[t][:, None] @ S)[:, 0])
                S += k[t][:, :, None] * u[:, None]
                o[t] = (q[t][:, None] @ S)[:, 0]
        return o

    def scan(self, q, k, v, decay):
        """S <- decay S + k v^T, o = S^T q; decay [T, H]."""
        o = torch.empty_like(v)
        for a, b in self.spans:
            S = torch.zeros((v.shape[1], k.shape[2], v.shape[2]), dtype=torch.float64, device=q.device)
            for t in range(a, b):
                S = decay[t][:, None, None] * S + k[t][:, :, None] * v[t][:, None]
                o[t] = (q[t][:, None] @ S)[:, 0]
        return o

    def experts(self, h, ids, weights, E, run):
        out = torch.zeros_like(h)
        for e in range(E):
            t, j = (ids == e).nonzero(as_tuple=True)
            if len(t):
                out.index_add_(0, t, run(h[t], e) * weights[t, j][:, None])
        return out

    def gated(self, h, p, ff, act, names=("gate", "up", "down")):
        return self.lin(act(self.lin(h, p + names[0], ff), self.lin(h, p + names[1], ff)), p + names[2], self.H)

    @staticmethod
    def clamped(limit):
        return lambda g, u: g.clamp(max=limit) * torch.sigmoid(1.702 * g.clamp(max=limit)) * (u.clamp(-limit, limit) + 1.0)

    # ---- the designs
    def qwen2moe(self):
        c, H, eps, T = self.cfg, self.H, self.cfg["rms_norm_eps"], len(self.tokens)
        nh, g = c["num_attention_heads"], c["num_key_value_heads"]
        hd = H // nh
        rot = {"dims": hd, "base": c["rope_theta"]}
        x = self.w("model.embed_tokens.weight", self.V, H)[self.tokens]
        names = ("gate_proj.weight", "up_proj.weight", "down_proj.weight")
        swiglu = lambda a, b: _silu(a) * b      # noqa: E731
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = _rms(x, eps, self.w(p + "input_layernorm.weight", H))
            q, k, v = (self.lin(h, f"{p}self_attn.{n}_proj.weight", m * hd, f"{p}self_attn.{n}_proj.bias").view(T, m, hd)
                       for n, m in (("q", nh), ("k", g), ("v", g)))
            o = self.attend(_rotate(q, self.pos, rot, "halves"), _rotate(k, self.pos, rot, "halves"), v, hd ** -0.5)
            x = x + self.lin(o.reshape(T, H), p + "self_attn.o_proj.weight", H)
            h = _rms(x, eps, self.w(p + "post_attention_layernorm.weight", H))
            p += "mlp."
            s, ids = torch.softmax(self.lin(h, p + "gate.weight", c["num_experts"]), -1).topk(c["num_experts_per_tok"], -1)
            y = self.experts(h, ids, s, c["num_experts"], lambda r, e: self.gated(r, f"{p}experts.{e}.", c["moe_intermediate_size"], swiglu, names))
            shared = self.gated(h, p + "shared_expert.", c["shared_expert_intermediate_size"], swiglu, names)
            x = x + y + torch.sigmoid(self.lin(h, p + "shared_expert_gate.weight", 1)) * shared
        return _rms(x, eps, self.w("model.norm.weight", H)), "lm_head.weight"

    def grouped(self, s, r, score):
        if r.get("groups"):
            n = r["groups"]["count"]
            by = score(s.view(len(s), n, -1))
            keep = torch.zeros_like(by).scatter_(1, by.topk(r["groups"]["keep"], -1).indices, 1.0)
            s = torch.where(keep.repeat_interleave(s.shape[1] // n, 1) > 0, s, -1.0)
        return s.topk(r["top"], -1)

    def felepel(self):
        c, W, eps, T = self.cfg, self.H, self.cfg["norm"]["eps"], len(self.tokens)
        x = self.w("embed", self.V, W)[self.tokens] + self.w("pos", c["max_positions"], W)[self.pos.long()]
        for i, layer in enumerate(c["layers"]):
            p, m, f = f"l{i}.mix.", layer["mixer"], layer["mlp"]
            H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            h = _rms(x, eps, self.w(f"l{i}.norm1", W))
            if layer["type"] == "attention":
                q, k, v = (self.lin(h, p + n, a * d, p + n + ".b").view(T, a, d) for n, a, d in (("q", H, D), ("k", G, D), ("v", G, V)))
                o = self.attend(q, k, v, m["scale"], chunk=m["mask"]["size"], cap=m["softcap"], far=(self.w(p + "r1", H), self.w(p + "r2", H)))
                y = self.lin(o.reshape(T, -1), p + "o", W, p + "o.b")
            else:
                q, k, v = (_silu(self.conv(self.lin(h, p + n, H * D), self.w(f"{p}{n}.conv", H * D, m["conv"]))).view(T, H, D) for n in "qkv")
                a = self.lin(self.lin(h, p + "a1", m["decay_rank"]), p + "a2", H * D, p + "dt_bias").view(T, H, D)
                gate = torch.sigmoid(self.lin(self.lin(h, p + "g1", m["gate_rank"]), p + "g2", H * V)).view(T, H, V)
                decay = torch.exp(-torch.exp(self.w(p + "A_log", H))[:, None] * _softplus(a))
                o = self.delta(_unit(q) * D ** -0.5, _unit(k), v, torch.sigmoid(self.lin(h, p + "b", H)), decay)
                y = self.lin((_rms(o, eps, self.w(p + "norm", V)) * gate).reshape(T, -1), p + "o", W)
            x = x + _rms(y, eps, self.w(f"l{i}.norm1b", W))
            h, p, E = _rms(x, eps, self.w(f"l{i}.norm2", W)), f"l{i}.mlp.", f["router"]["experts"]
            s, ids = self.grouped(torch.softmax(self.lin(h, p + "router", E), -1), f["router"], lambda s: s.amax(-1))
            y = self.experts(h, ids, s, E, lambda r, e: self.gated(r, f"{p}e{e}.", f["expert"]["ff"], lambda a, b: _silu(a) * b))
            x = x + _rms(y, eps, self.w(f"l{i}.norm2b", W))
        return _rms(x, eps, self.w("final.norm", W)), "head"

    def taminex(self):
        c, W, eps, T = self.cfg, self.H, self.cfg["norm"]["eps"], len(self.tokens)
        x = self.w("embed", self.V, W)[self.tokens]
        for i, layer in enumerate(c["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            H, G, D, V = m["heads"], m.get("kv_heads"), m["dim"], m["vdim"]
            if layer["type"] == "attention":
                q, k, v = (self.lin(x, p + n, a * D, p + n + ".b").view(T, a, D) for n, a in (("q", H), ("k", G), ("v", G)))
                q, k = (_rotate(_rms(u, eps, self.w(f"{p}{n}.norm", D)), self.pos, m["rot"], "pairs") for u, n in ((q, "q"), (k, "k")))
                o = self.attend(q, k, v, m["scale"], sink=self.w(p + "sink", H)).reshape(T, -1)
            elif layer["type"] == "delta":
                q, k, v = (_silu(self.conv(self.lin(x, p + n, H * D), self.w(f"{p}{n}.conv", H * D, m["conv"]))).view(T, H, D) for n in "qkv")
                decay = torch.exp(-torch.exp(self.w(p + "A_log", H)) * _softplus(self.lin(x, p + "a", H, p + "dt_bias")))
                o = self.delta(_unit(q) * D ** -0.5, _unit(k), v, torch.sigmoid(self.lin(x, p + "b", H)), decay[:, :, None])
                o = _rms(o, eps, self.w(p + "norm", V)).reshape(T, -1) * _silu(self.lin(x, p + "g", H * V))
            else:
                rank = m["kv_rank"]
                self.kept[i] = self.kept[m["kv_from"]] if "kv_from" in m else _rms(self.lin(x, p + "dkv", rank), eps, self.w(p + "dkv.norm", rank))
                k, v = (self.lin(self.kept[i], p + n, H * D).view(T, H, D) for n in ("uk", "uv"))
                o = self.attend(self.lin(x, p + "q", H * D).view(T, H, D), k, v, m["scale"]).reshape(T, -1) * torch.sigmoid(self.lin(x, p + "g", H * V))
            x = x + _rms(self.lin(o, p + "o", W), eps, self.w(f"l{i}.norm1", W))
            y = self.lin(self.lin(x, f"l{i}.mlp.up", layer["mlp"]["ff"]).clamp(min=0.0) ** 2, f"l{i}.mlp.down", W)
            x = x + _rms(y, eps, self.w(f"l{i}.norm2", W))
        return _rms(x, eps, self.w("final.norm", W)), "embed"

    def latent(self, h, m, p, eps, layout, window):
        """Latent attention with a query latent and a rotated key part that all heads share."""
        T, H, D, R, V, rank = len(h), m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        q = self.lin(_rms(self.lin(h, p + "dq", m["q_rank"]), eps, self.w(p + "dq.norm", m["q_rank"])), p + "uq", H * (D + R)).view(T, H, D + R)
        down = self.lin(h, p + "dkv", rank + R)
        latent = _rms(down[:, :rank], eps, self.w(p + "dkv.norm", rank))
        turned = _rotate(down[:, None, rank:], self.pos, m["rot"], layout).expand(T, H, R)
        k = torch.cat([self.lin(latent, p + "uk", H * D).view(T, H, D), turned], -1)
        q = torch.cat([q[..., :D], _rotate(q[..., D:], self.pos, m["rot"], layout)], -1)
        o = self.attend(q, k, self.lin(latent, p + "uv", H * V).view(T, H, V), m["scale"], window=window)
        return self.lin(o.reshape(T, -1), p + "o", self.H)

    def beronex(self):
        c, W, eps, T = self.cfg, self.H, self.cfg["norm"]["eps"], len(self.tokens)
        x = self.w("embed", self.V, W)[self.tokens] * c["embedding"]["scale"]
        for i, layer in enumerate(c["layers"]):
            p, m, f = f"l{i}.mix.", layer["mixer"], layer["mlp"]
            H, D, V = m["heads"], m["dim"], m["vdim"]
            h = _rms(x, eps, self.w(f"l{i}.norm1", W))
            if layer["type"] == "latent_attention":
                y = self.latent(h, m, p, eps, "halves", None)
            elif layer["type"] == "lightning":
                q, k, v = (_silu(self.lin(h, p + n, H * D)).view(T, H, D) for n in "qkv")
                o = self.scan(q, k, v, torch.tensor(m["decay"], dtype=torch.float64, device=DEVICE).expand(T, H))
                y = self.lin(_rms(o.reshape(T, -1), eps, self.w(p + "norm", H * V)) * torch.sigmoid(self.lin(h, p + "g", H * V)), p + "o", W)
            else:
                G = m["kv_heads"]
                self.kept[i] = self.kept[m["kv_from"]] if "kv_from" in m else (
                    _rms(_rotate(self.lin(h, p + "k", G * D).view(T, G, D), self.pos, m["rot"], "pairs"), eps), self.lin(h, p + "v", G * V).view(T, G, V))
                q = _rms(_rotate(self.lin(h, p + "q", H * D).view(T, H, D), self.pos, m["rot"], "pairs"), eps)
                o = self.attend(q, *self.kept[i], m["scale"], window=m["mask"]["size"]) * torch.sigmoid(self.lin(h, p + "g", H))[:, :, None]
                y = self.lin(o.reshape(T, -1), p + "o", W)
            x = x + _rms(y, eps, self.w(f"l{i}.norm1b", W))
            h, p = _rms(x, eps, self.w(f"l{i}.norm2", W)), f"l{i}.mlp."
            if f["kind"] == "dense":
                y = self.gated(h, p, f["ff"], lambda a, b: _gelu_tanh(a) * b)
            else:
                z, ids = self.lin(h, p + "router", f["router"]["experts"], p + "router.b").topk(f["router"]["top"], -1)
                y = self.experts(h, ids, torch.softmax(z, -1), f["router"]["experts"],
                                 lambda r, e: self.gated(r, f"{p}e{e}.", f["expert"]["ff"], self.clamped(f["expert"]["limit"])))
            x = x + _rms(y, eps, self.w(f"l{i}.norm2b", W))
        return _rms(x, eps, self.w("final.norm", W)), "head"

    def bosalix(self):
        c, W, eps, T, mult = self.cfg, self.H, self.cfg["norm"]["eps"], len(self.tokens), self.cfg["residual_mult"]
        x = self.w("embed", self.V, W)[self.tokens] * c["embedding"]["scale"]
        first = None
        for i, layer in enumerate(c["layers"]):
            p, m, f = f"l{i}.mix.", layer["mixer"], layer["mlp"]
            before = torch.cat([torch.zeros_like(x[:1]), x[:-1]])
            before[[a for a, _ in self.spans]] = 0.0
            h = x + (before - x) * self.w(f"l{i}.shift", W)
            if layer["type"] == "latent_attention":
                y = self.latent(h, m, p, eps, "pairs", m["mask"]["size"])
            else:
                H, G, D = m["heads"], m["kv_heads"], m["dim"]
                q, k, v = (self.lin(h, p + n, a * D, p + n + ".b").view(T, a, D) for n, a in (("q", H), ("k", G), ("v", G)))
                q, k = (_rotate(_rms(u, eps, self.w(f"{p}{n}.norm", D)), self.pos, m["rot"], "halves") for u, n in ((q, "q"), (k, "k")))
                v = _rms(v, eps)
                if first is not None:
                    mix = self.w(p + "vmix")
                    v = (1.0 - mix) * v + mix * first
                first = v if first is None else first
                o = self.attend(q, k, v, m["scale"], window=m["mask"]["size"], keep_first=m["mask"]["keep_first"],
                                sink=self.w(p + "pb", H), weights="sigmoid")
                y = self.lin(o.reshape(T, -1), p + "o", W, p + "o.b")
            x = x + mult * _rms(y, eps) * (1.0 + self.w(f"l{i}.norm1", W))
            p, E, n = f"l{i}.mlp.", f["router"]["experts"], f["router"]["identity"]
            s = torch.softmax(self.lin(x, p + "router", E + n), -1)
            ids = (s + self.w(p + "correction", E + n)).topk(f["router"]["top"], -1).indices
            s = s.gather(1, ids)
            y = self.experts(x, ids, s, E, lambda r, e: self.lin(torch.nn.functional.gelu(self.lin(r, f"{p}e{e}.up", f["expert"]["ff"])), f"{p}e{e}.down", W))
            y = y + (s * (ids >= E)).sum(-1, keepdim=True) * x
            x = x + mult * _rms(y, eps) * (1.0 + self.w(f"l{i}.norm2", W))
        return _rms(x, eps) * (1.0 + self.w("final.norm", W)), "head"

    def memory(self, h, m, p, eps):
        T, H, D, V, cap = len(h), m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q, k, v = (self.lin(h, p + n, H * D).view(T, H, D) for n in "qkv")
        q = q * D ** -0.5
        gi = cap * torch.tanh(self.lin(h, p + "i", H, p + "i.b") / cap)
        gf = -_softplus(-cap * torch.tanh(self.lin(h, p + "f", H, p + "f.b") / cap))
        o = torch.empty((T, H, V), dtype=torch.float64, device=h.device)
        for a, b in self.spans:
            S = torch.zeros((H, D, V + 1), dtype=torch.float64, device=h.device)      # the last column is n
            vv = torch.cat([v[a:b], torch.ones_like(v[a:b, :, :1])], -1)
            top = torch.zeros(H, dtype=torch.float64, device=h.device)
            for t in range(a, b):
                new = torch.maximum(gf[t] + top, gi[t])
                S = torch.exp(gf[t] + top - new)[:, None, None] * S + torch.exp(gi[t] - new)[:, None, None] * k[t][:, :, None] * vv[t - a][:, None]
                top = new
                r = (q[t][:, None] @ S)[:, 0]
                o[t] = r[:, :V] / (torch.maximum(r[:, V:].abs(), torch.exp(-new)[:, None]) + 1e-6)
        o = _rms(o, eps).reshape(T, -1) * self.w(p + "norm", H * V) * torch.sigmoid(self.lin(h, p + "g", H * V))
        return self.lin(o, p + "o", self.H)

    def gokezen(self):
        c, W, eps, T = self.cfg, self.H, self.cfg["norm"]["eps"], len(self.tokens)
        x = self.w("embed", self.V, W)[self.tokens] + self.w("pos", c["max_positions"], W)[self.pos.long()]
        for i, layer in enumerate(c["layers"]):      # the loop has one pass
            p, m, f = f"l{i}.mix.left.", layer["mixer"]["left"], layer["mlp"]
            if i == c["loop"]["start"]:
                x = x + self.w("loop.step", c["loop"]["times"], W)[0]
            h = _rms(x, eps, self.w(f"l{i}.norm1", W))
            q, k, v = (self.lin(h, p + n, a * m["dim"]).view(T, a, m["dim"]) for n, a in (("q", m["heads"]), ("k", m["kv_heads"]), ("v", m["kv_heads"])))
            left = self.lin(self.attend(q, k, v, m["scale"], window=m["mask"]["size"]).reshape(T, -1), p + "o", W)
            y = layer["mixer"]["left_scale"] * left + layer["mixer"]["right_scale"] * self.memory(h, layer["mixer"]["right"], f"l{i}.mix.right.", eps)
            p = f"l{i}.mlp."
            if f["kind"] == "dense":
                y = y + self.gated(h, p, f["ff"], lambda a, b: _gelu_tanh(a) * b)
            else:
                act, r = self.clamped(f["expert"]["limit"]), f["router"]
                s, ids = self.grouped(torch.sigmoid(self.lin(h, p + "router", r["experts"])), r, lambda s: s.topk(2, -1).values.sum(-1))
                y = y + self.experts(h, ids, s / (s.sum(-1, keepdim=True) + 1e-20) * r["scale"], r["experts"],
                                     lambda u, e: self.gated(u, f"{p}e{e}.", f["expert"]["ff"], act))
                y = y + self.gated(h, p + "shared.", f["shared"]["ff"], self.clamped(f["shared"]["limit"]))
            x = x + y
        return _rms(x, eps, self.w("final.norm", W)), "embed"

    def mamba2(self, h, m, p, eps):
        T, H, V, N, G = len(h), m["heads"], m["vdim"], m["state"], m["groups"]
        inner = H * V
        z, xbc, dt = self.lin(h, p + "in", 2 * inner + 2 * G * N + H).split([inner, inner + 2 * G * N, H], -1)
        xbc = _silu(self.conv(xbc, self.w(p + "conv", inner + 2 * G * N, m["conv"]), self.w(p + "conv.b", inner + 2 * G * N)))
        x, B, C = xbc.split([inner, G * N, G * N], -1)
        x = x.reshape(T, H, V)
        B, C = (u.reshape(T, G, N).repeat_interleave(H // G, 1) for u in (B, C))
        dt = _softplus(dt + self.w(p + "dt_bias", H))
        y = self.scan(C, B, x * dt[:, :, None], torch.exp(-torch.exp(self.w(p + "A_log", H)) * dt)) + self.w(p + "D", H)[:, None] * x
        y = _rms((y.reshape(T, inner) * _silu(z)).view(T, m["norm_groups"], -1), eps).reshape(T, inner)
        return self.lin(y * self.w(p + "norm", inner), p + "o", self.H)

    def pumozen(self):
        c, W, eps, T = self.cfg, self.H, self.cfg["norm"]["eps"], len(self.tokens)
        x = self.w("embed", self.V, W)[self.tokens]
        dim, n = c["token_side"]["dim"], len(c["layers"])
        side = self.w("side.embed", self.V, n * dim)[self.tokens]
        for i, layer in enumerate(c["layers"]):
            p, m, f = f"l{i}.mix.", layer["mixer"], layer["mlp"]
            H, G, D = m["heads"], m.get("kv_heads"), m.get("dim")
            if layer["type"] == "mamba2":
                y = self.mamba2(x, m, p, eps)
            elif layer["type"] == "attention":
                raw = self.lin(x, p + "k", G * D)
                q, k = (_rotate(_rms(u, eps, self.w(f"{p}{a}.norm", u.shape[1])).view(T, -1, D), self.pos, m["rot"], "halves")
                        for u, a in ((self.lin(x, p + "q", H * D), "q"), (raw, "k")))
                o = self.attend(q, k, raw.view(T, G, D), m["scale"], sink=torch.zeros(H, dtype=torch.float64, device=DEVICE))
                y = self.lin(o.reshape(T, -1), p + "o", W)
            else:
                V = m["vdim"]
                self.kept[i] = self.kept[m["kv_from"]] if "kv_from" in m else (
                    _rms(self.lin(x, p + "k", G * 2 * D).view(T, G, 2, D), eps, self.w(p + "k.norm", D)), self.lin(x, p + "v", G * V).view(T, G, V))
                q = _rms(self.lin(x, p + "q", H * 2 * D).view(T, H, 2, D), eps, self.w(p + "q.norm", D))
                q = q * (1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((self.pos + 1) / m["q_temp"]["every"]) + 1.0))[:, None, None, None]
                k, v = self.kept[i]
                a1, a2 = (self.attend(q[:, :, j].contiguous(), k[:, :, j].contiguous(), v, m["scale"]) for j in range(2))
                l1, l2 = (torch.exp(self.w(f"{p}lq{j}", D) @ self.w(f"{p}lk{j}", D)) for j in (1, 2))
                o = _rms(a1 - (l1 - l2 + m["diff"]) * a2, eps) * (1.0 - m["diff"])
                y = self.lin(o.reshape(T, -1) * torch.sigmoid(self.lin(x, p + "g", H * V)), p + "o", W)
            x = x + _layer_norm(y, self.w(f"l{i}.norm1", W), self.w(f"l{i}.norm1.b", W), eps)
            p = f"l{i}.mlp."
            if f["kind"] == "dense":
                y = self.gated(x, p, f["ff"], self.clamped(f["limit"]))
            else:
                r = f["router"]
                s, ids = torch.softmax(self.lin(x, p + "router", r["experts"]), -1).topk(r["top"], -1)
                y = self.experts(x, ids, s / (s.sum(-1, keepdim=True) + 1e-20) * r["scale"], r["experts"],
                                 lambda u, e: self.gated(u, f"{p}e{e}.", f["expert"]["ff"], self.clamped(f["expert"]["limit"])))
                y = y + torch.sigmoid(self.lin(x, p + "shared.sg", 1)) * self.gated(x, p + "shared.", f["shared"]["ff"], self.clamped(f["shared"]["limit"]))
            x = x + _layer_norm(y, self.w(f"l{i}.norm2", W), self.w(f"l{i}.norm2.b", W), eps)
            y = self.lin(_gelu_tanh(self.lin(x, f"l{i}.side.gate", dim)) * side[:, i * dim:(i + 1) * dim], f"l{i}.side.proj", W)
            x = x + _rms(y, eps, self.w(f"l{i}.side.norm", W))
        return _layer_norm(x, self.w("final.norm", W), self.w("final.norm.b", W), eps), "embed"

    def run(self):
        h, head = getattr(self, self.case["design"])()
        head = self.w(head, self.V, self.H)
        out = [h[rows] @ head.T * self.cfg.get("logit_scale", 1.0) for rows in self.rows]
        cap = self.cfg.get("logit_softcap")
        return out if cap is None else [cap * torch.tanh(y / cap) for y in out]


def exact(case, seed):
    return _Exact(case, seed).run()
