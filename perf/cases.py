"""What this framework is used for, as measurable cases: requests served by an `Engine`.

A pass of a case is a request batch from its first token to its last: slots are taken, the prompts run as one step (or
in pieces), then `new` tokens go through the captured decode step, and the slots are given back.  The tokens that are fed
are given beforehand (a replayed trace, or a text that is scored), so that every pass and every implementation computes the
same thing; the choice of the next token is made on the GPU in every step all the same, and is among the outputs beside
the logits.

A case's keys: `design` (the architecture), `width`, `layers`, `heads`, `kv_heads`, `head`, `ff`, `vocab` (its sizes; what
else a design needs follows from these, see `config_of`), `dtype`, `sequences`, `shortest`..`longest` (prompt lengths,
in uneven steps), `new` (tokens decoded per sequence), `piece` (prompts are fed in pieces of so many tokens; 0:
whole), `want` ("last": logits of the last prompt token; "all": of every prompt token), `temperature` (0: greedy).
"""
from __future__ import annotations

import hashlib
import math
import random

import numpy as np
import torch

import rbitnet_amd
from rbitnet_amd.engine.model import expected_tensors

DEVICE = "cuda:0"
F64 = torch.float64
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}


# ---------------------------------------------------------------------- the cases
def _case(name, design, sizes, dtype, sequences, lengths, new, piece=0, want="last", temperature=0.0):
    width, layers, heads, kv_heads, head, ff, vocab = sizes
    return {"name": name, "design": design, "width": width, "layers": layers, "heads": heads, "kv_heads": kv_heads, "head": head,
            "ff": ff, "vocab": vocab, "dtype": dtype, "sequences": sequences, "shortest": lengths[0], "longest": lengths[1],
            "new": new, "piece": piece, "want": want, "temperature": temperature}


TINY = (96, 3, 4, 1, 24, 256, 384)                       # the smallest configuration with grouped heads and scaled rotation
LLAMA3_8B = (4096, 32, 32, 8, 128, 14336, 128256)
LLAMA2_7B = (4096, 32, 32, 32, 128, 11008, 32000)
W3072 = (3072, 28, 24, 8, 128, 8192, 128256)
W2048 = (2048, 16, 32, 8, 64, 8192, 128256)
W1024 = (1024, 12, 16, 4, 64, 4096, 32000)


def listed():
    return [
        # a toy model in float32, sampled: every launch counts, nothing else does
        _case("tiny_float32", "llama", TINY, "float32", 4, (1, 77), 24, want="all", temperature=0.8),
        # one user's long document, fed in pieces, and a short answer: prefill on top of a cache, decode at batch 1
        _case("document_8b", "llama", LLAMA3_8B, "bfloat16", 1, (8000, 8000), 32, piece=2048),
        # the headline: a prompt of 2,048 tokens to its first token
        _case("prompt_8b", "llama", LLAMA3_8B, "bfloat16", 1, (2048, 2048), 0),
        # the headline: a chat server's ordinary batch
        _case("batch8_8b", "llama", LLAMA3_8B, "bfloat16", 8, (512, 512), 48),
        # the headline: a full server, short questions
        _case("batch64_8b", "llama", LLAMA3_8B, "bfloat16", 64, (24, 96), 24),
        # heads without groups, unequal prompts
        _case("ragged16_7b", "llama", LLAMA2_7B, "bfloat16", 16, (64, 1024), 24),
        # the exact mode: true float32, logits of every prompt token (a text that is scored), then a few tokens
        _case("scored_float32", "llama", W3072, "float32", 4, (65, 512), 12, want="all"),
        # the other designs, each at its middle size: a few prompts of ordinary lengths and an answer
        _case("bagonex_w2048", "bagonex", W2048, "bfloat16", 4, (200, 1500), 32),
        _case("tigutar_w2048", "tigutar", W2048, "bfloat16", 4, (200, 1500), 32),
        _case("menerax_w2048", "menerax", W2048, "bfloat16", 4, (200, 1500), 32),
        _case("lilevik_w2048", "lilevik", W2048, "bfloat16", 4, (200, 1500), 32),
        _case("goperax_w2048", "goperax", W2048, "bfloat16", 4, (200, 1500), 32),
    ]


def _spread(rng, lo, hi):
    """A whole number of lo..hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    """Any design at any of the sizes, from one short prompt to batches of 64, so many tokens that the case costs no more
    than the largest listed one."""
    design = rng.choice(["llama", "llama", "llama", "bagonex", "tigutar", "menerax", "lilevik", "goperax"])
    # the exact mode is drawn for the designs whose results have no jumps (a router's near tie may go either way)
    dtype = "float32" if rng.random() < 0.25 and design in ("llama", "bagonex", "menerax") else "bfloat16"
    if design == "llama":
        sizes = rng.choice([TINY, W1024, W2048, W3072, LLAMA2_7B, LLAMA3_8B])
    else:
        sizes = rng.choice([W1024, W2048]) if dtype == "bfloat16" else W1024
    if sizes[0] >= 1024:                                  # depth varies, the rest is the configuration's
        sizes = (sizes[0], _spread(rng, 4, sizes[1])) + sizes[2:]
    sequences = _spread(rng, 1, 64)
    # tokens of all prompts together: what the largest listed cases bring, less in float32 (a tenth of the rate)
    budget = 8000 if dtype == "bfloat16" else 1200
    budget = min(budget, 100 * sizes[1] + 400) if sizes[0] < 1024 else budget
    longest = max(2, min(_spread(rng, 8, 4096), budget // sequences))
    shortest = max(1, longest // rng.choice([1, 2, 4, 16]))
    case = _case("", design, sizes, dtype, sequences, (shortest, longest), max(_spread(rng, 4, 32), -(-16 // sequences)),
                 piece=rng.choice([0, 0, 0, max(16, longest // 3)]), want="all" if dtype == "float32" and rng.random() < 0.5 else "last")
    if case["width"] < 1024:                              # a longer sequence than the tiny configuration allows is an error
        case["longest"] = min(case["longest"], 200)
        case["shortest"] = min(case["shortest"], case["longest"])
    del case["name"]
    return case


# ---------------------------------------------------------------------- the configurations
def config_of(case):
    """config.json of the case's model, as a dict."""
    e, n, h, g, d, ff, vocab = (case[k] for k in ("width", "layers", "heads", "kv_heads", "head", "ff", "vocab"))
    if case["design"] == "llama":
        tiny = e < 1024
        config = {"architectures": ["LlamaForCausalLM"], "hidden_size": e, "num_hidden_layers": n, "num_attention_heads": h,
                  "num_key_value_heads": g, "head_dim": d, "intermediate_size": ff, "vocab_size": vocab,
                  "rope_theta": 10000.0 if g == h else 500000.0, "rms_norm_eps": 1e-6 if tiny else 1e-5,
                  "max_position_embeddings": 256 if tiny else 16384, "tie_word_embeddings": tiny, "rope_style": "half"}
        if tiny:
            config["rope_scaling"] = {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                                      "original_max_position_embeddings": 32}
        return config
    make = {"bagonex": _bagonex, "tigutar": _tigutar, "menerax": _menerax, "lilevik": _lilevik, "goperax": _goperax}
    config = make[case["design"]](e, n, h, g, ff)
    config.update({"architecture": case["design"].capitalize(), "vocab": vocab, "width": e})
    return config


def _bagonex(e, n, h, g, ff):
    """A delta rule with decays per channel alternates with attention through latents; every second latent layer reads the
    latents of the one before it."""
    dim, rank = e // 16, e // 16
    layers = []
    for i in range(n):
        if i % 2 == 0:
            mixer = {"heads": 16, "kv_heads": 16, "dim": dim, "vdim": dim, "conv": 4, "decay_rank": rank, "gate_rank": rank}
        else:
            mixer = {"heads": 16, "dim": dim, "vdim": dim, "q_rank": e * 3 // 8, "kv_rank": rank, "scale": dim ** -0.5}
            if i % 4 == 3:
                mixer["kv_from"] = i - 2
        layers.append({"type": "latent_attention" if i % 2 else "channel_delta", "mixer": mixer, "mlp": {"kind": "dense", "ff": ff}})
    return {"streams": 2, "norm": {"eps": 1e-6}, "canon": {"taps": 4}, "logit_softcap": 30.0, "layers": layers}


def _tigutar(e, n, h, g, ff):
    """Groups of four: gated attention with sinks, a gated delta rule, and twice windowed attention beside gated linear
    attention; dense feed-forwards alternate with 4 of 16 experts."""
    soft = {"heads": h, "kv_heads": g, "dim": 64, "vdim": 64, "rot": {"base": 10000.0, "dims": 64}, "scale": 0.125}
    left = {"heads": h // 2, "kv_heads": g // 2, "dim": 64, "vdim": 128, "rot": {"base": 250000.0, "dims": 64}, "scale": 0.125,
            "mask": {"size": 1024}}
    right = {"heads": h // 4, "dim": 64, "vdim": 128, "tau": 8.0, "decay_rank": 64}
    delta = {"heads": h // 2, "kv_heads": h // 4, "dim": 128, "vdim": 128, "conv": 4}
    dense = {"kind": "dense", "ff": ff}
    routed = {"kind": "moe", "expert": {"ff": ff // 4, "limit": 7.0}, "router": {"experts": 16, "top": 4}}
    layers = []
    for i in range(n):
        if i % 4 == 0:
            layers.append({"type": "attention", "mixer": dict(soft, kv_from=i - 4) if i % 8 == 4 else dict(soft), "mlp": dense})
        elif i % 4 == 1:
            layers.append({"type": "delta", "mixer": dict(delta), "mlp": routed})
        else:
            layers.append({"type": "parallel", "mixer": {"left": dict(left), "right": dict(right)}, "mlp": dense if i % 4 == 2 else routed})
    return {"residual_mult": 0.5, "norm": {"eps": 1e-5}, "layers": layers}


def _latent(e, h):
    return {"heads": h, "dim": 64, "rot_dim": 32, "vdim": 64, "q_rank": max(256, e * 3 // 8), "kv_rank": 96, "scale": 96 ** -0.5,
            "rot": {"base": 10000.0, "dims": 32}}


def _menerax(e, n, h, g, ff):
    """Of four layers three attend through latents, the third has windowed attention (kept first tokens, capped scores, a
    convolution) beside time mixing."""
    left = {"heads": h // 2, "kv_heads": g // 2, "dim": 128, "vdim": 128, "conv": 4,
            "rot": {"base": 1000000.0, "dims": 64, "scaling": {"factor": 4.0, "low": 1.0, "high": 2.0, "original": 4096}},
            "scale": 128 ** -0.5, "softcap": 50.0, "mask": {"size": 1024, "keep_first": 64}}
    right = {"heads": e // 128, "dim": 64, "decay_rank": 64}
    layers = []
    for i in range(n):
        mlp = {"kind": "dense", "ff": ff, "limit": 7.0}
        if i % 4 == 2:
            layers.append({"type": "parallel", "mlp": mlp,
                           "mixer": {"left": dict(left), "right": dict(right), "left_scale": 0.5, "right_scale": 1.0}})
        else:
            layers.append({"type": "latent_attention", "mixer": _latent(e, h), "mlp": mlp})
    return {"norm": {"eps": 1e-5}, "layers": layers}


def _lilevik(e, n, h, g, ff):
    """Groups of four: attention in chunks with sigmoid weights, lightning attention, attention through latents, chunks again;
    4 of 16 experts everywhere."""
    soft = {"heads": h, "kv_heads": g, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": 1024},
            "rot": {"base": 500000.0, "dims": 32, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
    m = e // 128
    light = {"heads": m, "dim": 128, "vdim": 128, "decay": [1.0 - 0.5 * 2.0 ** (-8.0 * (i + 1) / m) for i in range(m)]}
    kinds = [("attention", soft), ("lightning", light), ("latent_attention", _latent(e, h)), ("attention", soft)]
    routed = {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 16, "top": 4}}
    return {"norm": {"eps": 1e-5},
            "layers": [{"type": kinds[i % 4][0], "mixer": dict(kinds[i % 4][1]), "mlp": dict(routed)} for i in range(n)]}


def _goperax(e, n, h, g, ff):
    """Of four layers three have a state-space mixer, the fourth windowed attention whose values are its keys; the first
    feed-forward is dense, the others take 4 of 16 experts and a shared one; four copies of the stream."""
    scan = {"heads": e * 2 // 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}
    soft = {"heads": h, "kv_heads": g, "dim": 64, "vdim": 64, "scale": 0.125, "softcap": 30.0, "mask": {"size": 1024}}
    routed = {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 16, "top": 4}, "shared": {"ff": ff // 8}}
    layers = []
    for i in range(n):
        kind, mixer = ("attention", soft) if i % 4 == 3 else ("mamba2", scan)
        layers.append({"type": kind, "mixer": dict(mixer), "mlp": {"kind": "dense", "ff": ff} if i == 0 else routed})
    return {"streams": 4, "embedding": {"scale": 8.0}, "norm": {"eps": 1e-5}, "layers": layers}


# ---------------------------------------------------------------------- the weights and the requests
class Weights:
    """Tensors by name, drawn on the GPU from the seed and the name alone, in the dtype a weight file would hold them."""

    def __init__(self, case, seed, shapes=None):
        self.case, self.seed, self.shapes = case, seed, shapes
        self.dtype = DTYPES[case["dtype"]]

    def __getitem__(self, name):
        return self.drawn(name, self.shapes[name])

    def drawn(self, name, shape):
        gen = torch.Generator(device=DEVICE)
        gen.manual_seed(int.from_bytes(hashlib.blake2b(("%d/%s" % (self.seed, name)).encode(), digest_size=7).digest(), "little"))
        mean, std = self.spread(name, tuple(shape))
        t = torch.randn(tuple(shape), generator=gen, device=DEVICE, dtype=torch.float32 if len(shape) < 2 else self.dtype)
        t = t.mul_(std).add_(mean).to(self.dtype)
        if name.endswith(".mix") and ".hc" in name:       # a mixture of copies that keeps each
            t = t + torch.eye(shape[0], dtype=self.dtype, device=DEVICE)
        return t

    def spread(self, name, shape):
        """Mean and standard deviation: projections that keep the size of what goes through, what leads back to the stream
        smaller by the root of the number of sublayers (as deep models are initialised), decays and biases as such models
        have them, norm gains near one."""
        design, last = self.case["design"], name.rsplit(".", 1)[-1]
        shallow = (2 * self.case["layers"]) ** -0.5
        if design == "llama":
            if len(shape) < 2:
                return 1.0, 0.02
            if "embed_tokens" in name:
                return 0.0, 0.1 if self.case["vocab"] < 1000 else 0.5
            return 0.0, 0.02 * (shallow if "o_proj" in name or "down_proj" in name else 1.0)
        if design == "menerax" and (last in ("norm1", "norm2") or name in ("embed.norm", "final.norm")):
            return shallow - 1.0 if last in ("norm1", "norm2") else 0.0, 0.02     # stored as the distance from one
        if ".hc" in name:
            return (0.0, 0.05) if last == "mix" else (1.0 / shape[0] if last == "in" else 1.0, 0.05)
        if last == "A_log":
            return 0.5, 0.7
        if last in ("dt_bias", "w0"):
            return -3.0, 1.0
        if name.endswith("a2.b"):
            return 2.0, 1.0
        if last == "alpha":
            return 0.5, 0.05
        if "mu" in name.split(".")[-2:]:
            return 0.5, 0.2
        if last in ("conv", "canon1"):
            return 0.0, 0.4
        if last == "pb":
            return -4.0, 1.0
        if last in ("norm1b", "norm2b") or name.endswith(("left.out", "right.out")):
            return shallow, 0.05 * shallow
        if "norm" in last or last == "D" or last.startswith("ls"):
            return 1.0, 0.05
        if "norm1b" in name or "norm2b" in name:
            return 0.0, 0.1 * shallow
        if len(shape) < 2 or last in ("b", "u", "sink", "act"):
            return 0.0, 0.3
        if name == "embed":
            return 0.0, 0.1 if design == "goperax" else 0.5
        if ".mlp.e" in name and last == "down":           # small enough that a near tie of a router, which rounding decides, stays so
            shallow *= 0.25
        return 0.0, shape[-1] ** -0.5 * (shallow if last in ("o", "down") else 1.0)


def lengths_of(case):
    """The prompts' lengths: uneven steps from the shortest to the longest, the same for every seed."""
    n, span = case["sequences"], case["longest"] - case["shortest"]
    return [case["longest"] - int(span * ((i * 0.6180339887) % 1.0)) for i in range(n)]


def requests_of(case, seed):
    """(prompts, fed, uniforms): the prompts' token ids, and per decode step the token that each sequence is fed and the number
    that its sampling takes."""
    rng = np.random.default_rng([17, seed])
    prompts = [[int(t) for t in rng.integers(0, case["vocab"], size=n)] for n in lengths_of(case)]
    fed = [[int(t) for t in rng.integers(0, case["vocab"], size=case["sequences"])] for _ in range(case["new"])]
    uniforms = [[float(u) for u in rng.random(case["sequences"])] for _ in range(case["new"])]
    return prompts, fed, uniforms


# ---------------------------------------------------------------------- a pass
def prepare(case, seed):
    _, spec = rbitnet_amd.load_config(config_of(case))
    shapes = {name: ts.shape for name, ts in expected_tensors(spec).items()}
    prompts, fed, uniforms = requests_of(case, seed)
    room = sum((len(p) + case["new"] + 63) // 64 * 64 for p in prompts)
    engine = rbitnet_amd.Engine.from_spec(spec, Weights(case, seed, shapes), dtype=case["dtype"], max_tokens=room,
                                          max_batch=case["sequences"], max_seq_len=max(len(p) for p in prompts) + case["new"],
                                          device=DEVICE)
    return {"engine": engine, "prompts": prompts, "fed": fed, "uniforms": uniforms, "piece": case["piece"], "want": case["want"],
            "exact_choice": case["dtype"] == "float32",
            "temperatures": [case["temperature"]] * case["sequences"] if case["temperature"] > 0 else None}


def run(state):
    engine, prompts, piece = state["engine"], state["prompts"], state["piece"]
    slots = [engine.alloc_slot() for _ in prompts]
    out = {"prompt": [], "decoded": []}
    if not piece:
        out["prompt"].append(engine.step(list(zip(slots, prompts)), state["want"]))
    else:                                                 # a step asks for logits where a prompt ends
        for at in range(0, max(len(p) for p in prompts), piece):
            part = [(s, p[at:at + piece], at + piece >= len(p)) for s, p in zip(slots, prompts) if len(p) > at]
            want = "all" if state["want"] == "all" else [[len(t) - 1] if ends else [] for _, t, ends in part]
            logits = engine.step([(s, t) for s, t, _ in part], want)
            if logits.shape[0]:
                out["prompt"].append(logits)
    chosen = []
    for fed, uniforms in zip(state["fed"], state["uniforms"]):
        sampled = state["temperatures"] is not None
        chosen.append(engine.decode_step(slots, fed, state["temperatures"], uniforms if sampled else None))
        out["decoded"].append(engine.last_decode_logits.clone())
    if chosen and state["exact_choice"]:                  # in bfloat16 which of two nearly equal logits leads is rounding's to say
        out["chosen"] = np.array(chosen, dtype=np.int64)
    for slot in slots:
        engine.free_slot(slot)
    return out


def tolerance(case):
    """About four times the error against 64 bits that was measured for each design (for Llama three times: 0.011 at 32 layers;
    0.0042 Bagonex, 0.0041 Menerax; where routers choose, a near tie that falls the other way makes up to
    0.02; float32 4e-6).  Tokens are compared in float32 alone."""
    if case["dtype"] == "float32":
        return {"rel": 1.5e-5, "differ": 0.01}
    return {"rel": {"bagonex": 0.015, "menerax": 0.017, "lilevik": 0.02}.get(case["design"], 0.03)}


# ---------------------------------------------------------------------- what a pass cannot do without
def _mixing(config):
    """Per layer: [(heads, numbers of a score and an output, numbers kept per token, reach)] of its attention, and the numbers
    of its recurrent states."""
    out = []
    if "architectures" in config:
        d = config["head_dim"]
        one = ([(config["num_attention_heads"], 2 * d, 2 * config["num_key_value_heads"] * d, None)], 0)
        return [one] * config["num_hidden_layers"]
    for layer in config["layers"]:
        attention, states = [], 0
        kind, m = layer["type"], layer["mixer"]
        for kind, m in ([(layer["type"], layer["mixer"])] if kind != "parallel" else [("attention", m["left"]), ("state", m["right"])]):
            if kind == "latent_attention":
                kept = m["kv_rank"] + m.get("rot_dim", 0)
                attention.append((m["heads"], kept + m["kv_rank"], kept, None))
            elif kind == "attention":
                kept = m["kv_heads"] * (m["dim"] + (m["vdim"] if config["architecture"] != "Goperax" else 0))
                attention.append((m["heads"], m["dim"] + m["vdim"], kept, (m.get("mask") or {}).get("size")))
            else:
                states += m["heads"] * m.get("vdim", m.get("dim")) * m.get("state", m.get("dim"))
        out.append((attention, states))
    return out


def work(case):
    config = config_of(case)
    _, spec = rbitnet_amd.load_config(config)
    size = 2 if case["dtype"] == "bfloat16" else 4
    lengths = lengths_of(case)
    tied = "head" not in expected_tensors(spec) and "lm_head.weight" not in expected_tensors(spec)
    dense = experts = head = 0
    for name, ts in expected_tensors(spec).items():
        n = math.prod(ts.shape)
        embed = name in ("embed", "model.embed_tokens.weight")
        if name in ("head", "lm_head.weight") or (embed and tied):
            head += n
        elif embed:
            continue
        elif ".mlp.e" in name:
            experts += n
        else:
            dense += n
    n_experts, top = 1, 1
    for layer in config.get("layers", []):
        if layer["mlp"]["kind"] == "moe":
            n_experts, top = layer["mlp"]["router"]["experts"], layer["mlp"]["router"]["top"]
    piece = case["piece"] or max(lengths)
    steps = [[(at, min(piece, n - at)) for n in lengths if n > at] for at in range(0, max(lengths), piece)]
    steps += [[(n + j, 1) for n in lengths] for j in range(case["new"])]
    rows = [sum(n for _, n in s) if case["want"] == "all" else 0 for s in steps]
    for j in range(len(steps)):
        if j >= len(steps) - case["new"] or (case["want"] == "last" and j == len(steps) - case["new"] - 1):
            rows[j] = len(lengths)
    nbytes = flops = 0.0
    for step, asked in zip(steps, rows):
        tokens = sum(n for _, n in step)
        touched = 1.0 - (1.0 - top / n_experts) ** tokens
        nbytes += size * (dense + experts * touched + (head if asked else 0) + tokens * case["width"]) + 4.0 * asked * case["vocab"]
        flops += 2.0 * (tokens * (dense + experts * top / n_experts) + asked * head)
        for attention, states in _mixing(config):
            nbytes += 8.0 * states * len(step)            # read and written, 32 bits
            flops += 6.0 * states * tokens
            for heads, numbers, kept, reach in attention:
                for past, n in step:
                    seen = past + n if reach is None else min(past + n, reach + n)
                    nbytes += size * kept * seen
                    pairs = n * past + n * (n + 1) / 2.0 if reach is None else sum(min(past + i + 1, reach) for i in range(n))
                    flops += 2.0 * heads * numbers * pairs
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------- the same in 64 bits, from the equations
def exact(case, seed):
    config, w = config_of(case), Weights(case, seed)
    prompts, fed, _ = requests_of(case, seed)
    texts = [p + [step[i] for step in fed] for i, p in enumerate(prompts)]
    longest = max(len(t) for t in texts)
    ids = torch.zeros(len(texts), longest, dtype=torch.long, device=DEVICE)
    for i, t in enumerate(texts):                         # what lies behind a text's end changes nothing before it
        ids[i, :len(t)] = torch.tensor(t, device=DEVICE)
    stream = {"llama": _exact_llama, "bagonex": _exact_bagonex, "tigutar": _exact_tigutar, "menerax": _exact_menerax,
              "lilevik": _exact_lilevik, "goperax": _exact_goperax}[case["design"]]
    x, to_logits = stream(config, lambda name, *shape: w.drawn(name, shape).to(F64), ids)

    def logits(places):
        seq, pos = (torch.tensor(v, device=DEVICE) for v in zip(*places))
        return to_logits(x[seq, pos]).to(torch.float32 if len(places) * case["vocab"] > 5e7 else F64)

    piece = case["piece"] or max(len(p) for p in prompts)
    out = {"prompt": [], "decoded": []}
    for at in range(0, max(len(p) for p in prompts), piece):
        places = []
        for i, p in enumerate(prompts):
            if len(p) > at:
                end = min(len(p), at + piece)
                places += [(i, j) for j in range(at, end)] if case["want"] == "all" else [(i, end - 1)] if end == len(p) else []
        if places:
            out["prompt"].append(logits(places))
    for j in range(case["new"]):
        out["decoded"].append(logits([(i, len(p) + j) for i, p in enumerate(prompts)]))
    if case["new"] and case["dtype"] == "float32":
        out["chosen"] = None                              # whole numbers: compared with themselves
    return out


def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, gain, bias, eps):
    return _unit(x - x.mean(-1, keepdim=True), eps) * gain + bias


def _silu(x):
    return x * torch.sigmoid(x)


def _softplus(x):
    return x.clamp(min=0) + torch.log1p(torch.exp(-x.abs()))


def _before(x, back):
    """The row `back` tokens earlier, zeros before the start: x [B, T, C]."""
    return x if back == 0 else torch.cat([torch.zeros_like(x[:, :back]), x[:, :-back]], 1) if x.shape[1] > back else torch.zeros_like(x)


def _conv(x, taps):
    return sum(_before(x, d) * taps[:, taps.shape[1] - 1 - d] for d in range(taps.shape[1]))


def _rotated(x, freq, factor=1.0, pairs=False):
    """x [B, T, H, D]; of the first 2 len(freq) numbers of a head, i and i + len(freq) (or 2i and 2i + 1) turn together."""
    half = len(freq)
    a = torch.arange(x.shape[1], dtype=F64, device=x.device)[:, None] * torch.tensor(freq, dtype=F64, device=x.device)
    c, s = factor * torch.cos(a)[:, None, :], factor * torch.sin(a)[:, None, :]
    if pairs:
        u, v = x[..., 0:2 * half:2], x[..., 1:2 * half:2]
        turned = torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)
    else:
        u, v = x[..., :half], x[..., half:2 * half]
        turned = torch.cat([u * c - v * s, v * c + u * s], -1)
    return torch.cat([turned, x[..., 2 * half:]], -1)


def _frequencies(dims, base, scaling=None):
    """base^(-2i / dims); with low and high factors, wavelengths beyond original / low are stretched, those below
    original / high stay, and a blend lies between."""
    out = []
    for i in range(dims // 2):
        f = base ** (-2.0 * i / dims)
        if scaling:
            s = (scaling["original"] * f / (2.0 * math.pi) - scaling["low"]) / (scaling["high"] - scaling["low"])
            s = min(max(s, 0.0), 1.0)
            f = (1.0 - s) * f / scaling["factor"] + s * f
        out.append(f)
    return out


def _attend(q, k, v, scale, reach=None, chunk=None, keep_first=0, softcap=None, sink=None, one=False, sigmoid_bias=None):
    """q [B, T, H, D], k and v [B, T, G, .] -> [B, T, H, Dv], a few heads of a few sequences at a time."""
    b, t, h, _ = q.shape
    r = h // k.shape[2]
    i, j = torch.arange(t, device=q.device)[:, None], torch.arange(t, device=q.device)[None, :]
    seen = j <= i
    if reach is not None:
        seen = seen & ((i - j < reach) | (j < keep_first))
    if chunk is not None:
        seen = seen & (i // chunk == j // chunk)
    out = torch.empty(b, t, h, v.shape[-1], dtype=q.dtype, device=q.device)
    many = max(1, int(3e8 // (t * t * r)))
    for g in range(k.shape[2]):
        for at in range(0, b, many):
            qq = q[at:at + many, :, g * r:(g + 1) * r].transpose(1, 2)                     # [b, r, T, D]
            kk, vv = k[at:at + many, :, g], v[at:at + many, :, g]
            n = qq.shape[0]
            s = torch.bmm(qq.reshape(n, r * t, -1), kk.transpose(1, 2).contiguous()).view(n, r, t, t).mul_(scale)
            if softcap is not None:
                s = s.div_(softcap).tanh_().mul_(softcap)
            if sigmoid_bias is not None:
                s = torch.sigmoid(s + sigmoid_bias[g * r:(g + 1) * r].view(1, r, 1, 1)).masked_fill_(~seen, 0.0)
            else:
                s = s.masked_fill_(~seen, -math.inf)
                top = s.amax(-1, keepdim=True)
                extra = None
                if one:
                    extra = torch.zeros(1, 1, 1, 1, dtype=F64, device=q.device)
                elif sink is not None:
                    extra = sink[g * r:(g + 1) * r].view(1, r, 1, 1)
                if extra is not None:
                    top = torch.maximum(top, extra)
                s = s.sub_(top).exp_()
                total = s.sum(-1, keepdim=True)
                s = s.div_(total if extra is None else total + torch.exp(extra - top))
            o = torch.bmm(s.reshape(n, r * t, t), vv.contiguous()).view(n, r, t, -1)
            out[at:at + many, :, g * r:(g + 1) * r] = o.transpose(1, 2)
    return out


def _experts(h, w, prefix, mlp, e, route, act, names, shared=False):
    """Sum over a token's chosen experts; route(h) -> (chosen, weights); `names`: the matrices in front of the activation."""
    shape, h = h.shape, h.reshape(-1, e)
    chosen, weights, on_input = route(h)
    out, ff = torch.zeros_like(h), mlp["expert"]["ff"]
    for x in range(mlp["router"]["experts"]):
        t, at = torch.nonzero(chosen == x, as_tuple=True)
        if len(t):
            p = "%se%d." % (prefix, x)
            weight = weights[t, at][:, None]
            z = h[t] * weight if on_input else h[t]
            y = act(*[z @ w(p + n, ff, e).T for n in names]) @ w(p + "down", e, ff).T
            out.index_add_(0, t, y if on_input else y * weight)
    return out.view(shape)


def _heads(x, n):
    return x.view(*x.shape[:2], n, -1)


def _exact_llama(c, w, ids):
    e, h, g, d, ff, eps = (c[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim", "intermediate_size", "rms_norm_eps"))
    scaling = c.get("rope_scaling")
    if scaling:
        scaling = {"factor": scaling["factor"], "low": scaling["low_freq_factor"], "high": scaling["high_freq_factor"],
                   "original": scaling["original_max_position_embeddings"]}
    freq = _frequencies(d, c["rope_theta"], scaling)
    x = w("model.embed_tokens.weight", c["vocab_size"], e)[ids]
    for i in range(c["num_hidden_layers"]):
        p = "model.layers.%d." % i
        n = _unit(x, eps) * w(p + "input_layernorm.weight", e)
        q, k, v = (_heads(n @ w(p + "self_attn.%s_proj.weight" % s, m * d, e).T, m) for s, m in (("q", h), ("k", g), ("v", g)))
        o = _attend(_rotated(q, freq), _rotated(k, freq), v, d ** -0.5)
        x = x + o.flatten(2) @ w(p + "self_attn.o_proj.weight", e, h * d).T
        n = _unit(x, eps) * w(p + "post_attention_layernorm.weight", e)
        a = _silu(n @ w(p + "mlp.gate_proj.weight", ff, e).T) * (n @ w(p + "mlp.up_proj.weight", ff, e).T)
        x = x + a @ w(p + "mlp.down_proj.weight", e, ff).T
    out = w("model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight", c["vocab_size"], e)
    gain = w("model.norm.weight", e)
    return x, lambda rows: (_unit(rows, eps) * gain) @ out.T


def _delta_rule(q, k, v, g, beta):
    """q, k [B, T, H, dk], v [B, T, H, dv], g [B, T, H, dk or 1], beta [B, T, H]:
    S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q."""
    b, t, h, dk = q.shape
    s = torch.zeros(b, h, dk, v.shape[-1], dtype=F64, device=q.device)
    out = torch.empty(b, t, h, v.shape[-1], dtype=F64, device=q.device)
    for i in range(t):
        s *= g[:, i, :, :, None]
        u = beta[:, i, :, None] * (v[:, i] - torch.matmul(k[:, i, :, None, :], s)[:, :, 0])
        s += k[:, i, :, :, None] * u[:, :, None, :]
        out[:, i] = torch.matmul(q[:, i, :, None, :], s)[:, :, 0]
    return out


def _decaying_sum(q, k, v, keep, bonus=None):
    """S <- keep S + k v^T, o = S^T q; with `bonus` [H, dk] o = (S before the token + diag(bonus) k v^T)^T q."""
    b, t, h, dk = q.shape
    s = torch.zeros(b, h, dk, v.shape[-1], dtype=F64, device=q.device)
    out = torch.empty(b, t, h, v.shape[-1], dtype=F64, device=q.device)
    for i in range(t):
        if bonus is not None:
            own = (q[:, i] * bonus * k[:, i]).sum(-1, keepdim=True)
            out[:, i] = torch.matmul(q[:, i, :, None, :], s)[:, :, 0] + own * v[:, i]
        s *= keep[:, i, :, :, None]
        s += k[:, i, :, :, None] * v[:, i, :, None, :]
        if bonus is None:
            out[:, i] = torch.matmul(q[:, i, :, None, :], s)[:, :, 0]
    return out


def _unit_heads(q, k, dim):
    return (q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * dim ** -0.5, k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6))


def _exact_bagonex(c, w, ids):
    e, s, eps = c["width"], c["streams"], c["norm"]["eps"]
    xs = [w("embed", c["vocab"], e)[ids]] * s
    latents = {}
    for i, layer in enumerate(c["layers"]):
        m, ff = layer["mixer"], layer["mlp"]["ff"]
        for p in (1, 2):
            l = "l%d." % i
            reads = w(l + "hc%d.in" % p, s)
            n = _layer_norm(sum(reads[j] * xs[j] for j in range(s)), w(l + "norm%d" % p, e), w(l + "norm%d.b" % p, e), eps)
            if p == 1:
                n = n + _conv(n, w(l + "canon1", e, c["canon"]["taps"]))
                mix = lambda name, *shape: w(l + "mix." + name, *shape)
                h, dim, vdim = m["heads"], m["dim"], m["vdim"]
                if layer["type"] == "channel_delta":
                    q, k, v = (_heads(_silu(_conv(n @ mix(a, h * size, e).T, mix(a + ".conv", h * size, m["conv"]))), h)
                               for a, size in (("q", dim), ("k", dim), ("v", vdim)))
                    q, k = _unit_heads(q, k, dim)
                    a = _heads((n @ mix("a1", m["decay_rank"], e).T) @ mix("a2", h * dim, m["decay_rank"]).T + mix("dt_bias", h * dim), h)
                    g = torch.exp(-torch.exp(mix("A_log", h))[:, None] * _softplus(a))
                    o = _delta_rule(q, k, v, g, torch.sigmoid(n @ mix("b", h, e).T))
                    gate = torch.sigmoid((n @ mix("g1", m["gate_rank"], e).T) @ mix("g2", h * vdim, m["gate_rank"]).T)
                    o = (_unit(o, eps) * mix("norm", vdim)).flatten(2) * gate
                else:
                    rank, src = m["kv_rank"], m.get("kv_from", i)
                    if src == i:
                        latents[i] = _unit(n @ mix("dkv", rank, e).T, eps) * mix("dkv.norm", rank)
                    q = _heads((_unit(n @ mix("dq", m["q_rank"], e).T, eps) * mix("dq.norm", m["q_rank"])) @ mix("uq", h * dim, m["q_rank"]).T, h)
                    k, v = _heads(latents[src] @ mix("uk", h * dim, rank).T, h), _heads(latents[src] @ mix("uv", h * vdim, rank).T, h)
                    o = _attend(q, k, v, m["scale"], sink=mix("sink", h)).flatten(2)
                y = o @ mix("o", e, h * vdim).T
            else:
                a = w(l + "mlp.act", 2)
                z = n @ w(l + "mlp.up", ff, e).T
                z = torch.where(z > 0, _softplus(a[0]) * z * z, (0.5 + _softplus(a[1])) * (torch.expm1(z.clamp(max=0)) - z)) + z / 2
                y = z @ w(l + "mlp.down", e, ff).T
            y = y * w(l + "ls%d" % p, e)
            mix, out = _mixture(w, l + "hc%d." % p, s)
            xs = [sum(mix[a, j] * xs[a] for a in range(s)) + out[j] * y for j in range(s)]
    gain, bias, head, cap = w("final.norm", e), w("final.norm.b", e), w("head", c["vocab"], e), c["logit_softcap"]
    return sum(xs), lambda rows: cap * torch.tanh(_layer_norm(rows, gain, bias, eps) @ head.T / cap)


def _mixture(w, prefix, s):
    return w(prefix + "mix", s, s), w(prefix + "out", s)


def _exact_tigutar(c, w, ids):
    e, eps = c["width"], c["norm"]["eps"]
    x = w("embed", c["vocab"], e)[ids]
    kept = {}

    def soft(n, mix, m, i, gated):
        h, g, dim, vdim = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        freq, src = _frequencies(m["rot"]["dims"], m["rot"]["base"]), m.get("kv_from", i)
        q = _rotated(_heads(n @ mix("q", h * dim, e).T, h), freq)
        k, v = kept[src] if src != i else (_rotated(_heads(n @ mix("k", g * dim, e).T, g), freq), _heads(n @ mix("v", g * vdim, e).T, g))
        if gated:
            kept[i] = k, v
        o = _attend(q, k, v, m["scale"], reach=(m.get("mask") or {}).get("size"), sink=mix("sink", h) if gated else None)
        if gated:
            o = o * torch.sigmoid(n @ mix("g", h, e).T)[..., None]
        return o.flatten(2) @ mix("o", e, h * vdim).T

    for i, layer in enumerate(c["layers"]):
        l, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
        mix = lambda name, *shape: w(l + "mix." + name, *shape)
        n = _layer_norm(x, w(l + "norm1", e), w(l + "norm1.b", e), eps)
        if layer["type"] == "attention":
            y = soft(n, mix, m, i, True)
        elif layer["type"] == "delta":
            h, g, dim, vdim = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            q, k, v = (_heads(_silu(_conv(n @ mix(a, o * size, e).T, mix(a + ".conv", o * size, m["conv"]))), o)
                       for a, o, size in (("q", g, dim), ("k", g, dim), ("v", h, vdim)))
            q, k = (a.repeat_interleave(h // g, 2) for a in _unit_heads(q, k, dim))
            decay = torch.exp(-torch.exp(mix("A_log", h)) * _softplus(n @ mix("a", h, e).T + mix("dt_bias", h)))
            o = _delta_rule(q, k, v, decay[..., None], torch.sigmoid(n @ mix("b", h, e).T))
            o = (_unit(o, eps) * mix("norm", vdim)).flatten(2) * _silu(n @ mix("g", h * vdim, e).T)
            y = o @ mix("o", e, h * vdim).T
        else:
            r = m["right"]
            h, dim, vdim = r["heads"], r["dim"], r["vdim"]
            a = soft(n, lambda name, *shape: mix("left." + name, *shape), m["left"], i, False)
            q, k, v = (_heads(n @ mix("right." + s, h * size, e).T, h) for s, size in (("q", dim), ("k", dim), ("v", vdim)))
            z = (n @ mix("right.a1", r["decay_rank"], e).T) @ mix("right.a2", h * dim, r["decay_rank"]).T + mix("right.a2.b", h * dim)
            keep = _heads(torch.sigmoid(z).pow(1.0 / r["tau"]), h)
            o = _unit(_decaying_sum(q * dim ** -0.5, k, v, keep), eps) * mix("right.norm", vdim)
            b = (o.flatten(2) * _silu(n @ mix("right.g", h * vdim, e).T)) @ mix("right.o", e, h * vdim).T
            y = 0.5 * (_unit(a, eps) * mix("left.out", e) + _unit(b, eps) * mix("right.out", e))
        p = l + "mlp."
        if mlp["kind"] == "dense":
            z = _silu(n @ w(p + "gate", mlp["ff"], e).T) * (n @ w(p + "up", mlp["ff"], e).T)
            y = y + z @ w(p + "down", e, mlp["ff"]).T
        else:
            limit = mlp["expert"]["limit"]

            def route(rows):
                best = torch.sigmoid(rows @ w(p + "router", mlp["router"]["experts"], e).T).topk(mlp["router"]["top"], -1)
                return best.indices, best.values, True

            def act(a, b):
                a = a.clamp(max=limit)
                return a * torch.sigmoid(1.702 * a) * (b.clamp(-limit, limit) + 1)
            y = y + _experts(n, w, p, mlp, e, route, act, ("gate", "up"))
        x = x + c["residual_mult"] * y
    gain, bias, head = w("final.norm", e), w("final.norm.b", e), w("head", c["vocab"], e)
    return x, lambda rows: _layer_norm(rows, gain, bias, eps) @ head.T


def _latent_heads(n, mix, m, e, eps, freq, factor):
    h, dim, rot, vdim, rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
    q = _heads((_unit(n @ mix("dq", m["q_rank"], e).T, eps) * mix("dq.norm", m["q_rank"])) @ mix("uq", h * (dim + rot), m["q_rank"]).T, h)
    down = n @ mix("dkv", rank + rot, e).T
    latent = _unit(down[..., :rank], eps) * mix("dkv.norm", rank)
    q = torch.cat([q[..., :dim], _rotated(q[..., dim:], freq, factor, True)], -1)
    shared = _rotated(down[..., None, rank:], freq, factor, True).expand(-1, -1, h, -1)
    k = torch.cat([_heads(latent @ mix("uk", h * dim, rank).T, h), shared], -1)
    return _attend(q, k, _heads(latent @ mix("uv", h * vdim, rank).T, h), m["scale"])


def _exact_menerax(c, w, ids):
    e, eps = c["width"], c["norm"]["eps"]
    normed = lambda x, name: _unit(x, eps) * (1.0 + w(name, e))
    x = normed(w("embed", c["vocab"], e)[ids], "embed.norm")
    for i, layer in enumerate(c["layers"]):
        l, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
        mix = lambda name, *shape: w(l + "mix." + name, *shape)
        if layer["type"] == "latent_attention":
            h, vdim = m["heads"], m["vdim"]
            o = _latent_heads(x, mix, m, e, eps, _frequencies(m["rot_dim"], m["rot"]["base"]), 1.0)
            y = (o * torch.sigmoid(x @ mix("g", h, e).T)[..., None]).flatten(2) @ mix("o", e, h * vdim).T
        else:
            a, b = m["left"], m["right"]
            h, g, dim = a["heads"], a["kv_heads"], a["dim"]
            q, k, v = (_heads(_conv(x @ mix("left." + s, o * dim, e).T + mix("left.%s.b" % s, o * dim), mix("left.%s.conv" % s, o * dim, a["conv"])), o)
                       for s, o in (("q", h), ("k", g), ("v", g)))
            freq = _frequencies(a["rot"]["dims"], a["rot"]["base"], a["rot"]["scaling"])
            q, k = (_rotated(_unit(t, eps) * mix("left.%s.norm" % s, dim), freq) for s, t in (("q", q), ("k", k)))
            o = _attend(q, k, v, a["scale"], reach=a["mask"]["size"], keep_first=a["mask"]["keep_first"], softcap=a["softcap"]).flatten(2)
            left = (o * torch.sigmoid(x @ mix("left.g", h * dim, e).T)) @ mix("left.o", e, h * dim).T
            h, dim, rank = b["heads"], b["dim"], b["decay_rank"]
            mixed = {s: x + (_before(x, 1) - x) * mix("right.mu." + s, e) for s in "rkvgw"}
            r, k, v = (_heads(mixed[s] @ mix("right." + s, h * dim, e).T, h) for s in "rkv")
            z = torch.tanh(mixed["w"] @ mix("right.w1", rank, e).T) @ mix("right.w2", h * dim, rank).T + mix("right.w0", h * dim)
            o = _decaying_sum(r, k, v, _heads(torch.exp(-torch.exp(z)), h), bonus=mix("right.u", h, dim))
            o = _unit(o, eps).flatten(2) * mix("right.norm", h * dim) * _silu(mixed["g"] @ mix("right.g", h * dim, e).T)
            y = m["left_scale"] * left + m["right_scale"] * (o @ mix("right.o", e, h * dim).T)
        x = x + normed(y, l + "norm1")
        ff, limit = mlp["ff"], mlp["limit"]
        a = (x @ w(l + "mlp.gate", ff, e).T).clamp(max=limit)
        b = (x @ w(l + "mlp.up", ff, e).T).clamp(-limit, limit)
        x = x + normed((a * torch.sigmoid(1.702 * a) * (b + 1)) @ w(l + "mlp.down", e, ff).T, l + "norm2")
    head, gain = w("head", c["vocab"], e), 1.0 + w("final.norm", e)
    return x, lambda rows: (_unit(rows, eps) * gain) @ head.T


def _ramped(dims, base, scaling):
    """Frequencies of pairs that turn `fast` times over `original` positions stay, those that turn `slow` times are divided by
    the factor, with a ramp over the pair's index between; and the factor on cosine and sine."""
    index = lambda turns: dims * math.log(scaling["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(index(scaling["fast"])), 0), min(math.ceil(index(scaling["slow"])), dims - 1)
    out = []
    for i in range(dims // 2):
        f, r = base ** (-2.0 * i / dims), min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0)
        out.append(f / scaling["factor"] * r + f * (1.0 - r))
    return out, 0.1 * math.log(scaling["factor"]) + 1.0


def _exact_lilevik(c, w, ids):
    e, eps = c["width"], c["norm"]["eps"]
    norm = lambda x, name: torch.tanh(w(name + ".alpha") * x) * w(name, e) + w(name + ".b", e)
    embed = w("embed", c["vocab"], e)
    x = embed[ids]
    for i, layer in enumerate(c["layers"]):
        l, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
        mix = lambda name, *shape: w(l + "mix." + name, *shape)
        n, h, vdim, dim = norm(x, l + "norm1"), m["heads"], m["vdim"], m["dim"]
        if layer["type"] == "latent_attention":
            o = _latent_heads(n, mix, m, e, eps, _frequencies(m["rot_dim"], m["rot"]["base"]), 1.0).flatten(2)
        elif layer["type"] == "attention":
            g = m["kv_heads"]
            q = _heads(_unit(n @ mix("q", h * dim, e).T, eps) * mix("q.norm", h * dim), h)
            k = _heads(_unit(n @ mix("k", g * dim, e).T, eps) * mix("k.norm", g * dim), g)
            v = _unit(_heads(n @ mix("v", g * vdim, e).T, g), eps)
            freq, factor = _ramped(m["rot"]["dims"], m["rot"]["base"], m["rot"]["scaling"])
            o = _attend(_rotated(q, freq, factor, True), _rotated(k, freq, factor, True), v, m["scale"], chunk=m["mask"]["size"],
                        sigmoid_bias=mix("pb", h)).flatten(2)
        else:
            q, k, v = (_heads(_silu(n @ mix(s, h * size, e).T), h) for s, size in (("q", dim), ("k", dim), ("v", vdim)))
            keep = torch.tensor(m["decay"], dtype=F64, device=x.device).view(1, 1, h, 1).expand(*q.shape[:2], h, 1)
            o = _unit(_decaying_sum(q, k, v, keep).flatten(2), eps) * mix("norm", h * vdim) * torch.sigmoid(n @ mix("g", h * vdim, e).T)
        x = x + norm(o @ mix("o", e, h * vdim).T, l + "norm1b")

        def route(rows):
            count = mlp["router"]["experts"]
            best = (rows @ w(l + "mlp.router", count, e).T + w(l + "mlp.router.b", count)).topk(mlp["router"]["top"], -1)
            return best.indices, torch.softmax(best.values, -1), False
        y = _experts(norm(x, l + "norm2"), w, l + "mlp.", mlp, e, route, lambda a, b: _silu(a) * b, ("gate", "up"))
        x = x + norm(y, l + "norm2b")
    final = [w("final.norm.alpha"), w("final.norm", e), w("final.norm.b", e)]
    return x, lambda rows: (torch.tanh(final[0] * rows) * final[1] + final[2]) @ embed.T


def _exact_goperax(c, w, ids):
    e, s, eps = c["width"], c["streams"], c["norm"]["eps"]
    embed = w("embed", c["vocab"], e)
    angle = torch.arange(ids.shape[1], dtype=F64, device=ids.device)[:, None] * \
        10000.0 ** (-2.0 * torch.arange(e // 2, dtype=F64, device=ids.device) / e)
    waves = torch.stack([torch.sin(angle), torch.cos(angle)], -1).flatten(-2)
    xs = [embed[ids] * c["embedding"]["scale"] + waves] * s
    square = lambda z: z.clamp(min=0) ** 2
    for i, layer in enumerate(c["layers"]):
        l, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
        for p in (1, 2):
            reads = w(l + "hc%d.in" % p, s)
            n = _unit(sum(reads[j] * xs[j] for j in range(s)), eps) * w(l + "norm%d" % p, e)
            mix = lambda name, *shape: w(l + "mix." + name, *shape)
            if p == 2 and mlp["kind"] == "dense":
                y = square(n @ w(l + "mlp.up", mlp["ff"], e).T) @ w(l + "mlp.down", e, mlp["ff"]).T
            elif p == 2:
                def route(rows):
                    best = torch.softmax(rows @ w(l + "mlp.router", mlp["router"]["experts"], e).T, -1).topk(mlp["router"]["top"], -1)
                    return best.indices, best.values / best.values.sum(-1, keepdim=True), False
                y = _experts(n, w, l + "mlp.", mlp, e, route, square, ("up",))
                ff = mlp["shared"]["ff"]
                y = y + square(n @ w(l + "mlp.shared.up", ff, e).T) @ w(l + "mlp.shared.down", e, ff).T
            elif layer["type"] == "attention":
                h, g, dim = m["heads"], m["kv_heads"], m["dim"]
                q, k = _heads(n @ mix("q", h * dim, e).T, h), _heads(n @ mix("k", g * dim, e).T, g)
                o = _attend(q, k, k, m["scale"], reach=m["mask"]["size"], softcap=m["softcap"], one=True)
                y = o.flatten(2) @ mix("o", e, h * dim).T
            else:
                h, vdim, state, g = m["heads"], m["vdim"], m["state"], m["groups"]
                inner, keys = h * vdim, g * state
                z, xbc, dt = torch.split(n @ mix("in", 2 * inner + 2 * keys + h, e).T, [inner, inner + 2 * keys, h], -1)
                xbc = _silu(_conv(xbc, mix("conv", inner + 2 * keys, m["conv"])) + mix("conv.b", inner + 2 * keys))
                v, b, q = torch.split(xbc, [inner, keys, keys], -1)
                dt = _softplus(dt + mix("dt_bias", h))
                v = _heads(v, h)
                b, q = (_heads(t, g).repeat_interleave(h // g, 2) for t in (b, q))
                keep = torch.exp(-torch.exp(mix("A_log", h)) * dt)
                o = _decaying_sum(q, b * dt[..., None], v, keep[..., None]) + mix("D", h)[:, None] * v
                o = _unit(_heads(o.flatten(2) * _silu(z), m["norm_groups"]), eps).flatten(2) * mix("norm", inner)
                y = o @ mix("o", e, inner).T
            mix, out = _mixture(w, l + "hc%d." % p, s)
            xs = [sum(mix[a, j] * xs[a] for a in range(s)) + out[j] * y for j in range(s)]
    gain = w("final.norm", e)
    return sum(xs), lambda rows: (_unit(rows, eps) * gain) @ embed.T
