"""The work that a user of this framework has it do, as cases that can be timed and compared.

Two families of models, through the entry points that the command line, the server and the batch scheduler call:

* quantised Llama files (model.load_llama_model): a prompt (prefill), a conversation's turn (the new message behind a cached
  context, then a greedy or sampled reply), decode streams side by side (forward_batch);
* layer-stack models (stack.load_stack_model, Ganidra and Pabalix): a prompt, and requests of ragged lengths that are prefilled
  together and then decoded side by side.

Weights, tokens and random numbers come from the seed.  The shapes are the tiers nano, mini and goldie, and "wide": the largest
tier's layer width on four layers (a whole model of it does not load in the time that a case may take).
"""
from __future__ import annotations

import math
import random
from typing import Dict, List, Tuple

import numpy as np
import torch

from nanollama_amd.designs import DESIGNS
from nanollama_amd.gguf import GGUFMetadata, GGUFTensorInfo
from nanollama_amd.model import load_llama_model
from nanollama_amd.stack import load_stack_model
from nanollama_amd.synth_stack import ganidra_config, ganidra_layer, ganidra_shapes, pabalix_config, pabalix_layer, pabalix_shapes

# name: layers, width, query heads, key / value heads, vocabulary, feed-forward
TIERS = {"nano": (13, 576, 9, 9, 32000, 1536), "mini": (20, 768, 12, 3, 32000, 2048), "goldie": (28, 1536, 24, 6, 48000, 4096),
         "wide": (4, 4096, 64, 16, 32000, 11008)}
HEAD = 64
SEQ_LEN = 2048
EPS = 1e-5
# bytes and values of a block, ggml's type number
BLOCKS = {"f32": (4, 1, 0), "f16": (64, 32, 1), "q4_0": (18, 32, 2), "q5_0": (22, 32, 6), "q8_0": (34, 32, 8), "q4_k": (144, 256, 12), "q6_k": (210, 256, 14)}


# ---------------------------------------------------------------- the cases

def listed() -> List[dict]:
    return [
        # --- quantised Llama files ---
        # a chat line to the smallest tier: the smallest call, a handful of tokens against every weight once
        dict(name="nano-q8-line", family="llama", kind="prompt", tier="nano", wtype="q8_0", context=0, tokens=24),
        # one request to the smallest tier as the command line makes it with temperature 0
        dict(name="nano-q8-greedy", family="llama", kind="turn", tier="nano", wtype="q8_0", context=0, tokens=40, reply=64, sampled=False),
        # the same with the command line's default sampling settings
        dict(name="nano-q8-sampled", family="llama", kind="turn", tier="nano", wtype="q8_0", context=0, tokens=40, reply=48, sampled=True),
        # a document that fills the context, 4-bit weights
        dict(name="mini-q4-document", family="llama", kind="prompt", tier="mini", wtype="q4_0", context=0, tokens=2047),
        # a page to a file of 256-value super-blocks (4-bit layers, 6-bit output matrix), as most files found outside are
        dict(name="mini-q4k-page", family="llama", kind="prompt", tier="mini", wtype="q4_k", context=0, tokens=333),
        # a long prompt to an unquantised file
        dict(name="goldie-f16-prompt", family="llama", kind="prompt", tier="goldie", wtype="f16", context=0, tokens=993),
        # a turn in the middle of a long conversation
        dict(name="goldie-q8-turn", family="llama", kind="turn", tier="goldie", wtype="q8_0", context=700, tokens=33, reply=16, sampled=False),
        # a serving host's decode streams
        dict(name="goldie-q4-streams", family="llama", kind="streams", tier="goldie", wtype="q4_0", streams=64, context=100, steps=4),
        # the largest tier's layers, one stream
        dict(name="wide-q4-greedy", family="llama", kind="turn", tier="wide", wtype="q4_0", context=300, tokens=17, reply=32, sampled=False),
        # --- layer-stack models ---
        # a document to a linear-attention model
        dict(name="ganidra-document", family="ganidra", kind="prompt", size="goldie", dtype="bfloat16", tokens=2047),
        # requests of a serving host: ragged prompts in one step, then decoded side by side
        dict(name="ganidra-requests", family="ganidra", kind="requests", size="mini", dtype="bfloat16", streams=48, tokens=40, steps=12),
        # one request to a latent-attention model, its reply sampled on the host
        dict(name="pabalix-request", family="pabalix", kind="requests", size="mini", dtype="bfloat16", streams=1, tokens=300, steps=24),
    ]


def _spread(rng: random.Random, low: int, high: int) -> int:
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng: random.Random) -> dict:
    """Prompts of a line up to the whole context, turns and streams from the start of a conversation to its end; replies are cut to the
    cost of the largest listed case."""
    case = _draw(rng)
    most = [max(work(c)[k] for c in listed()) for k in ("bytes", "flops")]
    for part in ("reply", "steps", "tokens"):
        while case.get(part, 0) > (15 if part == "tokens" else 2) and (work(case)["bytes"] > most[0] or work(case)["flops"] > most[1]):
            case[part] = case[part] * 3 // 4
    return case


def _draw(rng: random.Random) -> dict:
    kind = rng.choice(["prompt", "prompt", "prompt", "turn", "turn", "streams", "stack prompt", "stack requests", "stack requests"])
    if kind.startswith("stack"):
        family, size = rng.choice(["ganidra", "pabalix"]), rng.choice(["mini", "mini", "goldie"])
        dtype = "float32" if size == "mini" and rng.random() < 0.25 else "bfloat16"
        if kind == "stack prompt":
            return dict(family=family, kind="prompt", size=size, dtype=dtype, tokens=_spread(rng, 16, 600 if dtype == "float32" else 2047 if size == "mini" else 1900))
        streams = _spread(rng, 1, 64)
        return dict(family=family, kind="requests", size=size, dtype=dtype, streams=streams, tokens=_spread(rng, 8, max(8, min(500, 1600 // streams))), steps=rng.randint(4, 20))
    tier = rng.choice(["nano", "mini", "mini", "goldie", "wide"])
    wtype = rng.choice(["q8_0", "q4_0", "f16", "q5_0"] + ([] if tier == "nano" else ["q4_k", "q6_k"]))
    super_blocks = wtype in ("q4_k", "q6_k")
    if kind == "prompt":
        context = rng.choice([0, 0, _spread(rng, 20, 300 if super_blocks else 900)])
        most = {"nano": 2047, "mini": 2047, "goldie": 993, "wide": 993}[tier] - context
        if super_blocks:
            most = min(most, {"mini": 333, "goldie": 120, "wide": 240}[tier])
        return dict(family="llama", kind="prompt", tier=tier, wtype=wtype, context=context, tokens=_spread(rng, 16, max(17, most)))
    if kind == "turn":
        context = rng.choice([0, _spread(rng, 20, 300 if super_blocks else 1800)])
        return dict(family="llama", kind="turn", tier=tier, wtype=wtype, context=context, tokens=_spread(rng, 16, 60), reply=rng.randint(8, 40), sampled=rng.random() < 0.4)
    return dict(family="llama", kind="streams", tier=tier, wtype=wtype, streams=_spread(rng, 3, 16 if super_blocks else 64), context=_spread(rng, 10, 60 if super_blocks else 900),
                steps=rng.randint(2, 5))


# ---------------------------------------------------------------- weights

def _llama_tensors(tier: str, wtype: str) -> List[Tuple[str, str, int, int]]:
    """(name, format, rows, columns); rows 0: a vector of float32.  A file of 4-bit super-blocks has a 6-bit output matrix."""
    L, D, H, G, V, F = TIERS[tier]
    out = [("token_embd.weight", wtype, V, D)]
    for i in range(L):
        p = f"blk.{i}."
        out += [(p + "attn_norm.weight", "f32", 0, D), (p + "attn_q.weight", wtype, H * HEAD, D), (p + "attn_k.weight", wtype, G * HEAD, D),
                (p + "attn_v.weight", wtype, G * HEAD, D), (p + "attn_output.weight", wtype, D, H * HEAD), (p + "ffn_norm.weight", "f32", 0, D),
                (p + "ffn_gate.weight", wtype, F, D), (p + "ffn_up.weight", wtype, F, D), (p + "ffn_down.weight", wtype, D, F)]
    return out + [("output_norm.weight", "f32", 0, D), ("output.weight", "q6_k" if wtype == "q4_k" else wtype, V, D)]


def _half_bits(rng: np.random.Generator, target: float, n: int) -> np.ndarray:
    """n binary16 numbers of target's magnitude with random mantissas, as their bytes [n, 2]."""
    e = max(1, min(30, int(math.floor(math.log2(target))) + 15))
    return (rng.integers(0, 1024, n, dtype=np.uint16) | np.uint16(e << 10)).view(np.uint8).reshape(n, 2)


def _pool(rng: np.random.Generator, fmt: str, most: float, n: int) -> np.ndarray:
    """n blocks of weights spread evenly over about +- most."""
    size = BLOCKS[fmt][0]
    raw = rng.integers(0, 1 << 63, size=(n * size + 7) // 8, dtype=np.int64).view(np.uint8)[:n * size].reshape(n, size)
    if fmt == "f16":
        return ((rng.random((n, 32), dtype=np.float32) * 2 - 1) * np.float32(most)).astype(np.float16).view(np.uint8).reshape(n, 64)
    if fmt == "q4_k":                      # d scale q - dmin min
        raw[:, 0:2], raw[:, 2:4] = _half_bits(rng, most / 470.0, n), _half_bits(rng, most / 64.0, n)
    elif fmt == "q6_k":                    # d scale (q - 32)
        raw[:, 208:210] = _half_bits(rng, most / 4096.0, n)
    else:
        raw[:, 0:2] = _half_bits(rng, most / {"q8_0": 127.0, "q4_0": 8.0, "q5_0": 16.0}[fmt], n)
    return raw


class _Llama:
    """A parsed model file in memory, as load_llama_model takes one.  A tensor is a run of a pool of random blocks from a place of
    its own on: drawing every block anew would take minutes for the larger tiers."""

    def __init__(self, tier: str, wtype: str, seed: int):
        L, D, H, G, V, F = TIERS[tier]
        self.rng = np.random.default_rng([seed, 1])
        self.meta = GGUFMetadata()
        m = self.meta
        m.num_layers, m.embed_dim, m.num_heads, m.num_kv_heads, m.head_dim = L, D, H, G, HEAD
        m.vocab_size, m.seq_len, m.interm_size, m.rope_theta, m.rms_norm_eps = V, SEQ_LEN, F, 10000.0, EPS
        plan = _llama_tensors(tier, wtype)
        self.plan = {t[0]: t for t in plan}
        self.tensor_order = [t[0] for t in plan]
        self.at = {t[0]: int(k) for t, k in zip(plan, self.rng.integers(0, 1 << 30, len(plan)))}
        self.seed, self.width, self.pools = seed, D, {}

    def raw(self, name: str) -> np.ndarray:
        _, fmt, rows, cols = self.plan[name]
        if rows == 0:
            return np.random.default_rng([self.seed, 2, self.at[name]]).uniform(0.5, 1.5, cols).astype(np.float32).view(np.uint8)
        size, values, _ = BLOCKS[fmt]
        most = 4.0 if name == "token_embd.weight" else math.sqrt(3.0 / self.width)
        if (fmt, most) not in self.pools:
            self.pools[fmt, most] = _pool(np.random.default_rng([self.seed, 3, values, size, int(most * 1e6)]), fmt, most, 262139 if values == 32 else 40949)
        pool, need, out, at = self.pools[fmt, most], rows * cols // values, [], self.at[name]
        while need:
            part = pool[at % len(pool):][:need]
            out.append(part)
            need, at = need - len(part), 0
        return (out[0] if len(out) == 1 else np.concatenate(out)).reshape(-1)

    def get_tensor(self, name: str):
        _, fmt, rows, cols = self.plan[name]
        return self.raw(name), GGUFTensorInfo(name, 2 if rows else 1, (cols, rows) if rows else (cols,), BLOCKS[fmt][2], 0)


def _stack_config(family: str, size: str) -> dict:
    """As the layer-stack benchmark's: every fourth Ganidra layer runs windowed softmax attention beside linear attention; Pabalix has its
    three kinds of latent attention in turn, and every fourth layer attends the latents of the one two before it."""
    L, D, _, _, V, F = TIERS[size]
    if family == "pabalix":
        dims = dict(heads=D // 128, dim=128, rot_dim=64, vdim=128, kv_rank=256, q_rank=D // 2, base=10000.0)
        yarn = (4.0, 4096.0, 32.0, 1.0)
        kinds = [pabalix_layer(1, F, yarn=yarn, **dims), pabalix_layer(2, F, **dims), pabalix_layer(3, F, yarn=yarn, **dims)]
        return pabalix_config(V, D, [kinds[i % 4] if i % 4 < 3 else pabalix_layer(2, F, kv_from=i - 2, **dims) for i in range(L)])
    lin = lambda h: dict(heads=h, dim=64, vdim=128, tau=16.0)
    par = ganidra_layer("parallel", F, left=dict(heads=D // 128, kv_heads=max(1, D // 512), dim=64, vdim=64, scale=0.125, mask={"size": 1024}),
                        left_scale=0.7, right=lin(D // 256), right_scale=0.7)
    return ganidra_config(V, D, [par if i % 4 == 3 else ganidra_layer("gla", F, **lin(D // 128)) for i in range(L)])


class _Stack:
    """Weights of a layer-stack model: bfloat16 bits by name, runs of a pool of normal values per row length."""

    def __init__(self, family: str, size: str, seed: int):
        self.cfg = _stack_config(family, size)
        self.shapes = (pabalix_shapes if family == "pabalix" else ganidra_shapes)(self.cfg)
        self.family, self.seed, self.pools = family, seed, {}
        self.at = {n: int(k) for n, k in zip(self.shapes, np.random.default_rng([seed, 4]).integers(0, 1 << 30, len(self.shapes)))}

    def bits(self, name: str) -> np.ndarray:
        shape = self.shapes[name]
        if len(shape) == 1:
            rng = np.random.default_rng([self.seed, 5, self.at[name]])
            if name.endswith("a2.b"):
                x = rng.uniform(-3.0, 5.0, shape)                    # decays from nearly none to strong
            elif name.endswith("sink"):
                x = rng.uniform(-1.0, 3.0, shape)
            elif "norm" in name:                                     # gains: near 1, of Ganidra's residual stream near 0 (1 + w)
                near_zero = self.family == "ganidra" and (name == "final.norm" or name.endswith((".norm1", ".norm2")))
                x = (0.0 if near_zero else 1.0) + 0.2 * rng.standard_normal(shape)
            else:
                x = 0.3 * rng.standard_normal(shape)                 # biases
            return torch.from_numpy(x).to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)
        scale = 1.0 if name == "embed" else shape[1] ** -0.5
        if self.family == "ganidra" and name.endswith((".o", ".down")):
            scale *= (2 * len(self.cfg["layers"])) ** -0.5           # branches of a residual stream that no norm follows, as models are initialised
        if scale not in self.pools:
            x = np.random.default_rng([self.seed, 6, int(scale * 1e6)]).standard_normal(1 << 20, dtype=np.float32) * np.float32(scale)
            self.pools[scale] = torch.from_numpy(x[:1048573]).to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)
        pool, need, out, at = self.pools[scale], shape[0] * shape[1], [], self.at[name]
        while need:
            part = pool[at % len(pool):][:need]
            out.append(part)
            need, at = need - len(part), 0
        return np.concatenate(out).reshape(shape)


# ---------------------------------------------------------------- inputs

def _vocab(case: dict) -> int:
    return TIERS[case["tier"] if case["family"] == "llama" else case["size"]][4]


def _ids(case: dict, seed: int, what: int, n: int) -> List[int]:
    return [int(t) for t in np.random.default_rng([seed, 7, what]).integers(3, _vocab(case), n)]


def _lengths(case: dict) -> List[int]:
    """Prompt lengths of a case's requests: from half of `tokens` to one and a half times as many, the first exactly that."""
    n = case["tokens"]
    return [max(1, n // 2 + (n - n // 2 + i * 37 * max(1, n // 5)) % (n + 1)) for i in range(case["streams"])]


def _prompts(case: dict, seed: int) -> List[List[int]]:
    """Every stream's tokens before the first decode step (of a prompt or a turn: its context and its message)."""
    if case["kind"] == "streams":
        return [[1] + _ids(case, seed, 10 + s, case["context"] - 1) for s in range(case["streams"])]
    if case["kind"] == "requests":
        return [[1] + _ids(case, seed, 10 + s, n - 1) for s, n in enumerate(_lengths(case))]
    return [[1] + _ids(case, seed, 10, case.get("context", 0) + case["tokens"] - 1)]


def _fed(case: dict, seed: int) -> List[List[int]]:
    """The tokens of each decode step, one per stream (what a host's sampler picked)."""
    flat = _ids(case, seed, 8, case["streams"] * case["steps"])
    return [flat[i * case["streams"]:(i + 1) * case["streams"]] for i in range(case["steps"])]


# the command line's defaults
SAMPLING = dict(temperature=0.8, top_p=0.9, top_k=50, rep_penalty=1.15, rep_window=64)


def prepare(case: dict, seed: int):
    """A loaded model, the tokens, and for turns and streams the conversation so far in its cache."""
    streams = case.get("streams", 1)
    if case["family"] == "llama":
        model = load_llama_model(_Llama(case["tier"], case["wtype"], seed), max_streams=streams)
    else:
        w = _Stack(case["family"], case["size"], seed)
        spec = DESIGNS["Pabalix" if case["family"] == "pabalix" else "Ganidra"](w.cfg, lambda n: w.shapes[n])
        model = load_stack_model(spec, lambda n: ("BF16", w.bits(n)), max_streams=streams, seq_len=SEQ_LEN, dtype=case["dtype"])
    state = dict(case=case, model=model, prompts=_prompts(case, seed))
    if case["kind"] in ("streams", "requests"):
        state["fed"] = _fed(case, seed)
    if case.get("sampled"):
        state["uniforms"] = np.random.default_rng([seed, 9]).random(case["reply"], dtype=np.float32)
    if case["kind"] == "streams":
        for s, prompt in enumerate(state["prompts"]):
            model.prefill(prompt, 0, s, want_logits=False)
    elif case.get("context"):
        model.prefill(state["prompts"][0][:case["context"]], want_logits=False)
    return state


def run(state):
    case, model, prompts = state["case"], state["model"], state["prompts"]
    if case["kind"] == "streams":
        ids, every = [], list(range(case["streams"]))
        for i, tokens in enumerate(state["fed"]):
            picked, logits = model.forward_batch(every, tokens, [case["context"] + i] * len(every), want_logits=i == case["steps"] - 1)
            ids.append(picked)
        return {"ids": np.array(ids), "logits": logits}
    if case["kind"] == "requests":
        if case["streams"] == 1:
            model.reset()
            model.prefill(prompts[0])
            rows = [model.state.logits.copy()]
            for i, (token,) in enumerate(state["fed"]):
                model.forward(token, len(prompts[0]) + i)
                rows.append(model.state.logits.copy())
            return {"logits": rows}
        every = list(range(case["streams"]))
        for s in every:
            model.reset(s)
        first = model.step([(s, p, 0, [len(p) - 1]) for s, p in enumerate(prompts)])
        for i, tokens in enumerate(state["fed"]):
            _, logits = model.forward_batch(every, tokens, [len(p) + i for p in prompts], want_logits=i == case["steps"] - 1)
        return {"first": np.concatenate(first), "logits": logits}
    context = case.get("context", 0)
    if not context:
        model.reset()
    model.prefill(prompts[0][context:], context)
    if case["kind"] == "prompt":
        return {"logits": model.state.logits}
    logits, pos = model.state.logits.copy(), len(prompts[0])
    if case["sampled"]:
        ids, _ = model.sample_decode(pos, case["reply"], uniforms=state["uniforms"], recent=[], **SAMPLING)
    else:
        ids = [int(np.argmax(logits))]
        ids += model.decode_greedy(ids[0], pos, case["reply"] - 1)
    return {"logits": logits, "ids": np.array(ids)}


# ---------------------------------------------------------------- what a pass cannot do without

def _matrix_sizes(case: dict) -> Tuple[float, float, float, float]:
    """(values of the layers' matrices, their bytes, values of the output matrix, its bytes)"""
    if case["family"] == "llama":
        plan = [t for t in _llama_tensors(case["tier"], case["wtype"]) if t[2] and t[0] != "token_embd.weight"]
        size = lambda t: t[2] * t[3] / BLOCKS[t[1]][1] * BLOCKS[t[1]][0]
        layers, out = [t for t in plan if t[0] != "output.weight"], plan[-1]
        return sum(t[2] * t[3] for t in layers), sum(map(size, layers)), out[2] * out[3], size(out)
    w = _Stack(case["family"], case["size"], 0)
    item = 4 if case["dtype"] == "float32" else 2
    n = sum(math.prod(s) for k, s in w.shapes.items() if len(s) == 2 and k not in ("embed", "head"))
    head = math.prod(w.shapes["embed"])
    return n, n * item, head, head * item


def _mixing(case: dict) -> Tuple[float, float, float, float]:
    """Per token: (flops of mixing per visible position, bytes cached per position, flops of the recurrences, bytes of their state), all layers"""
    if case["family"] == "llama":
        L, _, H, G, _, _ = TIERS[case["tier"]]
        return 4.0 * H * HEAD * L, 8.0 * G * HEAD * L, 0.0, 0.0
    item = 4 if case["dtype"] == "float32" else 2
    per, cached, rec, state = 0.0, 0.0, 0.0, 0.0
    for layer in _stack_config(case["family"], case["size"])["layers"]:
        m = layer["mixer"]
        if case["family"] == "pabalix":
            per += 2.0 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
            cached += item * (m["kv_rank"] + m["rot_dim"])
            continue
        lin = m
        if layer["type"] == "parallel":
            a, lin = m["left"], m["right"]
            per += 2.0 * a["heads"] * (a["dim"] + a["vdim"])
            cached += item * a["kv_heads"] * (a["dim"] + a["vdim"])
        rec += 4.0 * lin["heads"] * lin["dim"] * lin["vdim"]
        state += 4.0 * lin["heads"] * lin["dim"] * lin["vdim"]
    return per, cached, rec, state


def work(case: dict) -> Dict[str, float]:
    n_layers, b_layers, n_head, b_head = _matrix_sizes(case)
    per, cached, rec, state = _mixing(case)
    vocab = _vocab(case)

    def step(spans: List[Tuple[int, int]], heads: int) -> Tuple[float, float]:
        """Token runs (first position, tokens) of streams through the model once, `heads` rows of logits."""
        tokens = sum(n for _, n in spans)
        seen = sum(n * p + n * (n + 1) / 2 for p, n in spans)
        b = b_layers + (b_head if heads else 0) + sum((p + n) * cached for p, n in spans) + tokens * cached + len(spans) * 2 * state
        return b, 2.0 * n_layers * tokens + 2.0 * n_head * heads + per * seen + rec * tokens

    if case["kind"] == "streams":
        parts = [step([(case["context"] + i, 1)] * case["streams"], case["streams"]) for i in range(case["steps"])] + [(4.0 * vocab * case["streams"], 0.0)]
    elif case["kind"] == "requests":
        lens = _lengths(case)
        rows = case["streams"] * (2 if case["streams"] > 1 else 1 + case["steps"])
        parts = [step([(0, n) for n in lens], case["streams"])] + [step([(n + i, 1) for n in lens], case["streams"]) for i in range(case["steps"])] + [(4.0 * vocab * rows, 0.0)]
    else:
        parts = [step([(case.get("context", 0), case["tokens"])], 1), (4.0 * vocab, 0.0)]
        at = case.get("context", 0) + case["tokens"]
        parts += [step([(at + i, 1)], 1) for i in range(case.get("reply", 0))]
    return {"bytes": sum(b for b, _ in parts), "flops": sum(f for _, f in parts)}


def tolerance(case: dict):
    """Llama files and float32: sums in 32 bits, in any order, through up to 28 layers; ids where two logits are nearly equal.  Super-block
    files: up to 1.5e-5 from 64 bits was seen, since a block's least value is subtracted as a sum of its own.  bfloat16: products' inputs
    rounded to 8 bits."""
    if case.get("dtype") == "bfloat16":
        return {"rel": 0.025, "max": 0.25}
    if case.get("wtype") in ("q4_k", "q6_k"):
        return {"rel": 6e-5, "max": 6e-4, "differ": 0.01}
    return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}


# ---------------------------------------------------------------- the same in 64 bits

def _dequantise(raw: np.ndarray, fmt: str, rows: int, cols: int) -> torch.Tensor:
    """ggml's block formats, [rows, cols] in float64 on the GPU."""
    b = torch.from_numpy(np.array(raw)).cuda().view(-1, BLOCKS[fmt][0])
    half = lambda lo: b[:, lo:lo + 2].contiguous().view(torch.float16).double()
    if fmt == "f16":
        return b.view(torch.float16).double().view(rows, cols)
    if fmt == "q8_0":
        w = b[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif fmt in ("q4_0", "q5_0"):
        q = b[:, -16:].int()
        lo, hi, off = q & 15, q >> 4, 8
        if fmt == "q5_0":
            high = b[:, 2:6].contiguous().view(torch.int32)
            j = torch.arange(16, device="cuda", dtype=torch.int32)
            lo, hi, off = lo | ((high >> j & 1) << 4), hi | ((high >> (j + 16) & 1) << 4), 16
        w = (torch.cat([lo, hi], 1) - off).double() * half(0)
    elif fmt == "q4_k":
        s, q = b[:, 4:16].int(), b[:, 16:].int().view(-1, 4, 32)
        scale = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1).double()
        least = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        w = (half(0) * scale)[:, :, None] * q - (half(2) * least)[:, :, None]
    else:
        low, high, s = b[:, :128].int().view(-1, 2, 2, 32), b[:, 128:192].int().view(-1, 2, 32), b[:, 192:208].contiguous().view(torch.int8).double()
        q = torch.stack([(low[:, :, 0] & 15) | (high & 3) << 4, (low[:, :, 1] & 15) | (high >> 2 & 3) << 4,
                         (low[:, :, 0] >> 4) | (high >> 4 & 3) << 4, (low[:, :, 1] >> 4) | (high >> 6 & 3) << 4], 2)
        w = (q.reshape(-1, 16, 16) - 32).double() * (half(208) * s)[:, :, None]
    return w.reshape(rows, cols)


def _rms(x: torch.Tensor, eps: float) -> torch.Tensor:
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


class _ExactLlama:
    def __init__(self, tier: str, wtype: str, seed: int):
        self.L, self.D, self.H, self.G, self.V, _ = TIERS[tier]
        f = _Llama(tier, wtype, seed)
        self.w = {n: torch.from_numpy(f.raw(n).view(np.float32).copy()).cuda().double() if t[2] == 0 else _dequantise(f.raw(n), *t[1:]) for n, t in f.plan.items()}
        self.k, self.v = [None] * self.L, [None] * self.L

    def step(self, ids: torch.Tensor) -> torch.Tensor:
        """ids [streams, tokens] behind what the cache holds -> logits of all of them"""
        S, T = ids.shape
        x = self.w["token_embd.weight"][ids]
        past = 0 if self.k[0] is None else self.k[0].shape[2]
        angle = torch.arange(past, past + T, device="cuda").double()[:, None] * 10000.0 ** (-torch.arange(0, HEAD, 2, device="cuda").double() / HEAD)
        c, s = angle.cos(), angle.sin()
        seen = torch.arange(past + T, device="cuda")[None, :] <= torch.arange(past, past + T, device="cuda")[:, None]

        def heads(y, n, turn):
            y = y.view(S, T, n, HEAD).transpose(1, 2)
            if not turn:
                return y
            a, b = y[..., :HEAD // 2], y[..., HEAD // 2:]
            return torch.cat([a * c - b * s, a * s + b * c], -1)
        for i in range(self.L):
            w = lambda n: self.w[f"blk.{i}.{n}.weight"]
            h = _rms(x, EPS) * w("attn_norm")
            q, k, v = heads(h @ w("attn_q").T, self.H, True), heads(h @ w("attn_k").T, self.G, True), heads(h @ w("attn_v").T, self.G, False)
            k = self.k[i] = k if self.k[i] is None else torch.cat([self.k[i], k], 2)
            v = self.v[i] = v if self.v[i] is None else torch.cat([self.v[i], v], 2)
            r = self.H // self.G
            o = torch.empty_like(q)
            for j in range(self.H):
                p = (q[:, j] @ k[:, j // r].transpose(1, 2).contiguous() / math.sqrt(HEAD)).masked_fill(~seen, -math.inf).softmax(-1)
                o[:, j] = p @ v[:, j // r]
            x = x + o.transpose(1, 2).reshape(S, T, -1) @ w("attn_output").T
            h = _rms(x, EPS) * w("ffn_norm")
            x = x + (torch.nn.functional.silu(h @ w("ffn_gate").T) * (h @ w("ffn_up").T)) @ w("ffn_down").T
        return _rms(x, EPS) * self.w["output_norm.weight"]

    def logits(self, x: torch.Tensor) -> torch.Tensor:
        return x @ self.w["output.weight"].T


def _exact_llama(case: dict, seed: int):
    m, prompts = _ExactLlama(case["tier"], case["wtype"], seed), _prompts(case, seed)
    if case["kind"] == "streams":
        fed = torch.tensor(_fed(case, seed)).T
        x = m.step(torch.cat([torch.tensor(prompts), fed], 1).cuda())[:, case["context"]:]
        rows = m.logits(x)
        return {"ids": None, "logits": rows[:, -1]}
    row = m.logits(m.step(torch.tensor(prompts).cuda())[0, -1])
    if case["kind"] == "prompt":
        return {"logits": row}
    return {"logits": row, "ids": None}


def _silu(z):
    return z * torch.sigmoid(z)


class _ExactStack:
    def __init__(self, family: str, size: str, seed: int):
        w = _Stack(family, size, seed)
        self.cfg = w.cfg
        self.w = {n: torch.from_numpy(w.bits(n).view(np.int16).copy()).view(torch.bfloat16).cuda().double() for n in w.shapes}

    def recurrence(self, h, m, p):
        S, T, _ = h.shape
        H, dk, dv, w = m["heads"], m["dim"], m["vdim"], self.w
        q = (h @ w[p + "q"].T).view(S, T, H, dk) * dk ** -0.5
        k, v = (h @ w[p + "k"].T).view(S, T, H, dk), (h @ w[p + "v"].T).view(S, T, H, dv)
        alpha = torch.exp(torch.nn.functional.logsigmoid(h @ w[p + "a1"].T @ w[p + "a2"].T + w[p + "a2.b"]) / m["tau"]).view(S, T, H, dk)
        state, o = torch.zeros(S, H, dk, dv, dtype=torch.float64, device="cuda"), torch.empty(S, T, H, dv, dtype=torch.float64, device="cuda")
        for t in range(T):
            state = torch.addcmul(state * alpha[:, t, :, :, None], k[:, t, :, :, None], v[:, t, :, None, :])
            o[:, t] = (state * q[:, t, :, :, None]).sum(2)
        o = _rms(o, self.cfg["norm"]["eps"]) * w[p + "norm"]
        return (o.reshape(S, T, H * dv) * _silu(h @ w[p + "g"].T)) @ w[p + "o"].T

    def window(self, h, m, p):
        S, T, _ = h.shape
        H, G, dk, dv, w, eps = m["heads"], m["kv_heads"], m["dim"], m["vdim"], self.w, self.cfg["norm"]["eps"]
        q = _rms((h @ w[p + "q"].T).view(S, T, H, dk), eps) * w[p + "q.norm"]
        k = _rms((h @ w[p + "k"].T).view(S, T, G, dk), eps) * w[p + "k.norm"]
        v = (h @ w[p + "v"].T).view(S, T, G, dv)
        back = torch.arange(T, device="cuda")[:, None] - torch.arange(T, device="cuda")[None, :]
        seen = (back >= 0) & (back < m["mask"]["size"])
        out = torch.empty(S, T, H, dv, dtype=torch.float64, device="cuda")
        for a in range(H):
            g = a // (H // G)
            s = q[:, :, a].contiguous() @ k[:, :, g].transpose(1, 2).contiguous() * m["scale"] - 2.0 ** (-8.0 * (a + 1) / H) * back
            out[:, :, a] = s.masked_fill(~seen, -math.inf).softmax(-1) @ v[:, :, g].contiguous()
        return (out.view(S, T, H * dv) * torch.sigmoid(h @ w[p + "g"].T)) @ w[p + "o"].T

    def turn(self, x, rot, adjacent):
        """x [S, T, heads, dims]"""
        n, base = rot["dims"], rot["base"]
        f, size = base ** (-2.0 * torch.arange(n // 2, device="cuda").double() / n), 1.0
        if rot.get("scaling"):
            y = rot["scaling"]
            turns = lambda t: n * math.log(y["original"] / (2 * math.pi * t)) / (2 * math.log(base))
            lo, hi = max(math.floor(turns(y["fast"])), 0.0), min(math.ceil(turns(y["slow"])), n - 1.0)
            slow = ((torch.arange(n // 2, device="cuda").double() - lo) / max(hi - lo, 0.001)).clamp(0, 1)
            f, size = f / y["factor"] * slow + f * (1 - slow), 0.1 * math.log(y["factor"]) + 1.0
        a = (torch.arange(x.shape[1], device="cuda").double()[:, None] * f)[:, None, :]
        c, s = size * a.cos(), size * a.sin()
        first, second = (slice(0, n, 2), slice(1, n, 2)) if adjacent else (slice(0, n // 2), slice(n // 2, n))
        out = x.clone()
        out[..., first] = x[..., first] * c - x[..., second] * s
        out[..., second] = x[..., second] * c + x[..., first] * s
        return out

    def latent(self, h, m, p, kind, held):
        S, T, _ = h.shape
        H, d, r, dv, w, eps = m["heads"], m["dim"], m["rot_dim"], m["vdim"], self.w, self.cfg["norm"]["eps"]
        adjacent, third = kind.endswith("_2"), kind.endswith("_3")
        if m.get("kv_from") is None:
            c = h @ w[p + "dkv"].T
            held = _rms(c[..., :m["kv_rank"]], eps) * w[p + "dkv.norm"], self.turn(c[..., None, m["kv_rank"]:], m["rot"], adjacent)[:, :, 0]
        q = ((_rms(h @ w[p + "dq"].T, eps) * w[p + "dq.norm"]) @ w[p + "uq"].T).view(S, T, H, d + r)
        qr = self.turn(q[..., d:], m["rot"], adjacent)
        k, v = (held[0] @ w[p + "uk"].T).view(S, T, H, d), (held[0] @ w[p + "uv"].T).view(S, T, H, dv)
        hidden = torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1)
        out = torch.empty(S, T, H, dv, dtype=torch.float64, device="cuda")
        for a in range(H):
            s = q[:, :, a, :d].contiguous() @ k[:, :, a].transpose(1, 2).contiguous() + qr[:, :, a].contiguous() @ held[1].transpose(1, 2).contiguous()
            s = (s * m["scale"]).masked_fill(hidden, -math.inf)
            if third:                                                 # a score of the denominator alone
                s = torch.cat([s, w[p + "sink"][a].expand(S, T, 1)], -1)
            out[:, :, a] = s.softmax(-1)[..., :T].contiguous() @ v[:, :, a].contiguous()
        if third:
            out = out * torch.sigmoid(h @ w[p + "g"].T)[..., None]
        return out.view(S, T, H * dv) @ w[p + "o"].T, held

    def forward(self, ids: torch.Tensor) -> torch.Tensor:
        """ids [S, T] -> what the output matrix is multiplied with"""
        w, eps = self.w, self.cfg["norm"]["eps"]
        pabalix = self.cfg["architecture"] == "Pabalix"
        norm = lambda x, g: _rms(x, eps) * (w[g] if pabalix else 1.0 + w[g])
        x, held = w["embed"][ids] * (1.0 if pabalix else self.cfg["embedding"]["scale"]), {}
        for i, layer in enumerate(self.cfg["layers"]):
            p, m, h = f"l{i}.", layer["mixer"], norm(x, f"l{i}.norm1")
            if pabalix:
                o, held[i] = self.latent(h, m, p + "mix.", layer["type"], held.get(m.get("kv_from")))
                x = x + norm(o, p + "norm1b")
                h = norm(x, p + "norm2")
                h = _silu(h @ w[p + "mlp.gate"].T + w[p + "mlp.gate.b"]) * (h @ w[p + "mlp.up"].T + w[p + "mlp.up.b"])
                x = x + norm(h @ w[p + "mlp.down"].T + w[p + "mlp.down.b"], p + "norm2b")
                continue
            if layer["type"] == "parallel":
                x = x + m["left_scale"] * self.window(h, m["left"], p + "mix.left.") + m["right_scale"] * self.recurrence(h, m["right"], p + "mix.right.")
            else:
                x = x + self.recurrence(h, m, p + "mix.")
            h = norm(x, p + "norm2")
            x = x + (torch.nn.functional.gelu(h @ w[p + "mlp.gate"].T, approximate="tanh") * (h @ w[p + "mlp.up"].T)) @ w[p + "mlp.down"].T
        return norm(x, "final.norm")

    def logits(self, x):
        return x @ self.w["head" if self.cfg["architecture"] == "Pabalix" else "embed"].T


def exact(case: dict, seed: int):
    """What run returns, in 64 bits: logits (the ids that follow them are picked, not computed)."""
    if case["family"] == "llama":
        return _exact_llama(case, seed)
    m, prompts = _ExactStack(case["family"], case["size"], seed), _prompts(case, seed)
    if case["kind"] == "prompt":
        return {"logits": m.logits(m.forward(torch.tensor(prompts).cuda())[0, -1])}
    fed = list(zip(*_fed(case, seed)))
    whole = [p + list(f) for p, f in zip(prompts, fed)]
    most = max(map(len, whole))                                       # shorter ones are followed by tokens that nothing before them sees
    x = m.forward(torch.tensor([t + [1] * (most - len(t)) for t in whole]).cuda())
    if case["streams"] == 1:
        return {"logits": [m.logits(x[0, len(prompts[0]) - 1 + i]) for i in range(case["steps"] + 1)]}
    return {"first": torch.stack([m.logits(x[s, len(p) - 1]) for s, p in enumerate(prompts)]),
            "logits": torch.stack([m.logits(x[s, len(t) - 1]) for s, t in enumerate(whole)])}
