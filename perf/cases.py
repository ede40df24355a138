"""Workloads the decoder library is timed on, through its public entry points.

Three kinds of calls a program makes:

* single layers over device tensors (the C ABI's kernel-level entry points):
  a linear in each weight format and activation width, RoPE + KV append +
  attention, and a gated MLP block (norm, gate|up, SiLU gate, down);
* whole decoders (``runtime.Decoder``) on seeded random-init models of the
  preset widths, their depth cut so that a model is written in seconds.

Layer shapes are those of the presets in ``leaf_amd/models.py`` and of the
tests; drawn cases spread over the same ranges, odd sizes among them.
"""
from __future__ import annotations

import ctypes as C
import functools
import math
import os
import tempfile
from pathlib import Path

import numpy as np
import torch

from leaf_amd import artifact, models, runtime

# Layers kept of each preset (full width, full vocabulary).
DEPTH = {"tinyllama": 6, "smollm2": 6, "qwen": 4, "gpt2": 6}
CONTEXT = 2048
# (hidden, intermediate) of the presets' MLPs.
MLP_SIZES = ((768, 3072), (960, 2560), (896, 4864), (2048, 5632))
# (heads, kv_heads): the presets' groupings, and eight KV heads for 32.
HEADS = ((32, 4), (14, 2), (15, 5), (12, 12), (32, 8))
EPSILON = 1e-5


# ------------------------------------------------------------------- cases ---
def _linear(bits, act, tokens, cols, rows, group=0, bias=False):
    return {"kind": "linear", "bits": bits, "act": act, "tokens": tokens, "cols": cols, "rows": rows,
            "group": group, "bias": bias}


def _mlp(bits, tokens, hidden, ffn, group=0):
    return {"kind": "mlp", "bits": bits, "tokens": tokens, "hidden": hidden, "ffn": ffn, "group": group}


def _attention(tokens, position, heads, kv_heads, dim, window=0):
    return {"kind": "attention", "tokens": tokens, "position": position, "heads": heads, "kv_heads": kv_heads,
            "dim": dim, "window": window}


def _model(family, prompt, steps):
    return {"kind": "model", "family": family, "prompt": prompt, "steps": steps}


def listed():
    cases = {
        # One generated token through a stacked W8A8 gate|up projection: the smallest call, launch latency.
        "linear_w8a8_decode": _linear(8, 8, 1, 2048, 11264),
        # The stacked gate|up projection of a 512-token W8A8 prompt.
        "linear_w8a8_prefill": _linear(8, 8, 512, 2048, 11264),
        # A short prompt through an INT8 projection exported with a scale per 128 inputs.
        "linear_w8a8_grouped": _linear(8, 8, 96, 2048, 2048, group=128),
        # INT4 weights with 8-bit activations (an artifact of 4 bits run at activation bits 8), a ragged prompt.
        "linear_w4a8_prefill": _linear(4, 8, 201, 896, 4864, group=32),
        # A chat turn's few new tokens through an FP32 projection with a bias.
        "linear_f32_short": _linear(32, 32, 16, 3072, 768, bias=True),
        # The MLP block of a long prompt, weights kept as BF16.
        "mlp_bf16_prefill": _mlp(16, 2048, 960, 2560),
        # The MLP block of an INT4 model on a prompt of odd length.
        "mlp_int4_prefill": _mlp(4, 777, 896, 4864, group=32),
        # A long prompt's attention, grouped heads of 64.
        "attention_prefill": _attention(2048, 0, 14, 2, 64),
        # A prompt chunk behind cached keys, heads of 128.
        "attention_chunk_wide": _attention(256, 1000, 32, 8, 128),
        # One generated token at a long context.
        "attention_decode": _attention(1, 4095, 14, 2, 64),
        # A W8A8 decoder answers a 512-token prompt with 32 greedy tokens.
        "model_w8a8": _model("tinyllama", 512, 32),
        # A BF16 decoder reads a 256-token prompt, then a program samples 16 tokens from host logits.
        "model_bf16": _model("smollm2", 256, 16),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["linear"] * 9 + ["attention"] * 5 + ["mlp"] * 4 + ["model"] * 2)
    if kind == "linear":
        bits, act, group = rng.choice(((32, 32, 0), (16, 32, 0), (8, 32, 0), (4, 32, 32), (4, 32, 64),
                                       (8, 8, 0), (8, 8, 64), (8, 8, 128), (4, 8, 32), (4, 8, 64)))
        step = group or (4 if bits >= 16 and rng.random() < 0.25 else 64)
        cols = max(1, _log_int(rng, 256, 6144) // step) * step
        rows = _log_int(rng, 64, 16384)
        if rng.random() < 0.5:
            rows = -(-rows // 64) * 64
        # a single token over a small matrix is the price of a launch; matrices of an MLP or a head start there
        fewest = 1 if cols * rows * bits >= 1.6e8 else 5
        tokens = max(fewest, min(_log_int(rng, 1, 2048), int(1.2e10 / (2 * cols * rows))))
        return _linear(bits, act, tokens, cols, rows, group, rng.random() < 0.3)
    if kind == "attention":
        heads, kv_heads = rng.choice(HEADS)
        dim = rng.choice((64, 64, 64, 128, 80, 32))
        tokens = _log_int(rng, 1, 2048)
        position = 0 if tokens > 1 and rng.random() < 0.4 else _log_int(rng, 1, 4096)
        keys = position + tokens
        tokens = min(tokens, max(1, int(7e9 / (4 * heads * dim * keys))))
        return _attention(tokens, position, heads, kv_heads, dim, rng.choice((0, 0, 0, 512)))
    if kind == "mlp":
        bits, group = rng.choice(((32, 0), (16, 0), (8, 0), (4, 32)))
        hidden, ffn = rng.choice(MLP_SIZES)
        tokens = min(_log_int(rng, 1, 2048), int(3e10 / (6 * hidden * ffn)))
        return _mlp(bits, tokens, hidden, ffn, group)
    return _model(rng.choice(("tinyllama", "smollm2", "qwen", "gpt2")), _log_int(rng, 6, 512), rng.randint(4, 24))


# ------------------------------------------------------------------ inputs ---
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _activations(gen, rows, cols):
    """N(0, 1) with one value in a thousand an outlier twenty times as large."""
    x = torch.randn(rows, cols, generator=gen, device="cuda")
    outlier = torch.rand(rows, cols, generator=gen, device="cuda") < 0.001
    return torch.where(outlier, 20 * x, x)


class Matrix:
    """One weight matrix N(0, 0.02) in its artifact storage, on the device."""

    def __init__(self, gen, rows, cols, bits, group=0, bias=False):
        w = 0.02 * torch.randn(rows, cols, generator=gen, device="cuda")
        group = group or (cols if bits in (8, 4) else 0)
        self.scales = None
        self.integers = None
        if bits == 32:
            self.data = w
        elif bits == 16:
            self.data = w.bfloat16()
        else:
            limit = (1 << (bits - 1)) - 1
            grouped = w.view(rows, cols // group, group)
            self.scales = (grouped.abs().amax(-1) / limit).clamp_min(1e-12).contiguous()
            q = (grouped / self.scales[..., None]).round().clamp(-limit, limit).to(torch.int8).view(rows, cols)
            self.integers = q
            if bits == 4:
                nibbles = q.view(torch.uint8) & 15
                q = nibbles[:, 0::2] | (nibbles[:, 1::2] << 4)
            self.data = q.contiguous()
        self.bias = 0.1 * torch.randn(rows, generator=gen, device="cuda") if bias else None
        self.rows, self.cols, self.bits, self.group = rows, cols, bits, group
        self.desc = runtime.Weight(self.data.data_ptr(), self.scales.data_ptr() if self.scales is not None else None,
                                   self.bias.data_ptr() if bias else None, rows, cols, bits, group)

    def double(self):
        """The matrix in 64 bits."""
        if self.integers is None:
            return self.data.double()
        return self.integers.double() * self.scales.double().repeat_interleave(self.group, dim=1)


def _linear_bytes(bits, rows, cols, group):
    scales = 4 * rows * (cols // (group or cols)) if bits in (8, 4) else 0
    return rows * cols * bits // 8 + scales


def _rope_tables(positions, dim):
    angle = np.arange(positions, dtype=np.float32)[:, None] * \
        (np.float32(10000.0) ** (-np.arange(0, dim, 2, dtype=np.float32) / np.float32(dim)))[None, :]
    return (torch.from_numpy(np.cos(angle)).cuda().contiguous(), torch.from_numpy(np.sin(angle)).cuda().contiguous())


def _spec(family):
    return models.PRESETS[family](layers=DEPTH[family])


def _artifact(family):
    """The family's seeded artifact, written once per machine."""
    folder = Path(tempfile.gettempdir()) / f"leaf-cases-{os.getuid()}"
    folder.mkdir(exist_ok=True)
    path = folder / f"{family}-{DEPTH[family]}.leaf"
    if not path.exists():
        artifact.write_artifact(path, _spec(family), seed=11)
    return path


@functools.lru_cache(maxsize=4)
def _decoder(family):
    """A program's loaded decoder, kept for all of its prompts."""
    bits, math_policy = models.RUN_POLICY[family]
    context = min(CONTEXT, _spec(family).max_positions)
    return runtime.Decoder(_artifact(family), bits, math_policy, max_context=context, max_prefill=512)


def _inputs(case, seed):
    """The tensors of a layer case."""
    gen = _generator(seed)
    if case["kind"] == "linear":
        w = Matrix(gen, case["rows"], case["cols"], case["bits"], case["group"], case["bias"])
        return {"w": w, "x": _activations(gen, case["tokens"], case["cols"])}
    if case["kind"] == "mlp":
        hidden, ffn = case["hidden"], case["ffn"]
        return {"gate_up": Matrix(gen, 2 * ffn, hidden, case["bits"], case["group"]),
                "down": Matrix(gen, hidden, ffn, case["bits"], case["group"]),
                "gamma": 1 + 0.1 * torch.randn(hidden, generator=gen, device="cuda"),
                "x": _activations(gen, case["tokens"], hidden)}
    heads, kv, dim = case["heads"], case["kv_heads"], case["dim"]
    tokens, position = case["tokens"], case["position"]
    keys = torch.randn(kv, position + tokens, dim, generator=gen, device="cuda")
    values = torch.randn(kv, position + tokens, dim, generator=gen, device="cuda")
    keys[:, position:] = 0        # the rows this call appends
    values[:, position:] = 0
    return {"qkv": torch.randn(tokens, (heads + 2 * kv) * dim, generator=gen, device="cuda"), "keys": keys,
            "values": values}


def prepare(case, seed):
    if case["kind"] == "model":
        rng = np.random.default_rng(seed)
        vocab, steps = _spec(case["family"]).vocab, case["steps"]
        return {"case": case, "decoder": _decoder(case["family"]),
                "prompt": rng.integers(0, vocab, case["prompt"]).astype(np.uint32),
                "next": rng.integers(0, vocab, (steps, 1)).astype(np.uint32),
                "logits": np.empty((steps + 1, vocab), np.float32)}
    s = {"case": case, **_inputs(case, seed)}
    tokens = case["tokens"]
    if case["kind"] == "linear":
        s["y"] = torch.empty(tokens, case["rows"], device="cuda")
    elif case["kind"] == "mlp":
        s["normed"] = torch.empty(tokens, case["hidden"], device="cuda")
        s["pair"] = torch.empty(tokens, 2 * case["ffn"], device="cuda")
        s["act"] = torch.empty(tokens, case["ffn"], device="cuda")
        s["y"] = torch.empty(tokens, case["hidden"], device="cuda")
    else:
        s["cos"], s["sin"] = _rope_tables(case["position"] + tokens, case["dim"])
        s["q"] = torch.empty(case["heads"], tokens, case["dim"], device="cuda")
        s["out"] = torch.empty(tokens, case["heads"] * case["dim"], device="cuda")
    return s


# -------------------------------------------------------------------- runs ---
def _call_linear(lib, w, x, tokens, act, y):
    runtime.check(lib.lh_linear(C.byref(w.desc), x.data_ptr(), tokens, act, y.data_ptr(), None, None))


def run(state):
    case = state["case"]
    if case["kind"] == "model":
        return _run_model(state)
    lib = runtime.library()
    if case["kind"] == "linear":
        _call_linear(lib, state["w"], state["x"], case["tokens"], case["act"], state["y"])
        return state["y"]
    tokens = case["tokens"]
    if case["kind"] == "mlp":
        hidden, ffn = case["hidden"], case["ffn"]
        runtime.check(lib.lh_rmsnorm(state["x"].data_ptr(), tokens, hidden, state["gamma"].data_ptr(), EPSILON, 0,
                                     state["normed"].data_ptr(), None))
        _call_linear(lib, state["gate_up"], state["normed"], tokens, 32, state["pair"])
        runtime.check(lib.lh_silu_gate(state["pair"].data_ptr(), tokens, ffn, state["act"].data_ptr(), None))
        _call_linear(lib, state["down"], state["act"], tokens, 32, state["y"])
        return state["y"]
    heads, kv, dim, position = case["heads"], case["kv_heads"], case["dim"], case["position"]
    capacity = position + tokens
    runtime.check(lib.lh_rope_kv(state["qkv"].data_ptr(), tokens, heads, kv, dim, dim, position,
                                 state["cos"].data_ptr(), state["sin"].data_ptr(), state["q"].data_ptr(),
                                 state["keys"].data_ptr(), state["values"].data_ptr(), capacity, None))
    runtime.check(lib.lh_attention(state["q"].data_ptr(), state["keys"].data_ptr(), state["values"].data_ptr(),
                                   capacity, heads, kv, dim, tokens, position, case["window"],
                                   state["out"].data_ptr(), None))
    return {"out": state["out"], "keys": state["keys"], "values": state["values"]}


def _run_model(state):
    case, decoder, logits = state["case"], state["decoder"], state["logits"]
    decoder.reset()
    if case["family"] == "tinyllama":
        # greedy tokens on the device, then the logits that would choose the next one
        tokens, _, _ = decoder.generate(state["prompt"], case["steps"])
        decoder.forward_into(tokens[-1:], logits[0])
        return {"tokens": np.array(tokens, np.int64), "logits": logits[0]}
    # the program picks each token itself, from the logits it is handed
    decoder.forward_into(state["prompt"], logits[0])
    for step in range(case["steps"]):
        decoder.forward_into(state["next"][step], logits[step + 1])
    return {"logits": logits}


# -------------------------------------------------------- work and accuracy ---
def work(case):
    if case["kind"] == "linear":
        m, k, n = case["tokens"], case["cols"], case["rows"]
        return {"bytes": _linear_bytes(case["bits"], n, k, case["group"]) + 4 * m * (k + n), "flops": 2 * m * k * n}
    if case["kind"] == "mlp":
        m, h, f = case["tokens"], case["hidden"], case["ffn"]
        weights = _linear_bytes(case["bits"], 2 * f, h, case["group"]) + _linear_bytes(case["bits"], h, f,
                                                                                       case["group"])
        return {"bytes": weights + 8 * m * h, "flops": 6 * m * h * f}
    if case["kind"] == "attention":
        return _attention_work(case["tokens"], case["position"], case["heads"], case["kv_heads"], case["dim"],
                               case["window"])
    spec = _spec(case["family"])
    h, f, kv = spec.hidden, spec.intermediate, spec.kvwidth
    bits = 16 if spec.source_bf16 else spec.bits
    group = spec.group_size if bits == 4 else 0
    shapes = [(spec.qwidth + 2 * kv, h), (h, spec.qwidth), ((1 + spec.gated) * f, h), (h, f)]
    layer_bytes = sum(_linear_bytes(bits, n, k, group) for n, k in shapes)
    head_bits = 32 if "lm_head.weight" in spec.keep_fp32 else bits
    head_bytes = _linear_bytes(head_bits, spec.vocab, h, group if head_bits == 4 else 0)
    forwards = case["steps"] + 1
    rows = case["prompt"] + case["steps"]
    total = {"bytes": forwards * (spec.layers * layer_bytes + head_bytes),
             "flops": 2 * rows * spec.layers * sum(n * k for n, k in shapes) + 2 * forwards * spec.vocab * h}
    for tokens, position in [(case["prompt"], 0)] + [(1, case["prompt"] + i) for i in range(case["steps"])]:
        one = _attention_work(tokens, position, spec.heads, spec.kv_heads, spec.head_dim, 0)
        total = {key: total[key] + spec.layers * one[key] for key in total}
    return total


def _attention_work(tokens, position, heads, kv_heads, dim, window):
    visible = sum(min(position + t + 1, window or 1 << 30) for t in range(tokens))
    keys = min(position + tokens, window + tokens - 1 if window else 1 << 30)
    return {"bytes": 8 * kv_heads * dim * (keys + tokens) + 4 * tokens * (2 * heads + 2 * kv_heads) * dim,
            "flops": 4 * heads * dim * visible}


def tolerance(case):
    # Integer sums are exact and their epilogue has one order: nothing may
    # differ.  The W8A8 decoder runs in reference order, bit for bit.
    if case["kind"] == "linear" and case["act"] == 8 or case.get("family") == "tinyllama":
        return "exact"
    # Float32 sums in another order: about four times the error seen against
    # 64 bits (up to 1.8e-6 for linears, 5e-7 for attention, 1.1e-6 for logits).
    return {"rel": {"attention": 2e-6, "model": 5e-6}.get(case["kind"], 7e-6)}


def exact(case, seed):
    if case["kind"] == "model":
        # an int8 activation next to a rounding boundary has no 64-bit value
        return None if case["family"] == "tinyllama" else {"logits": _exact_model(case, seed)}
    s = _inputs(case, seed)
    if case["kind"] == "linear":
        return _exact_linear(s["w"], s["x"], case["act"])
    if case["kind"] == "mlp":
        x = s["x"].double()
        normed = x / (x.square().mean(-1, keepdim=True) + np.float32(EPSILON)).sqrt() * s["gamma"].double()
        gate, up = (normed @ s["gate_up"].double().T).chunk(2, dim=-1)
        return (up * gate * torch.sigmoid(gate)) @ s["down"].double().T
    heads, kv, dim = case["heads"], case["kv_heads"], case["dim"]
    tokens, position = case["tokens"], case["position"]
    cos, sin = (t.double() for t in _rope_tables(position + tokens, dim))
    q, k, v = s["qkv"].double().split([heads * dim, kv * dim, kv * dim], dim=-1)
    q = _rotate(q.view(tokens, heads, dim).transpose(0, 1), cos[position:], sin[position:])
    keys, values = s["keys"].double(), s["values"].double()
    keys[:, position:] = _rotate(k.view(tokens, kv, dim).transpose(0, 1), cos[position:], sin[position:])
    values[:, position:] = v.view(tokens, kv, dim).transpose(0, 1)
    return {"out": _exact_attention(q, keys, values, position, case["window"]), "keys": keys, "values": values}


def _exact_linear(w, x, act):
    bias = 0 if w.bias is None else w.bias.double()
    if act == 32:
        return x.double() @ w.double().T + bias
    scale = (x.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-12)
    q = (x * (1 / scale)).round().clamp(-127, 127)
    return (q.double() @ w.double().T) * scale.double() + bias


def _rotate(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def _exact_attention(q, keys, values, position, window):
    heads, tokens, dim = q.shape
    group = heads // keys.shape[0]
    at = torch.arange(position, position + tokens, device=q.device)[:, None]
    key = torch.arange(position + tokens, device=q.device)[None, :]
    seen = (key <= at) & (key > at - window if window else key >= 0)
    out = torch.empty(tokens, heads, dim, dtype=torch.float64, device=q.device)
    for h in range(heads):
        scores = (q[h] @ keys[h // group, :position + tokens].T.contiguous()) / math.sqrt(dim)
        out[:, h] = torch.softmax(scores.masked_fill(~seen, -math.inf), dim=-1) @ values[h // group,
                                                                                        :position + tokens]
    return out.view(tokens, heads * dim)


def _exact_model(case, seed):
    """The decoder's logits in 64 bits: teacher forcing makes the whole run one causal pass."""
    family = case["family"]
    spec, path = _spec(family), _artifact(family)
    rng = np.random.default_rng(seed)
    prompt = rng.integers(0, spec.vocab, case["prompt"])
    ids = torch.from_numpy(np.concatenate([prompt, rng.integers(0, spec.vocab, (case["steps"], 1))[:, 0]])).cuda()

    def tensor(name):
        data, scales, info = artifact.load_tensor(path, name)
        t = torch.from_numpy(np.array(data)).cuda()
        if info.bits == 16:
            return t.view(torch.bfloat16).double()
        if info.bits == 4:
            t = torch.stack((t & 15, t >> 4), dim=-1).view(info.rows, info.cols).to(torch.int16)
            t = torch.where(t > 7, t - 16, t)
        if scales is None:
            return t.double()
        return t.double() * torch.from_numpy(np.array(scales)).cuda().double().repeat_interleave(info.group, dim=1)

    def norm(x, name):
        if spec.norm == artifact.NORM_LAYER:
            x = x - x.mean(-1, keepdim=True)
        scaled = x / (x.square().mean(-1, keepdim=True) + np.float32(spec.epsilon)).sqrt() * tensor(name + ".weight")[0]
        return scaled + tensor(name + ".bias")[0] if spec.norm_bias else scaled

    def linear(x, name, bias):
        return x @ tensor(name + ".weight").T + (tensor(name + ".bias")[0] if bias else 0)

    def head_major(x, heads):
        return x.view(len(ids), heads, spec.head_dim).transpose(0, 1)

    embedding = tensor("model.embed_tokens.weight")
    x = embedding[ids]
    if spec.position == artifact.POS_LEARNED:
        x = x + tensor("model.position_embeddings.weight")[:len(ids)]
    exponent = np.arange(0, spec.head_dim, 2, dtype=np.float32) / np.float32(spec.head_dim)
    frequency = np.float32(1) / np.power(np.float64(spec.theta), exponent).astype(np.float32)
    angle = torch.from_numpy(np.arange(len(ids), dtype=np.float32)[:, None] * frequency[None, :]).double().cuda()
    for i in range(spec.layers):
        p = f"model.layers.{i}."
        normed = norm(x, p + "input_layernorm")
        q, k, v = (head_major(linear(normed, p + f"self_attn.{r}_proj", spec.attention_bias), n)
                   for r, n in (("q", spec.heads), ("k", spec.kv_heads), ("v", spec.kv_heads)))
        if spec.position == artifact.POS_ROPE:
            q, k = _rotate(q, angle.cos(), angle.sin()), _rotate(k, angle.cos(), angle.sin())
        x = x + linear(_exact_attention(q, k, v, 0, 0), p + "self_attn.o_proj", spec.o_bias)
        normed = norm(x, p + "post_attention_layernorm")
        up = linear(normed, p + "mlp.up_proj", spec.mlp_bias)
        if spec.gated:
            gate = linear(normed, p + "mlp.gate_proj", spec.mlp_bias)
            up = up * gate * torch.sigmoid(gate)
        else:
            up = torch.nn.functional.gelu(up, approximate="tanh")
        x = x + linear(up, p + "mlp.down_proj", spec.mlp_bias)
    return norm(x[case["prompt"] - 1:], "model.norm") @ tensor("lm_head.weight").T
