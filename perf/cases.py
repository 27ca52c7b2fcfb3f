"""The work this backend does for its users, as measured cases.

Each case is one pass through the public entry points (`HipBackend`,
`Lfm2Model`), in the order the LFM2 executor issues them:

- "linear":    one packed product.
- "head":      the end of a token pass: final norm, tied LM head, greedy choice.
- "ffn":       residual add + norm, gate/up products with SwiGLU, down product.
- "conv":      residual add + norm, in-projection, gated short convolution,
               out-projection.
- "attention": residual add + norm, q/k/v products, head norms with rotary,
               causal attention over a cache, output projection.
- "prefill":   a whole model's prompt pass from an empty prefix.
- "decode":    a whole model's greedy steps from a stored prefix.

All random values come from the seed.  Weights are N(0, 0.02) quantized by the
converter's rules; activations have per-channel gains and a few large
channels, as the residual stream of a trained model does.
"""
import math

import numpy as np
import torch

from runtime_amd import lfm2
from runtime_amd.backend import (CACHE, WEIGHT, CacheLength, GatedShortConvSpec, GqaSpec,
                                 HipBackend, PackedHeadSpec, RotarySpec)

HEAD_DIM = 64
CONV_WIDTH = 3
THETA = 1.0e6
EPSILON = 1.0e-5
VOCAB = 65536
NF4 = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
       -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
       0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
       0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0]
BITS = {"ternary": 2, "nf4": 4, "int8": 8}
# The formats a model's roles are stored in (embedding and head, convolution
# projections, attention projections, feed forward).
MODELS = {"350m": ("ternary", "ternary", "ternary", "ternary"),
          "1.2b": ("int8", "nf4", "nf4", "ternary")}


def listed():
    return [
        # The smallest block of a decode step: one token in the small model.
        {"name": "conv_1x1024_ternary", "kind": "conv", "rows": 1, "hidden": 1024,
         "format": "ternary"},
        # Choosing the next token of one sequence: norm, 134 MB head, argmax.
        {"name": "head_1x65536x2048_int8", "kind": "head", "rows": 1, "n": VOCAB, "k": 2048,
         "format": "int8"},
        # The feed forward of a few sequences (or drafted tokens) at once.
        {"name": "ffn_5x2048x8192_ternary", "kind": "ffn", "rows": 5, "hidden": 2048,
         "inter": 8192, "format": "ternary"},
        # One token's attention block late in a conversation.
        {"name": "attention_1x2048_past2047_nf4", "kind": "attention", "rows": 1, "hidden": 2048,
         "kv_heads": 8, "past": 2047, "format": "nf4"},
        # A short prompt of ragged length in a small model's feed forward.
        {"name": "ffn_346x1024x2560_nf4", "kind": "ffn", "rows": 346, "hidden": 1024,
         "inter": 2560, "format": "nf4"},
        # The commonest block of a prompt pass, ragged length.
        {"name": "conv_517x2048_nf4", "kind": "conv", "rows": 517, "hidden": 2048,
         "format": "nf4"},
        # A single eight-bit product over a medium prompt.
        {"name": "linear_512x8192x2048_int8", "kind": "linear", "rows": 512, "n": 8192,
         "k": 2048, "format": "int8"},
        # The feed forward of a long prompt: most of a prompt pass's time.
        {"name": "ffn_2048x2048x8192_ternary", "kind": "ffn", "rows": 2048, "hidden": 2048,
         "inter": 8192, "format": "ternary"},
        # Attention over a long prompt, causal from the first token.
        {"name": "attention_2048x2048_nf4", "kind": "attention", "rows": 2048, "hidden": 2048,
         "kv_heads": 8, "past": 0, "format": "nf4"},
        # Time to first token of the small model at a chat-sized prompt.
        {"name": "prefill_350m_128", "kind": "prefill", "model": "350m", "tokens": 128},
        # Time to first token of the large model at a document-sized prompt.
        {"name": "prefill_1.2b_2048", "kind": "prefill", "model": "1.2b", "tokens": 2048},
        # Greedy decoding of the large model behind that prompt.
        {"name": "decode_1.2b_2048_16", "kind": "decode", "model": "1.2b", "tokens": 2048,
         "steps": 16},
    ]


def _spread(rng, low, high):
    """An integer of [low, high], uniform over its logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    """One more case: decode, small-batch and prompt row counts alike."""
    kind = rng.choice(["linear", "linear", "head", "ffn", "ffn", "conv", "attention",
                       "attention", "prefill", "decode"])
    rows = _spread(rng, 1, 8) if rng.random() < 0.4 else _spread(rng, 9, 2048)
    fmt = rng.choice(["ternary", "nf4", "int8"])
    hidden = rng.choice([1024, 1024, 2048, 2048, 1536, 2560])
    if kind == "linear":
        k = 128 * _spread(rng, 4, 64)
        n = _spread(rng, 256, 16384)
        return {"kind": kind, "rows": max(rows, 9), "n": n, "k": k, "format": fmt}
    if kind == "head":
        return {"kind": kind, "rows": _spread(rng, 1, 8), "n": _spread(rng, 16384, VOCAB),
                "k": hidden, "format": fmt}
    if kind == "ffn":
        inter = 128 * _spread(rng, hidden // 64, hidden // 32)
        return {"kind": kind, "rows": rows, "hidden": hidden, "inter": inter, "format": fmt}
    if kind == "conv":
        return {"kind": kind, "rows": rows, "hidden": hidden, "format": fmt}
    if kind == "attention":
        heads = hidden // HEAD_DIM
        past = 0 if rng.random() < 0.3 else _spread(rng, 16, 2048)
        return {"kind": kind, "rows": rows, "hidden": hidden, "kv_heads": heads // rng.choice([2, 4]),
                "past": past, "format": fmt}
    model = rng.choice(["350m", "1.2b"])
    tokens = _spread(rng, 16, 2040)
    if kind == "prefill":
        return {"kind": kind, "model": model, "tokens": tokens}
    return {"kind": kind, "model": model, "tokens": tokens, "steps": _spread(rng, 4, 16)}


# ---- inputs ----------------------------------------------------------------

class _Source:
    """Seeded values, made on the GPU."""

    def __init__(self, seed):
        self.device = torch.device("cuda")
        self.generator = torch.Generator(self.device)
        self.generator.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.generator, device=self.device)

    def activations(self, rows, width):
        """Channels of different gains, one in 256 of them large."""
        gain = torch.exp(0.5 * self.normal(width))
        gain[::256] *= 16.0
        return self.normal(rows, width) * gain

    def norm_weight(self, width):
        return 1.0 + 0.1 * self.normal(width)

    def ids(self, count):
        return torch.randint(0, VOCAB, (count,), generator=self.generator, device=self.device)

    def packed(self, n, k, fmt):
        """(codes, scales) of an N(0, 0.02) matrix in one of the formats."""
        w = (0.02 * self.normal(n, k)).view(n, k // 128, 128)
        largest = w.abs().amax(dim=2)
        scale = (largest / 127.0 if fmt == "int8" else largest).half().float()
        scaled = w / scale.unsqueeze(2)
        if fmt == "int8":
            codes = torch.clamp(torch.round(scaled), -127, 127).to(torch.int8).view(torch.uint8)
        elif fmt == "nf4":
            levels = torch.tensor(NF4, device=self.device)
            codes = torch.bucketize(scaled, (levels[1:] + levels[:-1]) / 2).to(torch.uint8)
        else:
            codes = (torch.clamp(torch.round(scaled), -1, 1) + 1).to(torch.uint8)
        codes = codes.view(n, k)
        per_byte = 8 // BITS[fmt]
        if per_byte > 1:
            codes = codes.view(n, k // per_byte, per_byte)
            shifted = [codes[:, :, i] << (i * BITS[fmt]) for i in range(per_byte)]
            codes = shifted[0]
            for part in shifted[1:]:
                codes = codes | part
        return codes, scale


def _values(case, seed):
    """The case's inputs as torch tensors, by name; packed weights as pairs."""
    s, v = _Source(seed), {}
    kind = case["kind"]
    if kind == "linear":
        v["x"] = s.activations(case["rows"], case["k"])
        v["w"] = s.packed(case["n"], case["k"], case["format"])
    elif kind == "head":
        v["x"] = s.activations(case["rows"], case["k"])
        v["norm"] = s.norm_weight(case["k"])
        v["w"] = s.packed(case["n"], case["k"], case["format"])
    elif kind in ("ffn", "conv", "attention"):
        rows, h, fmt = case["rows"], case["hidden"], case["format"]
        v["left"], v["right"] = s.activations(rows, h), s.normal(rows, h)
        v["norm"] = s.norm_weight(h)
        if kind == "ffn":
            v["gate"] = s.packed(case["inter"], h, fmt)
            v["up"] = s.packed(case["inter"], h, fmt)
            v["down"] = s.packed(h, case["inter"], fmt)
        elif kind == "conv":
            v["in"] = s.packed(3 * h, h, fmt)
            v["taps"] = 0.5 * s.normal(h, CONV_WIDTH)
            v["history"] = s.normal(CONV_WIDTH - 1, h)
            v["out"] = s.packed(h, h, fmt)
        else:
            kv = case["kv_heads"] * HEAD_DIM
            v["q"] = s.packed(h, h, fmt)
            v["k"], v["v"] = s.packed(kv, h, fmt), s.packed(kv, h, fmt)
            v["o"] = s.packed(h, h, fmt)
            v["q_norm"], v["k_norm"] = s.norm_weight(HEAD_DIM), s.norm_weight(HEAD_DIM)
            capacity = case["past"] + rows
            v["keys"], v["values"] = s.normal(capacity, kv), s.normal(capacity, kv)
    else:
        cfg = _config(case)
        names = ("embedding", "conv", "attention", "ffn")
        formats = dict(zip(names, MODELS[case["model"]]))
        v["ids"] = s.ids(case["tokens"])
        for role, layer, shape, matmul in lfm2.role_shapes(cfg):
            if matmul:
                value = s.packed(*shape, formats[_group(role)])
            elif role == lfm2.CONV_KERNEL:
                value = 0.5 * s.normal(*shape)
            else:
                value = s.norm_weight(*shape)
            v[role, layer] = value
    return v


def _group(role):
    if role == lfm2.TOKEN_EMBEDDING:
        return "embedding"
    if role in (lfm2.CONV_IN, lfm2.CONV_OUT):
        return "conv"
    if role in (lfm2.QUERY, lfm2.KEY, lfm2.VALUE, lfm2.OUTPUT):
        return "attention"
    return "ffn"


def _config(case):
    make = lfm2.lfm2_350m if case["model"] == "350m" else lfm2.lfm2_1_2b
    return make(max_tokens=case["tokens"] + case.get("steps", 0))


_SHARED = []


def _backend():
    """The process's one backend instance (and stream)."""
    if not _SHARED:
        _SHARED.append(HipBackend(0))
    return _SHARED[0]


class Outputs(dict):
    """A pass's results by name.  They stay in the backend's buffers, where a
    program's next operation would read them; looking one up reads it back.
    The state that owns the buffers lives as long as its outputs."""

    def __init__(self, state, *names):
        super().__init__((name, state[name]) for name in names)
        self.state = state

    def __getitem__(self, name):
        return _backend().read(super().__getitem__(name))


def _upload(value, cls):
    array = value.cpu().numpy()
    if array.dtype == np.uint8:
        return _backend().upload_u8_classified(array.shape, array, cls)
    return _backend().upload_f32_classified(array.shape, array, cls)


def prepare(case, seed):
    backend = _backend()
    values = _values(case, seed)
    if case["kind"] in ("prefill", "decode"):
        model = lfm2.Lfm2Model(backend, _config(case))
        ids = values.pop("ids").cpu().numpy()
        for (role, layer), value in values.items():
            parts = value if isinstance(value, tuple) else (value,)
            model.set_weight(role, layer, *(_upload(part, WEIGHT) for part in parts))
        state = {"model": model, "ids": ids, "logits": model.logits}
        if case["kind"] == "decode":
            model.append(ids)
            state["prefix"] = model.snapshot()
            state["chosen"] = backend.allocate_f32((case["steps"],))
        return {"case": case, **state}
    state = {}
    for name, value in values.items():
        if isinstance(value, tuple):
            state[name] = tuple(_upload(part, WEIGHT) for part in value)
            backend.prepare_packed(*state[name])
        else:
            cls = CACHE if name in ("keys", "values", "history") else WEIGHT
            state[name] = _upload(value, cls)
    # Intermediate and output rows, allocated once as the executor does.
    rows = case["rows"]
    if case["kind"] == "linear":
        widths = {"y": case["n"]}
    elif case["kind"] == "head":
        widths = {"normed": case["k"], "logits": case["n"]}
    else:
        h = case["hidden"]
        widths = {"sum": h, "normed": h, "y": h}
        if case["kind"] == "ffn":
            widths.update(gated=case["inter"], lifted=case["inter"])
        elif case["kind"] == "conv":
            widths.update(projection=3 * h, convolved=h)
        else:
            kv = case["kv_heads"] * HEAD_DIM
            widths.update(query=h, key=kv, value=kv, query_rope=h, key_rope=kv, attended=h)
    for name, width in widths.items():
        state[name] = backend.allocate_f32((rows, width))
    if case["kind"] == "head":
        state["token"] = backend.allocate_f32((rows,))
    return {"case": case, **state}


def run(state):
    backend, case, s = _backend(), state["case"], state
    kind = case["kind"]
    if kind == "linear":
        backend.packed_linear(s["y"], s["x"], *s["w"])
        return Outputs(s, "y")
    if kind == "head":
        backend.row_rms_norm(s["normed"], s["x"], s["norm"], EPSILON)
        backend.packed_linear(s["logits"], s["normed"], *s["w"])
        backend.argmax(s["token"], s["logits"])
        return Outputs(s, "logits", "token")
    if kind == "prefill":
        s["model"].reset()
        s["model"].append(s["ids"])
        return Outputs(s, "logits")
    if kind == "decode":
        s["model"].restore(s["prefix"])
        s["model"].generate(case["steps"], s["chosen"])
        return Outputs(s, "logits", "chosen")
    backend.add_row_rms_norm(s["sum"], s["normed"], s["left"], s["right"], s["norm"], EPSILON)
    if kind == "ffn":
        # From 96 rows the executor forms SwiGLU in the gate/up product.
        if case["rows"] >= 96:
            backend.packed_swiglu_pair(s["gated"], s["normed"], *s["gate"], *s["up"])
            backend.packed_linear(s["y"], s["gated"], *s["down"])
        else:
            backend.packed_linear_pair(s["gated"], s["lifted"], s["normed"], *s["gate"], *s["up"])
            backend.packed_swiglu_linear(s["y"], s["gated"], s["lifted"], *s["down"])
        return Outputs(s, "sum", "y")
    if kind == "conv":
        backend.packed_linear(s["projection"], s["normed"], *s["in"])
        backend.gated_short_convolution(s["convolved"], s["projection"], s["taps"], s["history"],
                                        GatedShortConvSpec(case["hidden"], CONV_WIDTH))
        backend.packed_linear(s["y"], s["convolved"], *s["out"])
        return Outputs(s, "sum", "y", "history")
    heads, kv_heads, past = case["hidden"] // HEAD_DIM, case["kv_heads"], case["past"]
    backend.packed_linear(s["query"], s["normed"], *s["q"])
    backend.packed_linear_pair(s["key"], s["value"], s["normed"], *s["k"], *s["v"])
    backend.qk_norm_rope(s["query_rope"], s["key_rope"], s["query"], s["key"], s["q_norm"],
                         s["k_norm"], range(past, past + case["rows"]),
                         RotarySpec(PackedHeadSpec(heads, HEAD_DIM), THETA),
                         PackedHeadSpec(kv_heads, HEAD_DIM), EPSILON)
    backend.causal_gqa(s["attended"], s["query_rope"], s["key_rope"], s["value"], s["keys"],
                       s["values"], CacheLength(past), GqaSpec(heads, kv_heads, HEAD_DIM))
    backend.packed_linear(s["y"], s["attended"], *s["o"])
    return Outputs(s, "sum", "y", "keys", "values")


# ---- what a pass cannot do without ------------------------------------------

def _product(rows, n, k, fmt):
    """(weight bytes, flops): codes and binary16 group scales, 2 M N K."""
    return n * k * BITS[fmt] / 8 + n * k / 128 * 2, 2.0 * rows * n * k


def _pairs(rows, past):
    """(query, key) pairs of causal attention."""
    return rows * past + rows * (rows + 1) / 2


def work(case):
    kind = case["kind"]
    if kind in ("linear", "head"):
        rows, n, k = case["rows"], case["n"], case["k"]
        weight, flops = _product(rows, n, k, case["format"])
        extra = 4 * k if kind == "head" else 0
        return {"bytes": weight + 4.0 * rows * (n + k) + extra, "flops": flops}
    if kind in ("ffn", "conv", "attention"):
        rows, h, fmt = case["rows"], case["hidden"], case["format"]
        moved, flops = 4.0 * rows * h * 4 + 4 * h, 0.0  # left, right, sum, y; the norm
        if kind == "ffn":
            shapes = [(case["inter"], h), (case["inter"], h), (h, case["inter"])]
        elif kind == "conv":
            shapes = [(3 * h, h), (h, h)]
            moved += 4.0 * h * (CONV_WIDTH + 2 * (CONV_WIDTH - 1))
            flops += 2.0 * rows * h * (CONV_WIDTH + 2)
        else:
            kv = case["kv_heads"] * HEAD_DIM
            shapes = [(h, h), (kv, h), (kv, h), (h, h)]
            moved += 4.0 * 2 * kv * (case["past"] + rows) + 8 * HEAD_DIM
            flops += 4.0 * _pairs(rows, case["past"]) * h
        for n, k in shapes:
            weight, products = _product(rows, n, k, fmt)
            moved, flops = moved + weight, flops + products
        return {"bytes": moved, "flops": flops}
    cfg = _config(case)
    formats = dict(zip(("embedding", "conv", "attention", "ffn"), MODELS[case["model"]]))
    tokens, steps = case["tokens"], case.get("steps", 0)
    moved = flops = 0.0
    rows = steps if kind == "decode" else tokens
    reads = steps if kind == "decode" else 1
    last = len(cfg.layers) - 1
    for role, layer, shape, matmul in lfm2.role_shapes(cfg):
        if not matmul:
            moved += 4.0 * reads * math.prod(shape)
            continue
        # Only the last row passes the last layer's feed forward and the head.
        ends = role == lfm2.TOKEN_EMBEDDING or (layer == last and _group(role) == "ffn")
        count = reads if ends else rows
        weight, products = _product(count, *shape, formats[_group(role)])
        moved, flops = moved + reads * weight, flops + products
    attention = sum(1 for layer in cfg.layers if layer == lfm2.ATTENTION)
    if kind == "decode":
        flops += attention * 4.0 * _pairs(steps, tokens) * cfg.hidden
        moved += attention * 8.0 * cfg.kv_width * _pairs(steps, tokens)
    else:
        flops += attention * 4.0 * _pairs(tokens, 0) * cfg.hidden
        moved += attention * 8.0 * cfg.kv_width * tokens
    return {"bytes": moved + 4.0 * reads * cfg.vocab, "flops": flops}


def tolerance(case):
    # 32-bit sums throughout: single blocks measure up to 1.1e-6 from 64 bits.
    # A whole model carries one layer's rounding through all that follow (up
    # to 4e-6 measured).
    return {"rel": 2e-5} if case["kind"] in ("prefill", "decode") else {"rel": 5e-6}


# ---- the same in 64 bits ------------------------------------------------------

def _dense(packed, fmt):
    """The stored matrix's values."""
    codes, scale = packed
    n = codes.shape[0]
    if fmt == "int8":
        level = codes.view(torch.int8).double()
    else:
        bits = BITS[fmt]
        parts = [(codes >> (i * bits)) & ((1 << bits) - 1) for i in range(8 // bits)]
        code = torch.stack(parts, dim=2).reshape(n, -1)
        level = (torch.tensor(NF4, device=codes.device).double()[code.long()] if fmt == "nf4"
                 else code.double() - 1.0)
    return (level.view(n, -1, 128) * scale.double().unsqueeze(2)).view(n, -1)


def _rms(x, weight):
    epsilon = float(np.float32(EPSILON))
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + epsilon) * weight.double()


def _rotate(x, positions):
    # The rotation is defined on 32-bit frequencies and angles.
    half = x.shape[-1] // 2
    exponent = -2.0 * torch.arange(half, device=x.device).double() / x.shape[-1]
    frequency = torch.pow(torch.full_like(exponent, float(np.float32(THETA))), exponent).float()
    angle = (positions.float()[:, None, None] * frequency).double()
    cosine, sine = torch.cos(angle), torch.sin(angle)
    first, second = x[..., :half], x[..., half:]
    return torch.cat([first * cosine - second * sine, second * cosine + first * sine], dim=-1)


def _attend(query, key, value, past):
    """Causal attention of [rows, heads, d] over [past + rows, kv_heads, d]."""
    rows, heads, d = query.shape
    group = heads // key.shape[1]
    hidden = (torch.arange(key.shape[0], device=key.device)[None, :] >
              past + torch.arange(rows, device=key.device)[:, None])
    out = torch.empty_like(query)
    for i in range(heads):
        scores = query[:, i] @ key[:, i // group].T.contiguous() / math.sqrt(d)
        scores = scores.masked_fill(hidden, -math.inf)
        out[:, i] = torch.softmax(scores, dim=1) @ value[:, i // group].contiguous()
    return out.reshape(rows, heads * d)


def _attention(normed, w, keys, values, past, q_norm, k_norm):
    """(the block's output, all keys, all values); w gives q, k, v, o."""
    rows = normed.shape[0]
    positions = torch.arange(past, past + rows, device=normed.device)
    split = lambda t: t.reshape(t.shape[0], -1, HEAD_DIM)  # noqa: E731
    query = _rotate(_rms(split(normed @ w("q").T), q_norm), positions)
    key = _rotate(_rms(split(normed @ w("k").T), k_norm), positions)
    keys = torch.cat([keys[:past], key.reshape(rows, -1)])
    values = torch.cat([values[:past], normed @ w("v").T])
    return _attend(query, split(keys), split(values), past) @ w("o").T, keys, values


def _conv(projection, taps, history):
    """(the gated short convolution's output, the new history)."""
    h = projection.shape[1] // 3
    gated = torch.cat([history, projection[:, :h] * projection[:, 2 * h:]])
    rows = projection.shape[0]
    mixed = sum(gated[i:i + rows] * taps[:, i].double() for i in range(CONV_WIDTH))
    return mixed * projection[:, h:2 * h], gated[rows:]


def _silu(x):
    return x / (1.0 + torch.exp(-x))


class _Model:
    """The token pass in 64 bits, with its prefix state."""

    def __init__(self, cfg, model, values):
        formats = dict(zip(("embedding", "conv", "attention", "ffn"), MODELS[model]))
        self.cfg, self.length = cfg, 0
        self.w = {at: _dense(v, formats[_group(at[0])]) if isinstance(v, tuple) else v.double()
                  for at, v in values.items()}
        zeros = lambda rows, width: torch.zeros(rows, width, dtype=torch.float64,  # noqa: E731
                                                device="cuda")
        self.state = [zeros(CONV_WIDTH - 1, cfg.hidden) if kind == lfm2.CONV
                      else (zeros(0, cfg.kv_width), zeros(0, cfg.kv_width))
                      for kind in cfg.layers]

    def append(self, ids):
        x = self.w[lfm2.TOKEN_EMBEDDING, 0][ids]
        for i, kind in enumerate(self.cfg.layers):
            w = lambda role: self.w[role, i]  # noqa: E731
            normed = _rms(x, w(lfm2.OPERATOR_NORM))
            if kind == lfm2.CONV:
                mixed, self.state[i] = _conv(normed @ w(lfm2.CONV_IN).T, w(lfm2.CONV_KERNEL),
                                             self.state[i])
                op = mixed @ w(lfm2.CONV_OUT).T
            else:
                roles = {"q": lfm2.QUERY, "k": lfm2.KEY, "v": lfm2.VALUE, "o": lfm2.OUTPUT}
                op, *self.state[i] = _attention(normed, lambda name: w(roles[name]),
                                                *self.state[i], self.length,
                                                w(lfm2.QUERY_NORM), w(lfm2.KEY_NORM))
            x = x + op
            normed = _rms(x, w(lfm2.FFN_NORM))
            hidden = _silu(normed @ w(lfm2.FFN_W1).T) * (normed @ w(lfm2.FFN_W3).T)
            x = x + hidden @ w(lfm2.FFN_W2).T
        self.length += len(ids)
        return _rms(x[-1:], self.w[lfm2.EMBEDDING_NORM, 0]) @ self.w[lfm2.TOKEN_EMBEDDING, 0].T


def exact(case, seed):
    values, kind = _values(case, seed), case["kind"]
    host = lambda **outputs: {n: t.cpu().numpy() for n, t in outputs.items()}  # noqa: E731
    if kind in ("prefill", "decode"):
        ids = values.pop("ids")
        model = _Model(_config(case), case["model"], values)
        logits = model.append(ids)
        if kind == "prefill":
            return host(logits=logits)
        chosen = []
        for _ in range(case["steps"]):
            chosen.append(logits.argmax(dim=1))
            logits = model.append(chosen[-1])
        return host(logits=logits, chosen=torch.cat(chosen).double())
    fmt = case["format"]
    if kind == "linear":
        return host(y=values["x"].double() @ _dense(values["w"], fmt).T)
    if kind == "head":
        logits = _rms(values["x"].double(), values["norm"]) @ _dense(values["w"], fmt).T
        return host(logits=logits, token=logits.argmax(dim=1).double())
    total = values["left"].double() + values["right"].double()
    normed = _rms(total, values["norm"])
    w = lambda name: _dense(values[name], fmt)  # noqa: E731
    if kind == "ffn":
        hidden = _silu(normed @ w("gate").T) * (normed @ w("up").T)
        return host(sum=total, y=hidden @ w("down").T)
    if kind == "conv":
        mixed, history = _conv(normed @ w("in").T, values["taps"], values["history"].double())
        return host(sum=total, y=mixed @ w("out").T, history=history)
    y, keys, vals = _attention(normed, w, values["keys"].double(), values["values"].double(),
                               case["past"], values["q_norm"], values["k_norm"])
    return host(sum=total, y=y, keys=keys, values=vals)
