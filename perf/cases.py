"""The work that programs built on this framework give it, as cases to time.

Each case is one pass of a caller's program through the public entry points
(`HipRuntime`, `NeuralOps`), over device buffers that the program owns:

    decode    one decode step of a Gemma-like model: the token and PLE gathers,
              then every layer's fused ops, captured once and replayed
    token     one decode token of a Llama-like model (f32), captured and replayed
    prefill   one prefill chunk of a Gemma-like model with its KV appends
    half      the FP16 layer ops of a Llama-like prefill
    gather    the embedding and PLE gathers of a chunk from full-size tables
    project   one decode token's quantised projections, captured and replayed
    logits    the decode tail: soft cap and greedy argmax over a batch of rows
    host      the host-slice operators, from host arrays to host arrays

The GEMM and attention results between the ops are not this framework's; they
are inputs here, drawn N(0, 1) as after a projection, with norm weights
N(1, 0.1).  Widths are those of the benchmark configurations and tests
(hidden 576 to 8192, head_dim 64 to 512) or generic ones in between.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from atlas_amd import ATLAS_REDUCTION_AUTO, HipRuntime, NeuralOps

EPS = 1e-6
SQRT_HALF = float(np.float32(1.0) / np.sqrt(np.float32(2.0)))
PLE_SCALE = 16.0  # sqrt(256)
LOGIT_CAP = 30.0


def listed():
    return [
        # One sequence, one token through 35 layers: the smallest launches, where latency is everything.
        {"name": "decode_1", "kind": "decode", "batch": 1, "layers": 35, "hidden": 1536, "q_heads": 8, "head_dim": 256,
         "ffn": 6144, "vocab": 32768},
        # The batched decode step of the benchmark: 256 sequences, one row per CU.
        {"name": "decode_256", "kind": "decode", "batch": 256, "layers": 35, "hidden": 1536, "q_heads": 8,
         "head_dim": 256, "ffn": 6144, "vocab": 32768},
        # A small batch of a wider model.
        {"name": "decode_24_wide", "kind": "decode", "batch": 24, "layers": 16, "hidden": 4096, "q_heads": 16,
         "head_dim": 256, "ffn": 16384, "vocab": 32768},
        # The smallest model: a 30-layer, 576-wide f32 decode token.
        {"name": "token_576", "kind": "token", "layers": 30, "hidden": 576, "q_heads": 9, "kv_heads": 3,
         "head_dim": 64, "ffn": 1536, "vocab": 49152, "capacity": 2048},
        # The reference executor's prefill chunk: 512 tokens, Q8_0 cache.
        {"name": "prefill_512", "kind": "prefill", "tokens": 512, "layers": 5, "hidden": 1536, "q_heads": 8,
         "head_dim": 256, "ffn": 6144, "vocab": 32768, "cache": "q8_0"},
        # A long prompt at once: the benchmark's 4096 tokens, Q4_0 cache.
        {"name": "prefill_4096", "kind": "prefill", "tokens": 4096, "layers": 3, "hidden": 1536, "q_heads": 8,
         "head_dim": 256, "ffn": 6144, "vocab": 32768, "cache": "q4_0"},
        # A ragged chunk of a wider model with more heads, f32 cache.
        {"name": "prefill_1000_wide", "kind": "prefill", "tokens": 1000, "layers": 2, "hidden": 4096, "q_heads": 16,
         "head_dim": 256, "ffn": 16384, "vocab": 32768, "cache": "f32"},
        # FP16 storage: the benchmark's 2048-token Llama-like prefill.
        {"name": "half_2048", "kind": "half", "tokens": 2048, "layers": 4, "hidden": 2048, "heads": 32, "kv_heads": 32,
         "head_dim": 64, "ffn": 8192},
        # Every table format at the benchmark's gather: 4096 tokens of a 262144-row vocabulary.
        {"name": "gather_4096", "kind": "gather", "tokens": 4096, "hidden": 1536, "ple_layers": 35, "vocab": 262144},
        # One decode token's Q4_0 and F16 projections through 35 layers.
        {"name": "project_1536", "kind": "project", "layers": 35, "hidden": 1536, "q_width": 2048, "kv_width": 256,
         "ffn": 6144},
        # The decode tail of the batched step over the full vocabulary.
        {"name": "logits_256", "kind": "logits", "rows": 256, "vocab": 262144},
        # A program that holds its activations on the host and calls the operators one by one.
        {"name": "host_128", "kind": "host", "tokens": 128, "hidden": 576, "ffn": 1536},
    ]


LARGEST_BYTES = 2.2e9  # no drawn case moves more than the largest listed one


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "token", "prefill", "prefill", "half", "gather", "project", "logits", "host"])
    hidden = rng.choice([576, 768, 1024, 1536, 2048, 2304, 2560, 3072, 4096, 5120, 8192])
    if kind == "decode":
        case = {"batch": _log(rng, 1, 256), "layers": rng.randint(4, 35), "hidden": hidden,
                "q_heads": rng.choice([4, 8, 12, 16, 24, 32]), "head_dim": rng.choice([64, 128, 256, 256, 512]),
                "ffn": hidden * rng.choice([3, 4]), "vocab": 32768}
        shrink = "batch"
    elif kind == "token":
        case = {"layers": rng.randint(8, 32), "hidden": hidden, "q_heads": 0, "kv_heads": 0,
                "head_dim": rng.choice([64, 128]), "ffn": hidden * rng.choice([3, 4]), "vocab": 49152,
                "capacity": rng.choice([128, 512, 1024])}
        case["q_heads"] = max(2, hidden // case["head_dim"])
        case["kv_heads"] = max(1, min(case["q_heads"] // 4, 4096 // case["head_dim"]))
        shrink = "layers"
    elif kind == "prefill":
        case = {"tokens": _log(rng, 9, 4096), "layers": rng.randint(1, 3), "hidden": hidden,
                "q_heads": rng.choice([4, 8, 12, 16, 24]), "head_dim": rng.choice([64, 128, 256, 256, 512]),
                "ffn": hidden * rng.choice([3, 4]), "vocab": 32768, "cache": rng.choice(["f32", "q8_0", "q4_0"])}
        shrink = "tokens"
    elif kind == "half":
        case = {"tokens": _log(rng, 9, 4096), "layers": rng.randint(1, 4), "hidden": hidden, "heads": 0,
                "kv_heads": 0, "head_dim": rng.choice([64, 128]), "ffn": hidden * rng.choice([3, 4])}
        case["heads"] = max(2, hidden // case["head_dim"])
        case["kv_heads"] = rng.choice([case["heads"], max(1, case["heads"] // 4)])
        shrink = "tokens"
    elif kind == "gather":
        case = {"tokens": _log(rng, 1, 4096), "hidden": hidden - hidden % 256, "ple_layers": rng.randint(8, 42),
                "vocab": rng.choice([32768, 49152, 131072])}
        shrink = "tokens"
    elif kind == "project":
        hidden = min(hidden, 4096)
        case = {"layers": rng.randint(4, 35), "hidden": hidden, "q_width": rng.choice([576, 1024, 2048, 4096]),
                "kv_width": rng.choice([192, 256, 512, 1024]), "ffn": hidden * rng.choice([3, 4])}
        shrink = "layers"
    elif kind == "logits":
        case = {"rows": _log(rng, 1, 256), "vocab": rng.choice([32000, 32001, 49152, 50257, 128256, 151936, 262144])}
        shrink = "rows"
    else:
        case = {"tokens": _log(rng, 1, 2048), "hidden": min(hidden, 2560), "ffn": min(hidden, 2560) * 3}
        shrink = "tokens"
    case = {"kind": kind, **case}
    while work(case)["bytes"] > LARGEST_BYTES:
        case[shrink] = max(1, case[shrink] * 3 // 4)
    return case


def prepare(case, seed):
    state = _KINDS[case["kind"]].prepare(case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    return state.run()


def work(case):
    return _KINDS[case["kind"]].work(case)


def tolerance(case):
    return _KINDS[case["kind"]].tolerance(case)


def exact(case, seed):
    return _KINDS[case["kind"]].exact(case, seed)


# ---------------------------------------------------------------------------
# what the programs share
# ---------------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _runtime():
    return HipRuntime(0, ATLAS_REDUCTION_AUTO)


@functools.lru_cache(maxsize=None)
def _neural_ops():
    return NeuralOps(0)


class _Program:
    """A caller's program: the calls of one pass, with what they read and write; captured into a graph or issued one by one."""

    def __init__(self, calls, outputs, keep, capture):
        self.rt, self.calls, self.outputs, self.keep, self.graph = _runtime(), calls, outputs, keep, None
        if capture:
            torch.cuda.synchronize()
            self.rt.graph_begin()
            try:
                self._issue()
            finally:
                self.graph = self.rt.graph_end()

    def _issue(self):
        for call, args in self.calls:
            call(*args)

    def run(self):
        if self.graph is not None:
            self.rt.graph_launch(self.graph)
        else:
            self._issue()
        return self.outputs

    def __del__(self):
        if self.graph is not None and self.rt.ctx:
            self.rt.graph_destroy(self.graph)


def _p(t):
    return t.data_ptr()


def _zeros(*shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype, device="cuda")


class _Draw:
    """Inputs from a seed, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, mean=0.0, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda").mul_(std).add_(mean)

    def weight(self, *shape):
        return self.normal(*shape, mean=1.0, std=0.1)

    def uniform(self, low, high, *shape):
        return torch.rand(shape, generator=self.g, device="cuda") * (high - low) + low

    def ints(self, low, high, *shape):
        return torch.randint(low, high, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def blocks(self, rows, width, fmt, std=None):
        """A table of `rows` packed rows: random codes, f16 scales of the benchmark's ranges (or for weights of about `std`)."""
        values, size, at, low, high = {"q4_0": (32, 18, 0, 0.001, 0.05), "q8_0": (32, 34, 0, 0.001, 0.05),
                                       "q6_k": (256, 210, 208, 1e-4, 2e-3)}[fmt]
        if std is not None:
            low, high = 0.1 * std, 0.3 * std
        n = width // values
        t = torch.randint(0, 256, (rows, n, size), generator=self.g, device="cuda", dtype=torch.uint8)
        d = self.uniform(low, high, rows, n).to(torch.float16)
        t[:, :, at:at + 2] = d.view(torch.uint8).reshape(rows, n, 2)
        return t.reshape(rows, n * size)

    def rope(self, positions, pairs, theta):
        p = torch.arange(pairs, device="cuda", dtype=torch.float32)
        angle = positions.to(torch.float32)[:, None] / theta ** (p / pairs)[None, :]
        return torch.cos(angle).contiguous(), torch.sin(angle).contiguous()


def _row_bytes(width, fmt):
    return {"f32": width * 4, "q4_0": width // 32 * 18, "q8_0": width // 32 * 34, "q6_k": width // 256 * 210}[fmt]


def _unpack(rows, fmt):
    """Packed rows in float64."""
    n = rows.shape[0]
    size = {"q4_0": 18, "q8_0": 34, "q6_k": 210}[fmt]
    b = rows.reshape(n, -1, size)
    at = 208 if fmt == "q6_k" else 0
    d = b[:, :, at:at + 2].contiguous().view(torch.float16).to(torch.float64)
    if fmt == "q4_0":
        q = b[:, :, 2:]
        return ((torch.cat([q & 15, q >> 4], 2).to(torch.float64) - 8.0) * d).reshape(n, -1)
    if fmt == "q8_0":
        return (b[:, :, 2:].contiguous().view(torch.int8).to(torch.float64) * d).reshape(n, -1)
    ql, qh, sc = b[:, :, :128], b[:, :, 128:192], b[:, :, 192:208].contiguous().view(torch.int8).to(torch.float64)
    parts = []
    for half in range(2):
        lo, hi = ql[:, :, 64 * half:64 * half + 64], qh[:, :, 32 * half:32 * half + 32]
        for st in range(4):
            nib = lo[:, :, 32 * (st & 1):32 * (st & 1) + 32] >> (4 if st >= 2 else 0)
            code = (nib & 15) | (((hi >> (2 * st)) & 3) << 4)
            s = sc[:, :, 8 * half + 2 * st:8 * half + 2 * st + 2].repeat_interleave(16, 2)
            parts.append((code.to(torch.float64) - 32.0) * s)
    return (torch.cat(parts, 2) * d).reshape(n, -1)


def _norm64(x, w, eps):
    x = x.double()
    y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)
    return y if w is None else y * w.double()


def _gelu64(x):
    x = x.double()
    return 0.5 * x * (1.0 + torch.tanh(0.7978845608 * (x + 0.044715 * x * x * x)))


def _rope64(x, cos, sin):
    """Half-split rotation of x [tokens, heads, head_dim]."""
    half = x.shape[-1] // 2
    a, b, c, s = x[..., :half], x[..., half:], cos.double()[:, None, :], sin.double()[:, None, :]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _qk_norm_rope64(q, k, qw, kw, cos, sin, heads):
    t, d = k.shape
    both = torch.cat([_norm64(q.reshape(t, heads, d), qw, EPS), _norm64(k.reshape(t, 1, d), kw, EPS)], 1)
    both = _rope64(both, cos, sin)
    return both[:, :heads].reshape(t, heads * d), both[:, heads]


# ---------------------------------------------------------------------------
# decode: embed, PLE chain, then per layer QK-norm + RoPE, the two residual
# epilogues around GeGLU, the PLE gate product and the PLE epilogue
# ---------------------------------------------------------------------------


class _Decode:
    PLE = 256

    @classmethod
    def inputs(cls, c, seed):
        d = _Draw(seed)
        B, L, H, QH, D, F, V, W = (c["batch"], c["layers"], c["hidden"], c["q_heads"], c["head_dim"], c["ffn"],
                                   c["vocab"], cls.PLE)
        positions = d.ints(0, 131072, B)
        return {
            "tokens": d.blocks(V, H, "q4_0"), "ple_table": d.blocks(V, L * W, "q4_0"), "ids": d.ints(0, V, B),
            "ple_in": d.normal(B, L * W), "rope": [d.rope(positions, D // 2, theta) for theta in (1e4, 1e6)],
            "q": d.normal(L, B, QH * D), "k": d.normal(L, B, D), "qw": d.weight(L, D), "kw": d.weight(L, D),
            "attn": d.normal(L, B, H), "attn_w": d.weight(L, H), "gate": d.normal(L, B, F), "up": d.normal(L, B, F),
            "down": d.normal(L, B, H), "ffn_w": d.weight(L, H), "ple_gate": d.normal(L, B, W),
            "ple_out": d.normal(L, B, H), "ple_w": d.weight(L, H), "scale": d.uniform(0.5, 1.5, L),
        }

    @classmethod
    def prepare(cls, c, seed):
        B, L, H, QH, D, F, V, W = (c["batch"], c["layers"], c["hidden"], c["q_heads"], c["head_dim"], c["ffn"],
                                   c["vocab"], cls.PLE)
        i, rt = cls.inputs(c, seed), _runtime()
        o = {"state": _zeros(B, H), "ple": _zeros(B, L * W), "q": _zeros(L, B, QH * D), "k": _zeros(L, B, D),
             "ffn": _zeros(L, B, F), "gated": _zeros(L, B, W)}
        state = _p(o["state"])
        calls = [(rt.embed_q4_0, (_p(i["tokens"]), _p(i["ids"]), state, V, H, B, float(np.sqrt(np.float32(H))))),
                 (rt.ple_q4_0, (_p(i["ple_table"]), _p(i["ids"]), _p(i["ple_in"]), _p(o["ple"]), V, L, W, B, PLE_SCALE,
                                SQRT_HALF))]
        for n in range(L):
            cos, sin = i["rope"][n % 5 == 4]  # every fifth layer is global
            calls += [
                (rt.qk_norm_rope, (_p(i["q"][n]), _p(i["k"][n]), _p(i["qw"][n]), _p(i["kw"][n]), _p(cos), _p(sin),
                                   _p(o["q"][n]), _p(o["k"][n]), B, QH, 1, D, D // 2, EPS)),
                (rt.rms_norm_residual, (_p(i["attn"][n]), _p(i["attn_w"][n]), state, None, state, B, H, EPS)),
                (rt.geglu, (_p(i["gate"][n]), _p(i["up"][n]), _p(o["ffn"][n]), B * F)),
                (rt.rms_norm_residual, (_p(i["down"][n]), _p(i["ffn_w"][n]), state, None, state, B, H, EPS)),
                (rt.geglu_offset, (_p(i["ple_gate"][n]), _p(o["ple"]), _p(o["gated"][n]), n * W, L * W, W, B)),
                (rt.rms_norm_add_scale, (_p(i["ple_out"][n]), _p(i["ple_w"][n]), state, _p(i["scale"][n:]), B, H, EPS)),
            ]
        return _Program(calls, o, i, capture=True)

    @classmethod
    def work(cls, c):
        B, L, H, QH, D, F, W = c["batch"], c["layers"], c["hidden"], c["q_heads"], c["head_dim"], c["ffn"], cls.PLE
        once = B * (_row_bytes(H, "q4_0") + 4 * H + _row_bytes(L * W, "q4_0") + 8 * L * W + 4)
        layer = 4 * (2 * B * (QH + 1) * D + B * D + 2 * D + 3 * (3 * B * H + H) + 3 * B * F + 3 * B * W)
        return {"bytes": once + L * layer, "flops": L * B * (8 * (QH + 1) * D + 18 * H + 40 * F + 40 * W)}

    @classmethod
    def tolerance(cls, c):
        return {"rel": 1.6e-6, "max": 2e-5}  # f32 throughout; measured 5e-8 to 4.1e-7 from float64

    @classmethod
    def exact(cls, c, seed):
        B, L, H, W, i = c["batch"], c["layers"], c["hidden"], cls.PLE, cls.inputs(c, seed)
        ids = i["ids"].long()
        state = _unpack(i["tokens"][ids], "q4_0") * float(np.sqrt(np.float32(H)))
        ple = (_unpack(i["ple_table"][ids], "q4_0") * PLE_SCALE + i["ple_in"].double()) * SQRT_HALF
        q, k, ffn, gated = [], [], [], []
        for n in range(L):
            cos, sin = i["rope"][n % 5 == 4]
            a, b = _qk_norm_rope64(i["q"][n], i["k"][n], i["qw"][n], i["kw"][n], cos, sin, c["q_heads"])
            q.append(a)
            k.append(b)
            state = state + _norm64(i["attn"][n], i["attn_w"][n], EPS)
            ffn.append(_gelu64(i["gate"][n]) * i["up"][n].double())
            state = state + _norm64(i["down"][n], i["ffn_w"][n], EPS)
            gated.append(_gelu64(i["ple_gate"][n]) * ple[:, n * W:(n + 1) * W])
            state = (state + _norm64(i["ple_out"][n], i["ple_w"][n], EPS)) * i["scale"][n].double()
        return {"state": state, "ple": ple, "q": torch.stack(q), "k": torch.stack(k), "ffn": torch.stack(ffn),
                "gated": torch.stack(gated)}


# ---------------------------------------------------------------------------
# token: embed and input norm, then per layer RoPE of Q and K, the f32 KV
# append, add + norm, SwiGLU, add + norm
# ---------------------------------------------------------------------------


class _Token:
    EPS = 1e-5

    @classmethod
    def inputs(cls, c, seed):
        d = _Draw(seed)
        L, H, QD, KD, F = (c["layers"], c["hidden"], c["q_heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"],
                           c["ffn"])
        position = d.ints(0, c["capacity"], 1)
        return {"table": d.normal(c["vocab"], H, std=0.02), "id": d.ints(0, c["vocab"], 1), "position": position,
                "rope": d.rope(position, c["head_dim"] // 2, 1e4), "input_w": d.weight(L + 1, H),
                "q": d.normal(L, QD), "k": d.normal(L, KD), "v": d.normal(L, KD), "attn": d.normal(L, H),
                "post_w": d.weight(L, H), "gate": d.normal(L, F), "up": d.normal(L, F), "down": d.normal(L, H)}

    @classmethod
    def prepare(cls, c, seed):
        L, H, QH, KH, D, F, C = (c["layers"], c["hidden"], c["q_heads"], c["kv_heads"], c["head_dim"], c["ffn"],
                                 c["capacity"])
        i, rt = cls.inputs(c, seed), _runtime()
        o = {"state": _zeros(H), "residual": _zeros(H), "norm": _zeros(H), "q": _zeros(L, QH * D),
             "k": _zeros(L, KH * D), "cache": _zeros(L, 2, C, KH * D), "act": _zeros(L, F)}
        state, residual, norm = _p(o["state"]), _p(o["residual"]), _p(o["norm"])
        cos, sin = i["rope"]
        calls = [(rt.embed_f32, (_p(i["table"]), _p(i["id"]), state, c["vocab"], H, 1)),
                 (rt.rms_norm, (state, _p(i["input_w"]), norm, 1, H, cls.EPS))]
        for n in range(L):
            calls += [
                (rt.rope_half_qk, (_p(i["q"][n]), _p(i["k"][n]), _p(cos), _p(sin), _p(o["q"][n]), _p(o["k"][n]), 1, QH,
                                   KH, D, D // 2)),
                (rt.kv_append, ("f32", _p(o["k"][n]), _p(i["v"][n]), _p(o["cache"][n]), KH * D, C, _p(i["position"]), 1,
                                False, cls.EPS)),
                (rt.add_rms_norm, (_p(i["attn"][n]), state, _p(i["post_w"][n]), residual, norm, 1, H, cls.EPS)),
                (rt.swiglu, (_p(i["gate"][n]), _p(i["up"][n]), _p(o["act"][n]), F)),
                (rt.add_rms_norm, (_p(i["down"][n]), residual, _p(i["input_w"][n + 1]), state, norm, 1, H, cls.EPS)),
            ]
        return _Program(calls, o, i, capture=True)

    @classmethod
    def work(cls, c):
        L, H, QD, KD, F = (c["layers"], c["hidden"], c["q_heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"],
                           c["ffn"])
        layer = 2 * (QD + KD) + c["head_dim"] + 4 * KD + 2 * 5 * H + 3 * F
        return {"bytes": 4 * (5 * H + L * layer), "flops": L * (3 * (QD + KD) + 12 * H + 30 * F)}

    @classmethod
    def tolerance(cls, c):
        return {"rel": 1.6e-6, "max": 2e-5}  # f32 throughout; measured 3e-8 to 4.1e-7 from float64

    @classmethod
    def exact(cls, c, seed):
        L, QH, KH, D, i = c["layers"], c["q_heads"], c["kv_heads"], c["head_dim"], cls.inputs(c, seed)
        cos, sin = i["rope"]
        state = i["table"][i["id"].long()[0]].double()
        norm, residual = _norm64(state, i["input_w"][0], cls.EPS), None
        q, k, act = [], [], []
        cache = torch.zeros((L, 2, c["capacity"], KH * D), dtype=torch.float64, device="cuda")
        for n in range(L):
            q.append(_rope64(i["q"][n].double().reshape(1, QH, D), cos, sin).reshape(-1))
            k.append(_rope64(i["k"][n].double().reshape(1, KH, D), cos, sin).reshape(-1))
            cache[n, 0, i["position"].long()[0]] = k[-1]
            cache[n, 1, i["position"].long()[0]] = i["v"][n].double()
            residual = i["attn"][n].double() + state
            gate = i["gate"][n].double()
            act.append(gate * torch.sigmoid(gate) * i["up"][n].double())
            state = i["down"][n].double() + residual
            norm = _norm64(state, i["input_w"][n + 1], cls.EPS)
        return {"state": state, "residual": residual, "norm": norm, "q": torch.stack(q), "k": torch.stack(k),
                "cache": cache, "act": torch.stack(act)}


# ---------------------------------------------------------------------------
# prefill: the decode ops over a chunk of tokens, with the pre-norms, the KV
# append with the V norm, and the normalised values kept in place
# ---------------------------------------------------------------------------


class _Prefill:
    PLE = 256

    @classmethod
    def inputs(cls, c, seed):
        d = _Draw(seed)
        T, L, H, QH, D, F, V, W = (c["tokens"], c["layers"], c["hidden"], c["q_heads"], c["head_dim"], c["ffn"],
                                   c["vocab"], cls.PLE)
        positions = torch.arange(T, device="cuda", dtype=torch.int32) + 37
        return {
            "tokens": d.blocks(V, H, "q4_0"), "ple_table": d.blocks(V, L * W, "q4_0"), "ids": d.ints(0, V, T),
            "positions": positions, "ple_in": d.normal(T, L * W),
            "rope": [d.rope(positions, D // 2, theta) for theta in (1e4, 1e6)], "pre_w": d.weight(L, H),
            "q": d.normal(L, T, QH * D), "k": d.normal(L, T, D), "v": d.normal(L, T, D), "qw": d.weight(L, D),
            "kw": d.weight(L, D), "attn": d.normal(L, T, H), "attn_w": d.weight(L, H), "ffn_in_w": d.weight(L, H),
            "gate": d.normal(L, T, F), "up": d.normal(L, T, F), "down": d.normal(L, T, H), "ffn_w": d.weight(L, H),
            "ple_gate": d.normal(L, T, W), "ple_out": d.normal(L, T, H), "ple_w": d.weight(L, H),
            "scale": d.uniform(0.5, 1.5, L),
        }

    @classmethod
    def prepare(cls, c, seed):
        T, L, H, QH, D, F, V, W = (c["tokens"], c["layers"], c["hidden"], c["q_heads"], c["head_dim"], c["ffn"],
                                   c["vocab"], cls.PLE)
        i, rt, capacity = cls.inputs(c, seed), _runtime(), T + 64
        cache = _zeros(L, 2, capacity, D) if c["cache"] == "f32" else _zeros(L, 2, capacity, _row_bytes(D, c["cache"]),
                                                                            dtype=torch.uint8)
        o = {"state": _zeros(T, H), "residual": _zeros(T, H), "ple": _zeros(T, L * W), "norm": _zeros(L, T, H),
             "ffn_norm": _zeros(L, T, H), "q": _zeros(L, T, QH * D), "k": _zeros(L, T, D), "ffn": _zeros(L, T, F),
             "gated": _zeros(L, T, W), "cache": cache}
        state, residual = _p(o["state"]), _p(o["residual"])
        calls = [(rt.embed_q4_0, (_p(i["tokens"]), _p(i["ids"]), state, V, H, T, float(np.sqrt(np.float32(H))))),
                 (rt.ple_q4_0, (_p(i["ple_table"]), _p(i["ids"]), _p(i["ple_in"]), _p(o["ple"]), V, L, W, T, PLE_SCALE,
                                SQRT_HALF))]
        for n in range(L):
            cos, sin = i["rope"][n % 5 == 4]
            calls += [
                (rt.rms_norm, (state, _p(i["pre_w"][n]), _p(o["norm"][n]), T, H, EPS)),
                (rt.qk_norm_rope, (_p(i["q"][n]), _p(i["k"][n]), _p(i["qw"][n]), _p(i["kw"][n]), _p(cos), _p(sin),
                                   _p(o["q"][n]), _p(o["k"][n]), T, QH, 1, D, D // 2, EPS)),
                (rt.kv_append, (c["cache"], _p(o["k"][n]), _p(i["v"][n]), _p(cache[n]), D, capacity, _p(i["positions"]),
                                T, True, EPS)),
                (rt.rms_norm_residual, (_p(i["attn"][n]), _p(i["attn_w"][n]), state, None, residual, T, H, EPS)),
                (rt.rms_norm, (residual, _p(i["ffn_in_w"][n]), _p(o["ffn_norm"][n]), T, H, EPS)),
                (rt.geglu, (_p(i["gate"][n]), _p(i["up"][n]), _p(o["ffn"][n]), T * F)),
                (rt.rms_norm_residual, (_p(i["down"][n]), _p(i["ffn_w"][n]), residual, None, state, T, H, EPS)),
                (rt.geglu_offset, (_p(i["ple_gate"][n]), _p(o["ple"]), _p(o["gated"][n]), n * W, L * W, W, T)),
                (rt.rms_norm_add_scale, (_p(i["ple_out"][n]), _p(i["ple_w"][n]), state, _p(i["scale"][n:]), T, H, EPS)),
            ]
        # short chunks are captured, as the framework's own prefill chain offers; long ones are issued
        return _Program(calls, o, i, capture=T <= 1024)

    @classmethod
    def work(cls, c):
        T, L, H, QH, D, F, W = c["tokens"], c["layers"], c["hidden"], c["q_heads"], c["head_dim"], c["ffn"], cls.PLE
        once = T * (_row_bytes(H, "q4_0") + 4 * H + _row_bytes(L * W, "q4_0") + 8 * L * W + 4)
        layer = 4 * (2 * T * (QH + 1) * D + T * D + 2 * D + 3 * (3 * T * H + H) + 2 * (2 * T * H + H) + 3 * T * F +
                     3 * T * W + 2 * T * D + T) + 2 * T * _row_bytes(D, c["cache"])
        return {"bytes": once + L * layer, "flops": L * T * (8 * (QH + 1) * D + 26 * H + 40 * F + 40 * W + 12 * D)}

    @classmethod
    def tolerance(cls, c):
        # f32 throughout; measured 4e-8 to 2.2e-7 from float64; a cache code of a value on a rounding edge may differ
        return {"rel": 1e-6, "max": 2e-5, "differ": 1e-4}

    @classmethod
    def exact(cls, c, seed):
        T, L, H, D, W, i = c["tokens"], c["layers"], c["hidden"], c["head_dim"], cls.PLE, cls.inputs(c, seed)
        ids = i["ids"].long()
        state = _unpack(i["tokens"][ids], "q4_0") * float(np.sqrt(np.float32(H)))
        ple = (_unpack(i["ple_table"][ids], "q4_0") * PLE_SCALE + i["ple_in"].double()) * SQRT_HALF
        out = {k: [] for k in ("norm", "ffn_norm", "q", "k", "ffn", "gated")}
        cache, residual = torch.zeros((L, 2, T + 64, D), dtype=torch.float64, device="cuda"), None
        for n in range(L):
            cos, sin = i["rope"][n % 5 == 4]
            out["norm"].append(_norm64(state, i["pre_w"][n], EPS))
            q, k = _qk_norm_rope64(i["q"][n], i["k"][n], i["qw"][n], i["kw"][n], cos, sin, c["q_heads"])
            out["q"].append(q)
            out["k"].append(k)
            cache[n, 0, 37:37 + T] = k
            cache[n, 1, 37:37 + T] = _norm64(i["v"][n], None, EPS)
            residual = state + _norm64(i["attn"][n], i["attn_w"][n], EPS)
            out["ffn_norm"].append(_norm64(residual, i["ffn_in_w"][n], EPS))
            out["ffn"].append(_gelu64(i["gate"][n]) * i["up"][n].double())
            state = residual + _norm64(i["down"][n], i["ffn_w"][n], EPS)
            out["gated"].append(_gelu64(i["ple_gate"][n]) * ple[:, n * W:(n + 1) * W])
            state = (state + _norm64(i["ple_out"][n], i["ple_w"][n], EPS)) * i["scale"][n].double()
        return {"state": state, "residual": residual, "ple": ple, **{k: torch.stack(v) for k, v in out.items()},
                "cache": cache if c["cache"] == "f32" else None}


# ---------------------------------------------------------------------------
# half: FP16 storage, f32 math; per layer add + norm, RoPE of Q and K, SwiGLU,
# add + norm
# ---------------------------------------------------------------------------


class _Half:
    EPS = 1e-5

    @classmethod
    def inputs(cls, c, seed):
        d = _Draw(seed)
        T, L, H, QD, KD, F = (c["tokens"], c["layers"], c["hidden"], c["heads"] * c["head_dim"],
                              c["kv_heads"] * c["head_dim"], c["ffn"])
        positions = torch.arange(T, device="cuda", dtype=torch.int32)
        i = {"stream": d.normal(T, H), "attn": d.normal(L, T, H), "down": d.normal(L, T, H), "attn_w": d.weight(L, H),
             "down_w": d.weight(L, H), "q": d.normal(L, T, QD), "k": d.normal(L, T, KD), "gate": d.normal(L, T, F),
             "up": d.normal(L, T, F)}
        return {**{k: v.half() for k, v in i.items()}, "rope": d.rope(positions, c["head_dim"] // 2, 130000.0)}

    @classmethod
    def prepare(cls, c, seed):
        T, L, H, QH, KH, D, F = (c["tokens"], c["layers"], c["hidden"], c["heads"], c["kv_heads"], c["head_dim"],
                                 c["ffn"])
        i, rt = cls.inputs(c, seed), _runtime()
        h = torch.float16
        o = {"residual": _zeros(T, H, dtype=h), "stream": _zeros(T, H, dtype=h), "attn_norm": _zeros(L, T, H, dtype=h),
             "down_norm": _zeros(L, T, H, dtype=h), "q": _zeros(L, T, QH * D, dtype=h),
             "k": _zeros(L, T, KH * D, dtype=h), "act": _zeros(L, T, F, dtype=h)}
        cos, sin = i["rope"]
        calls = []
        for n in range(L):
            calls += [
                (rt.rope_half_qk, (_p(i["q"][n]), _p(i["k"][n]), _p(cos), _p(sin), _p(o["q"][n]), _p(o["k"][n]), T, QH,
                                   KH, D, D // 2, True)),
                (rt.add_rms_norm_f16, (_p(i["attn"][n]), _p(o["stream"] if n else i["stream"]), _p(i["attn_w"][n]),
                                       _p(o["residual"]), _p(o["attn_norm"][n]), T, H, cls.EPS)),
                (rt.swiglu_f16, (_p(i["gate"][n]), _p(i["up"][n]), _p(o["act"][n]), T * F)),
                (rt.add_rms_norm_f16, (_p(i["down"][n]), _p(o["residual"]), _p(i["down_w"][n]), _p(o["stream"]),
                                       _p(o["down_norm"][n]), T, H, cls.EPS)),
            ]
        return _Program(calls, o, i, capture=T <= 1024)

    @classmethod
    def work(cls, c):
        T, L, H, QD, KD, F = (c["tokens"], c["layers"], c["hidden"], c["heads"] * c["head_dim"],
                              c["kv_heads"] * c["head_dim"], c["ffn"])
        layer = 2 * (2 * (4 * T * H + H) + 2 * T * (QD + KD) + 3 * T * F) + 4 * T * c["head_dim"]
        return {"bytes": L * layer, "flops": L * T * (12 * H + 3 * (QD + KD) + 30 * F)}

    @classmethod
    def tolerance(cls, c):
        return {"rel": 1e-3, "max": 4e-3}  # outputs rounded to f16: measured 2e-4 to 4.8e-4 from float64

    @classmethod
    def exact(cls, c, seed):
        T, QH, KH, D, i = c["tokens"], c["heads"], c["kv_heads"], c["head_dim"], cls.inputs(c, seed)
        cos, sin = i["rope"]
        stream, residual = i["stream"].double(), None
        out = {k: [] for k in ("attn_norm", "down_norm", "q", "k", "act")}
        for n in range(c["layers"]):
            out["q"].append(_rope64(i["q"][n].double().reshape(T, QH, D), cos, sin).reshape(T, QH * D))
            out["k"].append(_rope64(i["k"][n].double().reshape(T, KH, D), cos, sin).reshape(T, KH * D))
            residual = stream + i["attn"][n].double()
            out["attn_norm"].append(_norm64(residual, i["attn_w"][n], cls.EPS))
            gate = i["gate"][n].double()
            out["act"].append(gate * torch.sigmoid(gate) * i["up"][n].double())
            stream = residual + i["down"][n].double()
            out["down_norm"].append(_norm64(stream, i["down_w"][n], cls.EPS))
        return {"residual": residual, "stream": stream, **{k: torch.stack(v) for k, v in out.items()}}


# ---------------------------------------------------------------------------
# gather: a chunk's rows of every table format, and the PLE chain of both
# ---------------------------------------------------------------------------


class _Gather:
    PLE = 256

    @classmethod
    def inputs(cls, c, seed):
        d = _Draw(seed)
        T, H, V, R = c["tokens"], c["hidden"], c["vocab"], c["ple_layers"] * cls.PLE
        return {"ids": d.ints(0, V, T), "ple_in": d.normal(T, R), "f32": d.normal(V, H, std=0.02),
                **{f: d.blocks(V, H, f) for f in ("q4_0", "q8_0", "q6_k")},
                **{"ple_" + f: d.blocks(V, R, f) for f in ("q4_0", "q6_k")}}

    @classmethod
    def prepare(cls, c, seed):
        T, H, V, L, W = c["tokens"], c["hidden"], c["vocab"], c["ple_layers"], cls.PLE
        i, rt = cls.inputs(c, seed), _runtime()
        scale = float(np.sqrt(np.float32(H)))
        o = {**{f: _zeros(T, H) for f in ("f32", "q4_0", "q8_0", "q6_k")},
             **{"ple_" + f: _zeros(T, L * W) for f in ("q4_0", "q6_k")}}
        ids = _p(i["ids"])
        calls = [(rt.embed_f32, (_p(i["f32"]), ids, _p(o["f32"]), V, H, T))]
        for f, call in (("q4_0", rt.embed_q4_0), ("q8_0", rt.embed_q8_0), ("q6_k", rt.embed_q6_k)):
            calls.append((call, (_p(i[f]), ids, _p(o[f]), V, H, T, scale)))
        for f, call in (("q4_0", rt.ple_q4_0), ("q6_k", rt.ple_q6_k)):
            calls.append((call, (_p(i["ple_" + f]), ids, _p(i["ple_in"]), _p(o["ple_" + f]), V, L, W, T, PLE_SCALE,
                                 SQRT_HALF)))
        return _Program(calls, o, i, capture=T <= 1024)

    @classmethod
    def work(cls, c):
        T, H, R = c["tokens"], c["hidden"], c["ple_layers"] * cls.PLE
        token = sum(_row_bytes(H, f) + 4 * H + 4 for f in ("f32", "q4_0", "q8_0", "q6_k"))
        ple = sum(_row_bytes(R, f) + 8 * R + 4 for f in ("q4_0", "q6_k"))
        return {"bytes": T * (token + ple), "flops": T * (8 * H + 8 * R)}

    @classmethod
    def tolerance(cls, c):
        return {"rel": 1.5e-7, "max": 1e-6}  # one to three roundings a value; measured up to 3.7e-8 from float64

    @classmethod
    def exact(cls, c, seed):
        i = cls.inputs(c, seed)
        ids, scale = i["ids"].long(), float(np.sqrt(np.float32(c["hidden"])))
        out = {f: _unpack(i[f][ids], f) * scale for f in ("q4_0", "q8_0", "q6_k")}
        for f in ("q4_0", "q6_k"):
            out["ple_" + f] = (_unpack(i["ple_" + f][ids], f) * PLE_SCALE + i["ple_in"].double()) * SQRT_HALF
        return {"f32": i["f32"][ids].double(), **out}


# ---------------------------------------------------------------------------
# project: the PLE projection, then per layer QKV and gate/up with the norm
# folded in, the plain output projection, and the PLE input gate
# ---------------------------------------------------------------------------


class _Project:
    PLE = 256

    @classmethod
    def inputs(cls, c, seed):
        d = _Draw(seed)
        L, H, Q, K, F, W = c["layers"], c["hidden"], c["q_width"], c["kv_width"], c["ffn"], cls.PLE

        def weights(out, inner):
            return d.blocks(L * out, inner, "q4_0", std=1.0 / math.sqrt(inner)).reshape(L, out, -1)

        return {"x": d.normal(L, H), "attn": d.normal(L, Q), "ffn_x": d.normal(L, H), "ple_x": d.normal(L, H),
                "attn_w": d.weight(L, H), "ffn_w": d.weight(L, H), "ple": d.normal(L, W), "ple_w": d.weight(W),
                "token_x": d.normal(H), "f16": (d.normal(L * W, H) / math.sqrt(H)).half(), "q": weights(Q, H),
                "k": weights(K, H), "v": weights(K, H), "out": weights(H, Q), "gate": weights(F, H),
                "up": weights(F, H), "ple_gate": weights(W, H)}

    @classmethod
    def prepare(cls, c, seed):
        L, H, Q, K, F, W = c["layers"], c["hidden"], c["q_width"], c["kv_width"], c["ffn"], cls.PLE
        i, rt = cls.inputs(c, seed), _runtime()
        o = {"ple": _zeros(L * W), "q": _zeros(L, Q), "k": _zeros(L, K), "v": _zeros(L, K), "out": _zeros(L, H),
             "gate": _zeros(L, F), "up": _zeros(L, F), "ple_gate": _zeros(L, W)}
        calls = [(rt.ple_projection_f16, (_p(i["token_x"]), _p(i["f16"]), _p(i["ple_w"]), _p(o["ple"]), H, W, L,
                                          1.0 / math.sqrt(H), EPS))]
        for n in range(L):
            calls += [
                (rt.matmul_q4_0_qkv_rms, (_p(i["x"][n]), _p(i["q"][n]), _p(i["k"][n]), _p(i["v"][n]), _p(o["q"][n]),
                                          _p(o["k"][n]), _p(o["v"][n]), H, Q, K, _p(i["attn_w"][n]), EPS)),
                (rt.matvec_q4_0_rms, (_p(i["attn"][n]), _p(i["out"][n]), _p(o["out"][n]), Q, H, None, EPS)),
                (rt.matmul_q4_0_gate_up_rms, (_p(i["ffn_x"][n]), _p(i["gate"][n]), _p(i["up"][n]), _p(o["gate"][n]),
                                              _p(o["up"][n]), H, F, _p(i["ffn_w"][n]), EPS)),
                (rt.ple_gate_gelu, (_p(i["ple_x"][n]), _p(i["ple_gate"][n]), _p(i["ple"]), n * W, _p(o["ple_gate"][n]),
                                    H, W)),
            ]
        return _Program(calls, o, i, capture=True)

    @classmethod
    def work(cls, c):
        L, H, Q, K, F, W = c["layers"], c["hidden"], c["q_width"], c["kv_width"], c["ffn"], cls.PLE
        by_hidden = Q + 2 * K + 2 * F + W
        layer = (by_hidden * _row_bytes(H, "q4_0") + H * _row_bytes(Q, "q4_0") + 4 * (5 * H + Q) +
                 4 * (by_hidden + H + W))
        return {"bytes": 2 * L * W * H + 4 * (H + L * W) + L * layer,
                "flops": 2 * L * W * H + 2 * L * (by_hidden * H + H * Q)}

    @classmethod
    def tolerance(cls, c):
        return {"rel": 1e-6, "max": 1e-5}  # f32 sums of up to 4096 products; measured 1.3e-7 to 2.5e-7 from float64

    @classmethod
    def exact(cls, c, seed):
        L, H, W, i = c["layers"], c["hidden"], cls.PLE, cls.inputs(c, seed)

        def times(name, n, x):
            return _unpack(i[name][n], "q4_0") @ x

        p = (i["f16"].double() @ i["token_x"].double() * (1.0 / math.sqrt(H))).reshape(L, W)
        out = {k: [] for k in ("q", "k", "v", "out", "gate", "up", "ple_gate")}
        for n in range(L):
            x = _norm64(i["x"][n], i["attn_w"][n], EPS)
            for name in ("q", "k", "v"):
                out[name].append(times(name, n, x))
            out["out"].append(times("out", n, i["attn"][n].double()))
            x = _norm64(i["ffn_x"][n], i["ffn_w"][n], EPS)
            for name in ("gate", "up"):
                out[name].append(times(name, n, x))
            out["ple_gate"].append(_gelu64(times("ple_gate", n, i["ple_x"][n].double())) * i["ple"][n].double())
        return {"ple": _norm64(p, i["ple_w"], EPS).reshape(-1), **{k: torch.stack(v) for k, v in out.items()}}


# ---------------------------------------------------------------------------
# logits: capped logits and the selected token of each row
# ---------------------------------------------------------------------------


class _Logits:
    @classmethod
    def inputs(cls, c, seed):
        return _Draw(seed).normal(c["rows"], c["vocab"], std=8.0)

    @classmethod
    def prepare(cls, c, seed):
        logits, rt = cls.inputs(c, seed), _runtime()
        o = {"capped": _zeros(c["rows"], c["vocab"]), "selected": _zeros(c["rows"], dtype=torch.int32)}
        calls = [(rt.softcap_argmax, (_p(logits), _p(o["capped"]), _p(o["selected"]), c["rows"], c["vocab"],
                                      LOGIT_CAP))]
        return _Program(calls, o, logits, capture=False)

    @classmethod
    def work(cls, c):
        n = c["rows"] * c["vocab"]
        return {"bytes": 8 * n + 4 * c["rows"], "flops": 40 * n}

    @classmethod
    def tolerance(cls, c):
        return {"rel": 2e-7, "max": 1e-6, "differ": 0.0}  # measured 4.4e-8 from float64

    @classmethod
    def exact(cls, c, seed):
        x = cls.inputs(c, seed)
        out = torch.empty(x.shape, dtype=torch.float64, device="cuda")
        for n in range(x.shape[0]):
            out[n] = LOGIT_CAP * torch.tanh(x[n].double() / LOGIT_CAP)
        return {"capped": out, "selected": None}


# ---------------------------------------------------------------------------
# host: norm, RoPE, SiLU, product and residual add over host arrays
# ---------------------------------------------------------------------------


class _Host:
    EPS = 1e-5

    @classmethod
    def inputs(cls, c, seed):
        r = np.random.default_rng(seed)
        T, H, F = c["tokens"], c["hidden"], c["ffn"]
        angle = np.float32(c["tokens"]) / np.float32(1e4) ** (np.arange(H // 2, dtype=np.float32) / np.float32(H // 2))
        i = {"x": r.standard_normal(T * H, dtype=np.float32), "res": r.standard_normal(T * H, dtype=np.float32),
             "w": (1.0 + 0.1 * r.standard_normal(H)).astype(np.float32),
             "gate": r.standard_normal(T * F, dtype=np.float32), "up": r.standard_normal(T * F, dtype=np.float32)}
        return {**i, "cos": np.cos(angle), "sin": np.sin(angle)}

    @classmethod
    def prepare(cls, c, seed):
        return _HostProgram(_neural_ops(), cls.inputs(c, seed), c["tokens"], c["hidden"])

    @classmethod
    def work(cls, c):
        T, H, F = c["tokens"], c["hidden"], c["ffn"]
        return {"bytes": 4 * (2 * T * H + H + 2 * T * H + H + 5 * T * F + 3 * T * H), "flops": T * (8 * H + 30 * F)}

    @classmethod
    def tolerance(cls, c):
        return {"rel": 2.5e-7, "max": 5e-6}  # measured up to 5.7e-8 from float64

    @classmethod
    def exact(cls, c, seed):
        i = {k: v.astype(np.float64) for k, v in cls.inputs(c, seed).items()}
        x = i["x"].reshape(c["tokens"], c["hidden"])
        norm = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + cls.EPS) * i["w"]
        a, b = x[:, 0::2], x[:, 1::2]
        rope = np.stack([a * i["cos"] - b * i["sin"], a * i["sin"] + b * i["cos"]], 2)
        silu = i["gate"] / (1.0 + np.exp(-i["gate"]))
        return {"norm": norm.reshape(-1), "rope": rope.reshape(-1), "silu": silu, "product": silu * i["up"],
                "sum": i["x"] + i["res"]}


class _HostProgram:
    def __init__(self, ops, i, tokens, hidden):
        self.ops, self.i, self.tokens, self.hidden = ops, i, tokens, hidden

    def run(self):
        ops, i, T, H = self.ops, self.i, self.tokens, self.hidden
        norm, _ = ops.rms_norm(i["x"], T, H, i["w"], _Host.EPS)
        rope, _ = ops.rope(i["x"], T, H, i["cos"], i["sin"])
        silu, _ = ops.silu(i["gate"])
        product, _ = ops.multiply(silu, i["up"])
        total, _ = ops.add(i["x"], i["res"])
        return {"norm": norm, "rope": rope, "silu": silu, "product": product, "sum": total}


_KINDS = {"decode": _Decode, "token": _Token, "prefill": _Prefill, "half": _Half, "gather": _Gather,
          "project": _Project, "logits": _Logits, "host": _Host}
