"""Performance cases: the work a user of this framework has it do, through
its public entry points (the C ABI of include/vkml_hip.h and vkml.Llama).

Each case is a dict of plain values; its "kind" says which path it takes:

  step       one greedy decode step of a two-layer model, launched through
             the C ABI and replayed as a HIP graph, as the model itself does:
             embedding, per layer q|k|v + RoPE + KV append, attention + o,
             gate|up + SwiGLU, down, then the final norm, head and argmax
  llama      vkml.Llama on a GGUF file: forward() of one token (a sampled
             decode step) or of a whole prompt, the logits back on the host
  mlp        a prompt's MLP block with quantized weights: RMSNorm + Q8_0,
             gate, up, SwiGLU + Q8_0, down + residual, for 2 to 1500 rows
             (up to 8 rows take the GEMV, more the matrix cores)
  float_mlp  the same block with f32, f16 or bf16 weights, from 1 row (decode)
  attention  a prompt's causal attention over the KV cache: scores, softmax,
             probs v, or the matrix-core form ("fast")
  attend     one query's attention over a long KV cache, with its merge
"""
import atexit
import ctypes as C
import itertools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "vkml-framework_amd", "python"))

from vkml_amd import gguf, synth  # noqa: E402
from vkml_amd import hip as H  # noqa: E402
from vkml_amd.llama import Llama  # noqa: E402

DEV = "cuda"
EPS = 1e-5
TYPES = {"f32": H.F32, "f16": H.F16, "bf16": H.BF16, "q8_0": H.Q8_0, "q4_0": H.Q4_0, "q4_1": H.Q4_1, "q4_K": H.Q4_K}
FLOATS = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# Bytes a weight takes in its format (q8_0 and q4 with f16 scales).
WEIGHT_BYTES = {"f32": 4.0, "f16": 2.0, "bf16": 2.0, "q8_0": 34 / 32, "q4_0": 18 / 32, "q4_1": 20 / 32, "q4_K": 144 / 256}

# Model shapes: (hidden, heads, kv_heads, head_dim, ffn). tiny, 1b and 7b are
# the repository's own configurations; 3b is a generic size between them.
SHAPES = {
    "tiny": (256, 4, 2, 64, 688),
    "1b": (2048, 32, 8, 64, 8192),
    "3b": (3072, 24, 8, 128, 8192),
    "7b": (4096, 32, 8, 128, 14336),
}
THETA = {"tiny": 1e4, "1b": 5e5, "3b": 5e5, "7b": 1e6}


def listed():
    return [
        # The smallest call: a sampled decode step of a tiny f32 model, where
        # launches and the host round trip are everything.
        {"name": "llama-tiny-f32-decode", "kind": "llama", "shape": "tiny", "wtype": "f32", "kv": "f32", "vocab": 4096, "position": 32, "tokens": 1, "fast": False},
        # A chat prompt through the whole model: 300 tokens, q4_K.
        {"name": "llama-1b-prompt-300", "kind": "llama", "shape": "1b", "wtype": "q4_K", "kv": "f16", "vocab": 8192, "position": 0, "tokens": 300, "fast": False},
        # Decode of a small model early in a chat, and of the 7B shape at a 4K context.
        {"name": "step-1b-q4k-pos640", "kind": "step", "shape": "1b", "wtype": "q4_K", "kv": "f16", "vocab": 32768, "position": 640},
        {"name": "step-7b-q4k-pos4224", "kind": "step", "shape": "7b", "wtype": "q4_K", "kv": "f16", "vocab": 32768, "position": 4224},
        # Decode attention over a long context (GQA 4:1).
        {"name": "attend-32k", "kind": "attend", "heads": 32, "kv_heads": 8, "head_dim": 128, "kv": "f16", "keys": 32768, "fast": False},
        # A few rows: the tail of a chat turn that reuses its cached prefix.
        {"name": "mlp-7b-q4k-5rows", "kind": "mlp", "shape": "7b", "wtype": "q4_K", "rows": 5},
        # A prompt's projections: the common 512 tokens, and a ragged q8_0 one.
        {"name": "mlp-7b-q4k-512rows", "kind": "mlp", "shape": "7b", "wtype": "q4_K", "rows": 512},
        {"name": "mlp-1b-q8-131rows", "kind": "mlp", "shape": "1b", "wtype": "q8_0", "rows": 131},
        # Prompt attention: the second half of a 4096-token prompt, and the
        # matrix-core option on a ragged prompt after a cached prefix.
        {"name": "attention-2048q-4096k", "kind": "attention", "heads": 32, "kv_heads": 8, "head_dim": 128, "kv": "f16", "rows": 2048, "first": 2048, "fast": False},
        {"name": "attention-fast-1000q", "kind": "attention", "heads": 32, "kv_heads": 8, "head_dim": 128, "kv": "f16", "rows": 1000, "first": 37, "fast": True},
        # Unquantized weights: a bf16 decode step's MLP, an f16 prompt's.
        {"name": "mlp-7b-bf16-decode", "kind": "float_mlp", "shape": "7b", "wtype": "bf16", "rows": 1},
        {"name": "mlp-1b-f16-200rows", "kind": "float_mlp", "shape": "1b", "wtype": "f16", "rows": 200},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "llama", "mlp", "mlp", "float_mlp", "attention", "attention", "attend"])
    if kind == "step":
        return {"kind": kind, "shape": rng.choice(["1b", "3b", "7b"]), "wtype": rng.choice(["q4_K", "q4_K", "q8_0"]),
                "kv": rng.choice(["f16", "f16", "f32"]), "vocab": 32 * _log(rng, 32, 1024), "position": _log(rng, 1, 8000)}
    if kind == "llama":
        decode = rng.random() < 0.5
        return {"kind": kind, "shape": rng.choice(["tiny", "1b"]), "wtype": rng.choice(["q4_K", "q8_0", "f32"]), "kv": rng.choice(["f16", "f32"]),
                "vocab": 32 * _log(rng, 32, 256), "position": _log(rng, 9, 400) if decode else 0, "tokens": 1 if decode else _log(rng, 9, 400),
                "fast": False}
    if kind == "mlp":
        few = rng.random() < 0.35
        return {"kind": kind, "shape": rng.choice(["1b", "3b", "7b"]), "wtype": rng.choice(["q4_K", "q4_K", "q8_0", "q4_0", "q4_1"]),
                "rows": rng.randint(2, 8) if few else _log(rng, 9, 1500)}
    if kind == "float_mlp":
        few = rng.random() < 0.5
        return {"kind": kind, "shape": rng.choice(["tiny", "1b", "3b"]), "wtype": rng.choice(["f32", "f16", "bf16"]),
                "rows": rng.randint(1, 8) if few else _log(rng, 9, 500)}
    hd = rng.choice([64, 128, 128])
    kv_heads = rng.choice([2, 4, 8])
    heads = kv_heads * rng.choice([4, 4, 8] if kind == "attend" else [4])
    if kind == "attend":
        fast = rng.random() < 0.3
        return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "head_dim": hd, "kv": "f16" if fast else rng.choice(["f16", "f16", "f32"]),
                "keys": _log(rng, 17, 40000), "fast": fast}
    fast = rng.random() < 0.35
    return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "head_dim": hd, "kv": "f16" if fast else rng.choice(["f16", "f16", "f32"]),
            "rows": _log(rng, 9, 1800), "first": rng.choice([0, rng.randint(1, 2000)]), "fast": fast}


# ---------------------------------------------------------------- weights

class _Rng:
    """Tensors from a seed, on the GPU, one stream per tensor."""

    def __init__(self, seed):
        self.seed, self.index = seed, 0

    def _gen(self):
        self.index += 1
        g = torch.Generator(device=DEV)
        g.manual_seed(self.seed * 100003 + self.index)
        return g

    def normal(self, *shape, scale=1.0, dtype=torch.float32):
        return (torch.randn(shape, generator=self._gen(), device=DEV) * scale).to(dtype)

    def bytes(self, *shape, high=256):
        return torch.randint(0, high, shape, generator=self._gen(), device=DEV, dtype=torch.uint8)


def _f16_bytes(x):
    return x.to(torch.float16).view(torch.uint8).reshape(*x.shape, 2)


class _Matrix:
    """A [rows, cols] weight: the device buffers the C ABI takes, its bytes as
    a GGUF file holds them (llama cases), and its values in float64."""

    def __init__(self, rng, wtype, rows, cols):
        self.wtype, self.rows, self.cols, self.scales = wtype, rows, cols, None
        blocks = rows * cols // 32
        if wtype in FLOATS:
            self.values = rng.normal(rows, cols, scale=0.02, dtype=FLOATS[wtype])
        elif wtype == "q4_K":
            # codes and 6-bit scales and mins uniform, f16 d and dmin half-normal
            n = rows * cols // 256
            raw = rng.bytes(n, 144)
            raw[:, 0:2] = _f16_bytes(rng.normal(n).abs() * (0.01 / 63))
            raw[:, 2:4] = _f16_bytes(rng.normal(n).abs() * (0.01 * 7.5 / 63))
            self.raw = raw
            self.values, self.scales = raw[:, 16:].contiguous(), raw[:, :16].contiguous()
        elif wtype == "q8_0":
            self.values = (rng.bytes(blocks, 32, high=255).to(torch.int16) - 127).to(torch.int8)
            self.scales = (rng.normal(blocks).abs() * 0.0003).to(torch.float16)
        else:
            self.values = rng.bytes(blocks, 16)
            s = (rng.normal(blocks).abs() * 0.003).to(torch.float16)
            self.scales = s if wtype == "q4_0" else torch.stack([s, -7.5 * s], 1).contiguous()

    @property
    def code(self):
        return TYPES[self.wtype]

    @property
    def v(self):
        return _ptr(self.values)

    @property
    def s(self):
        return _ptr(self.scales)

    def gguf(self):
        """(type, bytes or values) as the file holds them."""
        if self.wtype == "q4_K":
            return gguf.Q4_K, self.raw.cpu().numpy().reshape(self.rows, -1)
        if self.wtype == "q8_0":
            both = torch.cat([_f16_bytes(self.scales), self.values.view(torch.uint8)], 1)
            return gguf.Q8_0, both.cpu().numpy().reshape(self.rows, -1)
        return gguf.F32, self.values.cpu().numpy()

    def exact(self):
        if self.wtype in FLOATS:
            return self.values.double()
        if self.wtype == "q8_0":
            w = self.values.double() * self.scales.double()[:, None]
        elif self.wtype == "q4_K":
            # sub-block scales f16(d sc) and offsets f16(-dmin m), as the format's repack defines them
            h = self.scales
            d, dmin = h[:, 0:2].contiguous().view(torch.float16), h[:, 2:4].contiguous().view(torch.float16)
            b = h[:, 4:].to(torch.int32)
            sc = torch.cat([b[:, 0:4] & 63, (b[:, 8:12] & 15) | ((b[:, 0:4] >> 6) << 4)], 1)
            mn = torch.cat([b[:, 4:8] & 63, (b[:, 8:12] >> 4) | ((b[:, 4:8] >> 6) << 4)], 1)
            s = (d.double() * sc.double()).to(torch.float32).to(torch.float16).double()
            o = (-dmin.double() * mn.double()).to(torch.float32).to(torch.float16).double()
            q = self.values.reshape(-1, 4, 32)
            codes = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
            w = codes * s[:, :, None] + o[:, :, None]
        else:
            # word w of a block: values 8 w .. 8 w + 3 in the low nibbles of its bytes, the next four in the high ones
            q = self.values.reshape(-1, 4, 4)
            codes = torch.stack([q & 15, q >> 4], 2).reshape(-1, 32).double()
            if self.wtype == "q4_0":
                w = (codes - 8) * self.scales.double()[:, None]
            else:
                w = codes * self.scales[:, 0:1].double() + self.scales[:, 1:2].double()
        return w.reshape(self.rows, self.cols)


def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def _zeros(*shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype, device=DEV)


def _rope_table(positions, hd, theta):
    freq = theta ** (-torch.arange(0, hd, 2, dtype=torch.float64, device=DEV) / hd)
    angle = torch.arange(positions, dtype=torch.float64, device=DEV)[:, None] * freq[None]
    return torch.stack([angle.cos(), angle.sin()], 2).to(torch.float32)  # [positions, hd / 2, 2]


class _Model:
    """A two-layer decoder's weights."""

    layers = 2

    def __init__(self, case, seed):
        rng = _Rng(seed)
        self.hidden, self.heads, self.kv_heads, self.hd, self.ffn = SHAPES[case["shape"]]
        d, qd, kvd, ff = self.hidden, self.heads * self.hd, self.kv_heads * self.hd, self.ffn
        self.theta, self.vocab = THETA[case["shape"]], case["vocab"]
        # (rows of 688 hold no whole blocks of 32: such a matrix stays f32, and rows of no whole 256 take q8_0)
        kind = lambda cols: case["wtype"] if cols % 256 == 0 or case["wtype"] == "f32" else "q8_0" if cols % 32 == 0 else "f32"  # noqa: E731
        flat = case["wtype"] == "f32"
        self.embed = _Matrix(rng, "f32" if flat else kind(d), self.vocab, d)
        self.head = _Matrix(rng, "f32" if flat else "q8_0", self.vocab, d)
        norm = lambda: 1.0 + rng.normal(d, scale=0.1)  # noqa: E731
        self.final_norm = norm()
        self.blocks = []
        for _ in range(self.layers):
            self.blocks.append({"attn_norm": norm(), "ffn_norm": norm(), "qkv": _Matrix(rng, kind(d), qd + 2 * kvd, d), "o": _Matrix(rng, kind(qd), d, qd),
                                "gate": _Matrix(rng, kind(d), ff, d), "up": _Matrix(rng, kind(d), ff, d), "down": _Matrix(rng, kind(ff), d, ff)})
        self.rng = rng

    def weight_bytes(self):
        ms = [self.head] + [m for b in self.blocks for m in b.values() if isinstance(m, _Matrix)]
        return sum(m.rows * m.cols * WEIGHT_BYTES[m.wtype] for m in ms)


def _model_work(case):
    """(weights in bytes without the head, head bytes, weights as a count, KV bytes a position)."""
    d, heads, kv, hd, ff = SHAPES[case["shape"]]
    w = _Model.layers * ((heads + 2 * kv) * hd * d + d * heads * hd + 3 * d * ff)
    flat = case["wtype"] == "f32"
    wb = WEIGHT_BYTES[case["wtype"]]
    return w * wb, case["vocab"] * d * (4 if flat else 34 / 32), w, _Model.layers * 2 * kv * hd * (2 if case["kv"] == "f16" else 4)


# ---------------------------------------------------------------- float64

def _q8(x):
    """Q8_0 in float64: per 32 values the scale absmax / 127 and codes rounded to nearest."""
    b = x.reshape(-1, 32)
    s = b.abs().amax(1, keepdim=True) / 127
    codes = torch.where(s > 0, torch.round(b / torch.where(s > 0, s, torch.ones_like(s))), torch.zeros_like(b)).clamp(-127, 127)
    return (codes * s).reshape(x.shape)


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _times(x, m):
    return (_q8(x) if m.wtype not in FLOATS else x) @ m.exact().T


def _attention64(q, k, v, first):
    """q [heads, t, hd], k and v [kv_heads, keys, hd]: query i sees keys 0 .. first + i."""
    heads, t, hd = q.shape
    group, keys = heads // k.shape[0], k.shape[1]
    mask = torch.arange(keys, device=DEV)[None] > first + torch.arange(t, device=DEV)[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        s = (q[h] @ k[h // group].T) / math.sqrt(hd)
        out[h] = torch.softmax(s.masked_fill(mask, -math.inf), 1) @ v[h // group]
    return out


def _run64(m, tokens, position, caches, kv, table):
    """Logits of the last of tokens run from position; caches [(k, v)] per layer, float64 [kv_heads, rows, hd], written in place."""
    t, hd = len(tokens), m.hd
    stored = (lambda x: x.float().half().double()) if kv == "f16" else (lambda x: x)
    x = m.embed.exact()[torch.tensor(tokens, device=DEV)]
    cs = table[position:position + t].double()
    c, s = cs[:, None, :, 0], cs[:, None, :, 1]

    def rope(y):  # [t, heads, hd], interleaved pairs
        a, b = y[..., 0::2], y[..., 1::2]
        return torch.stack([a * c - b * s, a * s + b * c], -1).reshape(y.shape)

    for b, (kc, vc) in zip(m.blocks, caches):
        qkv = _times(_norm64(x, b["attn_norm"]), b["qkv"])
        q, k, v = qkv.split([m.heads * hd, m.kv_heads * hd, m.kv_heads * hd], 1)
        q, k, v = rope(q.reshape(t, -1, hd)), rope(k.reshape(t, -1, hd)), v.reshape(t, -1, hd)
        kc[:, position:position + t], vc[:, position:position + t] = stored(k.transpose(0, 1)), stored(v.transpose(0, 1))
        a = _attention64(q.transpose(0, 1).contiguous(), kc[:, :position + t], vc[:, :position + t], position)
        x = x + _times(a.transpose(0, 1).reshape(t, -1), b["o"])
        y = _norm64(x, b["ffn_norm"])
        g, u = _times(y, b["gate"]), _times(y, b["up"])
        x = x + _times(g * torch.sigmoid(g) * u, b["down"])
    return x, _times(_norm64(x[-1:], m.final_norm), m.head)[0]


# ---------------------------------------------------------------- calls

class _Calls:
    """Launches through the C ABI, each an entry point with its arguments."""

    def __init__(self):
        H.init()
        self.calls, self.keep = [], []

    def add(self, name, *args):
        args = tuple(C.byref(a) if isinstance(a, C.Structure) else a for a in args)
        self.calls.append((getattr(H.lib(), name), args))
        self.keep.append(args)

    def run(self):
        for fn, args in self.calls:
            status = fn(*args)
            if status:
                H.check(status)


class _Graph:
    """The calls captured as a HIP graph, as the model captures its decode step."""

    def __init__(self, calls):
        self.calls, handle = calls, C.c_uint64()
        torch.cuda.synchronize()
        H.call("vkml_graph_begin")
        calls.run()
        H.call("vkml_graph_end", C.byref(handle))
        self.handle = handle.value

    def run(self):
        H.call("vkml_graph_launch", self.handle)

    def __del__(self):
        try:
            H.lib().vkml_graph_destroy(self.handle)
        except Exception:
            pass


# ---------------------------------------------------------------- step

def _step_inputs(case, seed):
    m = _Model(case, seed)
    pos = case["position"]
    rows = 128 * ((pos + 1 + 127) // 128) + 256  # room to go on generating
    dtype = FLOATS[case["kv"]]
    caches = []
    for _ in range(m.layers):
        k, v = m.rng.normal(m.kv_heads, rows, m.hd, dtype=dtype), m.rng.normal(m.kv_heads, rows, m.hd, dtype=dtype)
        k[:, pos:] = 0
        v[:, pos:] = 0
        caches.append((k, v))
    token = int(m.rng.bytes(1).item()) % m.vocab
    return m, caches, rows, token, _rope_table(rows, m.hd, m.theta)


def _prepare_step(case, seed):
    m, caches, rows, token, table = _step_inputs(case, seed)
    d, qd, kvd, ff, pos = m.hidden, m.heads * m.hd, m.kv_heads * m.hd, m.ffn, case["position"]
    kv = TYPES[case["kv"]]
    all_chunks = (rows + 127) // 128
    x, qkv, attn, h, logits = _zeros(d), _zeros(qd + 2 * kvd), _zeros(qd), _zeros(ff), _zeros(m.vocab)
    partial, stats = _zeros(m.heads * all_chunks * m.hd), _zeros(m.heads * all_chunks * 2)
    aq, as_, hq, hs = _zeros(qd // 4, dtype=torch.int32), _zeros(qd // 32), _zeros(ff // 4, dtype=torch.int32), _zeros(ff // 32)
    xq, xs, xn = _zeros(d // 4, dtype=torch.int32), _zeros(d // 32), _zeros(d)
    state, log = _zeros(4, dtype=torch.int32), _zeros(16, dtype=torch.int32)
    sync = _zeros(int(H.lib().vkml_attend_fused_sync_bytes(m.layers)) // 4, dtype=torch.int32)
    c = _Calls()
    c.add("vkml_state_set", _ptr(state), token, pos, 0)
    c.add("vkml_embedding_state", H.EmbeddingParams(d, d, m.vocab, m.embed.code, H.F16), m.embed.v, m.embed.s, _ptr(state), _ptr(x))
    # The chunks the position needs, in powers of two from 8, where the one
    # launch takes these shapes; else the whole cache's.
    tier = 8
    while tier < (pos + 1 + 127) // 128:
        tier *= 2
    for i, (b, (k, v)) in enumerate(zip(m.blocks, caches)):
        w = b["qkv"]
        c.add("vkml_gemv_rope", H.GemvRopeParams(w.rows, d, w.code, H.F16, EPS, 0, m.heads, m.kv_heads, m.hd, rows, kv, 1), _ptr(x), _ptr(b["attn_norm"]),
              w.v, w.s, _ptr(qkv), _ptr(table), _ptr(state), _ptr(k), _ptr(v))
        o = H.GemvDotParams(1, d, qd, b["o"].code, H.F16)
        p = H.AttendStepParams(m.heads, m.kv_heads, m.hd, rows, 0, 0, kv, all_chunks, 0, 1, 1.0 / math.sqrt(m.hd), 0.0, 0, 1, 0)
        if H.lib().vkml_attend_step_fused_supported(C.byref(p), C.byref(o)) == 1:
            p.chunks = min(tier, all_chunks)
            p.ready_chunks = min(tier // 2, p.chunks) if tier > 8 else 0
        c.add("vkml_attend_step_fused", p, _ptr(qkv), _ptr(table), _ptr(k), _ptr(v), _ptr(partial), _ptr(stats), _ptr(attn), _ptr(aq), _ptr(as_), _ptr(state),
              o, b["o"].v, b["o"].s, _ptr(x), _ptr(sync), i, m.layers)
        g, u, dn = b["gate"], b["up"], b["down"]
        c.add("vkml_gemv_fused", H.GemvFusedParams(ff, d, g.code, H.F16, 2, 1, EPS, 1), _ptr(x), None, _ptr(b["ffn_norm"]), g.v, g.s, u.v, u.s, None, _ptr(h),
              _ptr(hq), _ptr(hs))
        c.add("vkml_gemv_dot_add", H.GemvDotParams(1, d, ff, dn.code, H.F16), _ptr(hq), dn.v, _ptr(x), dn.s, _ptr(hs), _ptr(x))
    c.add("vkml_rms_norm_quantize", H.RmsNormParams(1, d, EPS), _ptr(x), _ptr(m.final_norm), _ptr(xn), _ptr(xq), _ptr(xs))
    c.add("vkml_gemv_dot", H.GemvDotParams(1, m.vocab, d, m.head.code, H.F16), _ptr(xq), m.head.v, _ptr(logits), m.head.s, _ptr(xs))
    c.add("vkml_step_finish", m.vocab, _ptr(logits), _ptr(state), _ptr(log), 16)
    keep = (m, caches, table, x, qkv, attn, h, logits, partial, stats, aq, as_, hq, hs, xq, xs, xn, state, log, sync)
    outputs = {"logits": logits, "x": x, "k0": caches[0][0], "v0": caches[0][1], "k1": caches[1][0], "v1": caches[1][1]}
    return {"go": _Graph(c), "keep": keep, "outputs": outputs}


def _exact_step(case, seed):
    m, caches, rows, token, table = _step_inputs(case, seed)
    c64 = [(k.double(), v.double()) for k, v in caches]
    x, logits = _run64(m, [token], case["position"], c64, case["kv"], table)
    return {"logits": logits, "x": x[0], "k0": c64[0][0], "v0": c64[0][1], "k1": c64[1][0], "v1": c64[1][1]}


# ---------------------------------------------------------------- llama

_files = itertools.count()
_llamas = []


@atexit.register
def _close_models():
    for m in _llamas:
        m.close()


def _llama_inputs(case, seed):
    m = _Model(case, seed)
    n = case["position"] + case["tokens"]
    tokens = (m.rng.bytes(n, 2).to(torch.int32) * torch.tensor([256, 1], dtype=torch.int32, device=DEV)).sum(1) % m.vocab
    return m, tokens.cpu().numpy().astype(np.int32)


def _prepare_llama(case, seed):
    H.init()
    m, tokens = _llama_inputs(case, seed)
    w = gguf.Writer()
    for key, value in (("context_length", 4096), ("embedding_length", m.hidden), ("block_count", m.layers), ("feed_forward_length", m.ffn),
                       ("attention.head_count", m.heads), ("attention.head_count_kv", m.kv_heads), ("attention.key_length", m.hd),
                       ("attention.value_length", m.hd), ("attention.layer_norm_rms_epsilon", EPS), ("rope.freq_base", float(m.theta))):
        w.add("llama." + key, value)
    w.kv.insert(0, ("general.architecture", 8, "llama"))

    def mat(name, x):
        t, data = x.gguf()
        w.tensor(name, (x.rows, x.cols), t, data)

    def vec(name, x):
        w.tensor(name, (x.numel(),), gguf.F32, x.cpu().numpy())

    mat("token_embd.weight", m.embed)
    vec("output_norm.weight", m.final_norm)
    mat("output.weight", m.head)
    qd, kvd = m.heads * m.hd, m.kv_heads * m.hd
    for i, b in enumerate(m.blocks):
        p = "blk.%d." % i
        t, data = b["qkv"].gguf()
        for name, lo, n in (("attn_q", 0, qd), ("attn_k", qd, kvd), ("attn_v", qd + kvd, kvd)):
            w.tensor(p + name + ".weight", (n, m.hidden), t, data[lo:lo + n])
        mat(p + "attn_output.weight", b["o"])
        vec(p + "attn_norm.weight", b["attn_norm"])
        vec(p + "ffn_norm.weight", b["ffn_norm"])
        mat(p + "ffn_gate.weight", b["gate"])
        mat(p + "ffn_up.weight", b["up"])
        mat(p + "ffn_down.weight", b["down"])
    path = os.path.join(synth.scratch_dir(), "vkml_perf_%d_%d.gguf" % (os.getpid(), next(_files)))
    try:
        w.write(path)
        model = Llama(path, 1024, kv_f16=case["kv"] == "f16", fast_attention=case["fast"])
    finally:
        if os.path.exists(path):
            os.unlink(path)
    _llamas[:] = [x for x in _llamas if x._h]
    _llamas.append(model)
    if case["position"]:
        model.forward(tokens[:case["position"]])
    return {"model": _Owned(model), "tokens": tokens[case["position"]:], "position": case["position"]}


class _Owned:
    """Frees the model with the state that holds it."""

    def __init__(self, model):
        self.model = model

    def __del__(self):
        try:
            self.model.close()
        except Exception:
            pass


def _run_llama(state):
    model = state["model"].model
    if model.position > state["position"]:
        model.rewind(state["position"])  # another reply from the same prefix
    return model.forward(state["tokens"])


def _exact_llama(case, seed):
    m, tokens = _llama_inputs(case, seed)
    n = len(tokens)
    table = _rope_table(n, m.hd, m.theta)
    caches = [tuple(torch.zeros(m.kv_heads, n, m.hd, dtype=torch.float64, device=DEV) for _ in range(2)) for _ in m.blocks]
    return _run64(m, [int(t) for t in tokens], 0, caches, case["kv"], table)[1]


# ---------------------------------------------------------------- mlp

def _mlp_inputs(case, seed):
    rng = _Rng(seed)
    d, _, _, _, ff = SHAPES[case["shape"]]
    t, wt = case["rows"], case["wtype"]
    return rng.normal(t, d), 1.0 + rng.normal(d, scale=0.1), _Matrix(rng, wt, ff, d), _Matrix(rng, wt, ff, d), _Matrix(rng, wt, d, ff)


def _prepare_mlp(case, seed):
    x, nw, g, u, dn = _mlp_inputs(case, seed)
    t, d, ff = case["rows"], g.cols, g.rows
    y, gate, up, out = _zeros(t, d), _zeros(t, ff), _zeros(t, ff), _zeros(t, d)
    c = _Calls()
    if case["kind"] == "mlp":
        xq, xs, hq, hs = _zeros(t * d // 4, dtype=torch.int32), _zeros(t * d // 32), _zeros(t * ff // 4, dtype=torch.int32), _zeros(t * ff // 32)
        product = "vkml_gemv_dot" if t <= 8 else "vkml_matmul_dot"
        c.add("vkml_rms_norm_quantize", H.RmsNormParams(t, d, EPS), _ptr(x), _ptr(nw), _ptr(y), _ptr(xq), _ptr(xs))
        c.add(product, H.GemvDotParams(t, ff, d, g.code, H.F16), _ptr(xq), g.v, _ptr(gate), g.s, _ptr(xs))
        c.add(product, H.GemvDotParams(t, ff, d, u.code, H.F16), _ptr(xq), u.v, _ptr(up), u.s, _ptr(xs))
        c.add("vkml_swiglu_quantize", t * ff, _ptr(gate), _ptr(up), _ptr(hq), _ptr(hs))
        p = H.GemvDotParams(t, d, ff, dn.code, H.F16)
        if t <= 8:
            c.add(product, p, _ptr(hq), dn.v, _ptr(y), dn.s, _ptr(hs))
            c.add("vkml_binary", 0, t * d, t * d, _ptr(x), _ptr(y), _ptr(out))
        else:
            c.add("vkml_matmul_dot_add", p, _ptr(hq), dn.v, _ptr(out), dn.s, _ptr(hs), _ptr(x))
        keep = (xq, xs, hq, hs)
    else:
        def product(m, a, to):
            if t <= 8:
                c.add("vkml_gemv", H.GemvParams(t, m.rows, m.cols, m.code, H.F16, 0, 1, 1), _ptr(a), m.v, _ptr(to), None)
            else:
                c.add("vkml_matmul", H.MatmulParams(t, m.rows, m.cols, 0, 1, 1, 1, m.code, H.F16, 0, 0), _ptr(a), m.v, _ptr(to), None)

        c.add("vkml_rms_norm", H.RmsNormParams(t, d, EPS), _ptr(x), _ptr(nw), _ptr(y))
        product(g, y, gate)
        product(u, y, up)
        h, z = _zeros(t, ff), _zeros(t, d)
        c.add("vkml_unary", 0, t * ff, 0.0, _ptr(gate), _ptr(h))
        c.add("vkml_binary", 2, t * ff, t * ff, _ptr(h), _ptr(up), _ptr(h))
        product(dn, h, z)
        c.add("vkml_binary", 0, t * d, t * d, _ptr(x), _ptr(z), _ptr(out))
        keep = (h, z)
    return {"go": c, "keep": (x, nw, g, u, dn, y, keep), "outputs": {"gate": gate, "up": up, "out": out}}


def _exact_mlp(case, seed):
    x, nw, g, u, dn = _mlp_inputs(case, seed)
    y = _norm64(x.double(), nw)
    gate, up = _times(y, g), _times(y, u)
    return {"gate": gate, "up": up, "out": x.double() + _times(gate * torch.sigmoid(gate) * up, dn)}


# ---------------------------------------------------------------- attention

def _attention_inputs(case, seed):
    rng = _Rng(seed)
    t, keys = case.get("rows", 1), case["first"] + case["rows"] if case["kind"] == "attention" else case["keys"]
    dtype = FLOATS[case["kv"]]
    rows = (keys + 255) // 128 * 128  # a cache with room to go on
    q = rng.normal(case["heads"], t, case["head_dim"])
    return q, rng.normal(case["kv_heads"], rows, case["head_dim"], dtype=dtype), rng.normal(case["kv_heads"], rows, case["head_dim"], dtype=dtype), keys, rows


def _prepare_attention(case, seed):
    q, k, v, keys, rows = _attention_inputs(case, seed)
    heads, t, hd = q.shape
    kv_heads, kv, first, scale = case["kv_heads"], TYPES[case["kv"]], case["first"], 1.0 / math.sqrt(hd)
    c = _Calls()
    if case["fast"]:
        out = _zeros(t, heads, hd)
        p = H.AttendPromptParams(heads, kv_heads, hd, rows, t, first, kv, scale, 0.0)
        c.add("vkml_attend_prompt_fast", p, _ptr(q), _ptr(k), _ptr(v), _ptr(out))
        keep = ()
    else:
        out, scores, probs = _zeros(heads, t, hd), _zeros(heads, t, keys), _zeros(heads, t, keys)
        group, stride = heads // kv_heads, rows * hd
        c.add("vkml_matmul", H.MatmulParams(t, keys, hd, stride, group, heads, 1, kv, H.F16, 1, first), _ptr(q), _ptr(k), _ptr(scores), None)
        c.add("vkml_softmax", H.SoftmaxParams(heads * t, keys, scale, 1, t, first, 0, 0.0, 0), _ptr(scores), _ptr(probs))
        c.add("vkml_matmul", H.MatmulParams(t, hd, keys, stride, group, heads, 0, kv, H.F16, 1, first), _ptr(probs), _ptr(v), _ptr(out), None)
        keep = (scores, probs)
    return {"go": c, "keep": (q, k, v, keep), "outputs": out}


def _exact_attention(case, seed):
    q, k, v, keys, _ = _attention_inputs(case, seed)
    out = _attention64(q.double(), k[:, :keys].double(), v[:, :keys].double(), case["first"])
    return out.transpose(0, 1).contiguous() if case["fast"] else out


def _prepare_attend(case, seed):
    q, k, v, keys, rows = _attention_inputs(case, seed)
    heads, kv_heads, hd = case["heads"], case["kv_heads"], case["head_dim"]
    chunks = (keys + 127) // 128
    partial, stats, out = _zeros(heads * chunks * hd), _zeros(heads * chunks * 2), _zeros(heads, hd)
    values, scales = _zeros(heads * hd // 4, dtype=torch.int32), _zeros(heads * hd // 32)
    p = H.AttendParams(0, keys, rows, heads, kv_heads, hd, TYPES[case["kv"]], chunks, 1.0 / math.sqrt(hd), 0.0)
    c = _Calls()
    keep = ()
    if case["fast"]:
        sync = _zeros(int(H.lib().vkml_attend_fused_sync_bytes(1)) // 4, dtype=torch.int32)
        c.add("vkml_attend_fast", p, _ptr(q), _ptr(k), _ptr(v), _ptr(partial), _ptr(stats), _ptr(out), _ptr(values), _ptr(scales), _ptr(sync), None)
        keep = (sync,)
    else:
        c.add("vkml_attend", p, _ptr(q), _ptr(k), _ptr(v), _ptr(partial), _ptr(stats), None)
        c.add("vkml_attend_merge", p, _ptr(partial), _ptr(stats), _ptr(out), _ptr(values), _ptr(scales))
    return {"go": c, "keep": (q, k, v, partial, stats, keep), "outputs": {"out": out, "codes": values.view(torch.int8), "scales": scales}}


def _exact_attend(case, seed):
    q, k, v, keys, _ = _attention_inputs(case, seed)
    out = _attention64(q.double(), k[:, :keys].double(), v[:, :keys].double(), keys)[:, 0]
    return {"out": out, "codes": None, "scales": out.reshape(-1, 32).abs().amax(1) / 127}


# ---------------------------------------------------------------- the module's contract

def prepare(case, seed):
    kind = case["kind"]
    state = {"step": _prepare_step, "llama": _prepare_llama, "mlp": _prepare_mlp, "float_mlp": _prepare_mlp, "attention": _prepare_attention,
             "attend": _prepare_attend}[kind](case, seed)
    state["kind"] = kind
    torch.cuda.synchronize()
    return state


def run(state):
    if state["kind"] == "llama":
        return _run_llama(state)
    state["go"].run()
    return state["outputs"]


def exact(case, seed):
    return {"step": _exact_step, "llama": _exact_llama, "mlp": _exact_mlp, "float_mlp": _exact_mlp, "attention": _exact_attention,
            "attend": _exact_attend}[case["kind"]](case, seed)


def work(case):
    kind = case["kind"]
    if kind in ("step", "llama"):
        wb, hb, w, kvb = _model_work(case)
        d, heads, _, hd, _ = SHAPES[case["shape"]]
        t, pos = (1, case["position"]) if kind == "step" else (case["tokens"], case["position"])
        seen = t * pos + t * (t + 1) // 2  # (query, key) pairs a head
        return {"bytes": wb + hb + kvb * (pos + t) + t * d * WEIGHT_BYTES[case["wtype"]] + case["vocab"] * 4,
                "flops": 2.0 * w * t + 2.0 * case["vocab"] * d + 4.0 * _Model.layers * heads * hd * seen}
    if kind in ("mlp", "float_mlp"):
        d, _, _, _, ff = SHAPES[case["shape"]]
        return {"bytes": 3 * d * ff * WEIGHT_BYTES[case["wtype"]] + case["rows"] * (2 * d + 2 * ff) * 4, "flops": 6.0 * case["rows"] * d * ff}
    heads, kv, hd, size = case["heads"], case["kv_heads"], case["head_dim"], 2 if case["kv"] == "f16" else 4
    t, first = (case["rows"], case["first"]) if kind == "attention" else (1, case["keys"] - 1)
    seen = t * first + t * (t + 1) // 2
    return {"bytes": 2 * kv * (first + t) * hd * size + 2 * heads * t * hd * 4, "flops": 4.0 * heads * hd * seen}


def tolerance(case):
    """About four times the error measured against exact(). Where activations
    are quantized to Q8_0, a last-bit change in an f32 value can move a code,
    and its block's contribution with it: by one step in a single block
    (3e-4 of the result at most measured), and through all that follows in
    a decode step (0.6%) and a whole model with its prompt (0.9%)."""
    kind = case["kind"]
    if kind == "llama":
        return {"rel": 2e-6, "max": 1e-4} if case["wtype"] == "f32" else {"rel": 0.03, "max": 0.3}
    if kind == "step":
        return {"rel": 0.024, "max": 0.3}
    if kind == "mlp":
        return {"rel": 1.2e-3, "max": 0.05}
    if kind == "attend":
        return {"rel": 2e-6, "max": 1e-4, "differ": 0.005}
    return {"rel": 5e-6, "max": 3e-4}
