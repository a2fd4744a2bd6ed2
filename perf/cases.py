"""Performance cases of the LFM3 step on one MI355X.

Each case is work that a program using this library does, through the C ABI
or the binding's Model and Session:

* `round`: one decode round of a serving loop, the whole 24-layer model.
* `prompt`: one prompt (or prompt chunk) of a session, the whole model.
* `decode_mlp`, `decode_attention`: a decode step's blocks, 1 to 8 rows.
* `prompt_mlp`, `prompt_attention`, `prompt_conv`: a prompt chunk's layers.
* `float_mlp`: the MLP of a BF16, F16 or F32 model, decode and prompt rows.
* `sample`: the serving loop's sampler over a batch of logits rows.

Model sizes are the two that the benchmark and the tests run (`reference`
and `nominal` below); rows, contexts, depths, weight types and options vary.
"""
import ctypes as C
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath(os.path.join("lfm3-gufo-extension_amd", "python")))
import lfm3amd as L  # noqa: E402

DIMS = {"reference": L.Dims(), "nominal": L.Dims(**L.NOMINAL)}
TYPES = {"bf16": L.TYPE_BF16, "f16": L.TYPE_F16, "f32": L.TYPE_F32}
TORCH_TYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
EMBED_ROWS = 1024       # rows of the embedding table that feeds a block case
WEIGHT_STD = 0.0116     # what uniform Q8_0 codes at this scale spread have
D_STD = 0.02            # spread of a Q8_0 block's largest weight
ROUND_SPAN = 64         # tokens a round's sessions decode before they go back
CHECKPOINT_SEED = 77    # the model file of the whole-model cases


# ------------------------------------------------------------------- cases

def listed():
    return [
        # The serving loop at its full batch: eight sessions, ragged contexts.
        {"name": "round_8_sessions", "kind": "round", "dims": "reference", "rows": 8,
         "context_min": 128, "context_max": 8192},
        # A long conversation's next chunk: the deepest prefill the benchmark has.
        {"name": "prompt_512_at_24576", "kind": "prompt", "dims": "reference", "rows": 512,
         "position": 24576},
        # One user decoding alone: the smallest call, launches and latency.
        {"name": "decode_mlp_1", "kind": "decode_mlp", "dims": "reference", "rows": 1,
         "layers": 4},
        # A batch's attention over ragged chat contexts, the 32 x 64 heads.
        {"name": "decode_attention_8", "kind": "decode_attention", "dims": "nominal", "rows": 8,
         "context_min": 1, "context_max": 4096, "sliding": False},
        # One session at the deepest context that is quoted (128K).
        {"name": "decode_attention_128k", "kind": "decode_attention", "dims": "reference",
         "rows": 1, "context_min": 131072, "context_max": 131072, "sliding": False},
        # A full prompt chunk's MLP: the largest matrix products.
        {"name": "prompt_mlp_512", "kind": "prompt_mlp", "dims": "reference", "rows": 512},
        # A chat turn's MLP: a short, odd number of rows.
        {"name": "prompt_mlp_77", "kind": "prompt_mlp", "dims": "reference", "rows": 77},
        # A mid-size chunk's attention layer over some history.
        {"name": "prompt_attention_300", "kind": "prompt_attention", "dims": "reference",
         "rows": 300, "position": 3000, "sliding": False},
        # A short prompt's convolution layer (half of the model's layers).
        {"name": "prompt_conv_37", "kind": "prompt_conv", "dims": "reference", "rows": 37},
        # The reference precision: a BF16 model's decode batch and prompt chunk.
        {"name": "bf16_mlp_8", "kind": "float_mlp", "dims": "reference", "type": "bf16",
         "rows": 8},
        {"name": "bf16_mlp_512", "kind": "float_mlp", "dims": "reference", "type": "bf16",
         "rows": 512},
        # The sampler at the serving loop's defaults.
        {"name": "sample_8", "kind": "sample", "dims": "reference", "rows": 8, "top_k": 50,
         "temperature": 0.1, "repeat_penalty": 1.1, "recent": 64},
    ]


def draw(rng):
    def log_int(lo, hi):
        return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))

    kind = rng.choice(["round", "prompt", "decode_mlp", "decode_attention", "prompt_mlp",
                       "prompt_attention", "prompt_conv", "float_mlp", "sample"])
    dims = rng.choice(["reference", "nominal"])
    depth = rng.choice([0, log_int(16, 24000), log_int(16, 24000)])
    if kind == "round":
        lo = log_int(1, 4000)
        return {"kind": kind, "dims": "reference", "rows": rng.randint(1, 8), "context_min": lo,
                "context_max": log_int(lo, 8192)}
    if kind == "prompt":
        return {"kind": kind, "dims": "reference", "rows": log_int(2, 511), "position": depth}
    if kind == "decode_mlp":
        return {"kind": kind, "dims": dims, "rows": rng.randint(1, 8),
                "layers": rng.randint(2, 5)}
    if kind == "decode_attention":
        lo = log_int(1, 32768)
        rows = rng.randint(1, 8)
        return {"kind": kind, "dims": dims, "rows": rows, "context_min": lo,
                "context_max": log_int(lo, 32768), "sliding": rng.random() < 0.3}
    if kind == "prompt_attention":
        return {"kind": kind, "dims": dims, "rows": log_int(16, 512), "position": depth,
                "sliding": rng.random() < 0.3}
    if kind in ("prompt_mlp", "prompt_conv"):
        return {"kind": kind, "dims": dims, "rows": log_int(16, 512)}
    if kind == "float_mlp":
        return {"kind": kind, "dims": dims, "type": rng.choice(["bf16", "bf16", "f16", "f32"]),
                "rows": log_int(1, 512)}
    return {"kind": kind, "dims": dims, "rows": rng.randint(1, 8),
            "top_k": rng.choice([0, 1, log_int(2, 1024), 50]),
            "temperature": round(rng.uniform(0.1, 1.2), 3), "repeat_penalty": 1.1,
            "recent": log_int(1, 256)}


# ------------------------------------------------------------------ inputs

def _generator(seed, name):
    g = torch.Generator(device="cuda")
    g.manual_seed(L.key(seed & 0xffffffff, name) & 0x7fffffffffffffff)
    return g


def _normal(seed, name, *shape, mean=0.0, std=1.0):
    return torch.randn(*shape, device="cuda", generator=_generator(seed, name)) * std + mean


def _norm_weight(seed, name, n):
    return _normal(seed, name, n, mean=1.0, std=0.02)


def _q8(seed, name, rows, cols):
    """GGUF Q8_0 rows as bytes [rows][cols / 32][34], on the GPU."""
    g = _generator(seed, name)
    q = torch.randint(-127, 128, (rows, cols // 32, 32), dtype=torch.int8, device="cuda",
                      generator=g)
    d = torch.randn(rows, cols // 32, 1, device="cuda", generator=g).abs().mul_(D_STD / 127)
    return torch.cat([d.half().view(torch.uint8), q.view(torch.uint8)], 2)


def _q8_f64(blob):
    d = blob[:, :, :2].contiguous().view(torch.float16).double()
    q = blob[:, :, 2:].contiguous().view(torch.int8).double()
    return (d * q).reshape(blob.shape[0], -1)


def _matrix(kind, seed, name, rows, cols):
    """A weight matrix in its GGUF form: Q8_0 bytes, or float values."""
    if kind == "q8":
        return _q8(seed, name, rows, cols)
    return _normal(seed, name, rows, cols, std=WEIGHT_STD).to(TORCH_TYPES[kind])


def _f64(m):
    return _q8_f64(m) if m.dtype == torch.uint8 else m.double()


class Tiled:
    """One device matrix: sources packed into the library's tiles, side by
    side by row tile, or interleaved (gate and up)."""

    def __init__(self, sources, cols, interleave=False, halves=False):
        self.cols = cols
        tiles = [(s.shape[0] + 15) // 16 for s in sources]
        self.rows = sources[0].shape[0] if interleave else 16 * sum(tiles)
        self.offsets = [16 * sum(tiles[:i]) for i in range(len(tiles))]
        stored = 16 * sum(tiles)
        stride = len(sources) if interleave else 1
        at = list(range(len(sources))) if interleave else [o // 16 for o in self.offsets]
        lib = L.lib()
        if sources[0].dtype == torch.uint8:
            cb, sb = C.c_size_t(), C.c_size_t()
            lib.lfm3_q8_tiled_bytes(stored, cols, C.byref(cb), C.byref(sb))
            self.codes = torch.zeros(cb.value, dtype=torch.uint8, device="cuda")
            self.scales = torch.zeros(sb.value, dtype=torch.uint8, device="cuda")
            for s, o in zip(sources, at):
                L.check(lib.lfm3_q8_pack_device(s.data_ptr(), s.shape[0], cols,
                                                self.codes.data_ptr(), self.scales.data_ptr(), o,
                                                stride, None))
            if halves:
                self.halves = torch.zeros(lib.lfm3_q8_half_tiles_bytes(stored, cols),
                                          dtype=torch.uint8, device="cuda")
                L.check(lib.lfm3_q8_half_tiles(self.codes.data_ptr(), stored, cols,
                                               self.halves.data_ptr(), None))
            torch.cuda.synchronize()
            return
        name = next(k for k, v in TORCH_TYPES.items() if v == sources[0].dtype)
        self.type = TYPES[name]
        host = np.zeros(lib.lfm3_float_tiled_bytes(self.type, stored, cols), np.uint8)
        for s, o in zip(sources, at):
            src = s.cpu().contiguous().view(torch.uint8).numpy()
            L.check(lib.lfm3_float_pack_host(self.type, L.ptr(src), s.shape[0], cols,
                                             L.ptr(host), o, stride))
        self.codes = torch.from_numpy(host).cuda()


def _zeros(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype, device="cuda")


def _p(t):
    return t.data_ptr() if t is not None else None


def _tokens(seed, rows):
    return torch.randint(0, EMBED_ROWS, (rows,), dtype=torch.int32, device="cuda",
                         generator=_generator(seed, "tokens"))


def _contexts(case, seed):
    """Each row's number of keys before the current one."""
    lo, hi = case["context_min"], case["context_max"]
    return np.sort(L.uniform_u32(seed & 0xffffffff, "contexts", case["rows"], lo,
                                 hi)).astype(np.uint32) if hi > lo else np.full(
        case["rows"], lo, np.uint32)


def _pointers(tensors):
    return torch.tensor([t.data_ptr() for t in tensors], dtype=torch.int64, device="cuda")


def _rope_tables(d, sliding):
    theta = d.theta_swa if sliding else d.theta
    i = torch.arange(d.head_dim // 2, dtype=torch.float64)
    freq = torch.pow(torch.tensor(theta, dtype=torch.float64), -2.0 * i / d.head_dim).float()
    factors = torch.ones(d.head_dim // 2)
    factors[d.head_dim // 4:] = 1e30
    return freq.cuda(), factors.cuda()


class State:
    """What a program holds before a pass: its tensors, and the calls of a
    pass with their arguments, addresses included, as a compiled program has
    them; run() makes the calls."""

    def __init__(self, case):
        self.case, self.d, self.calls = case, DIMS[case["dims"]], []
        self.seq = C.c_uint32(0)  # the launches that publish through flags count up

    def call(self, name, *args):
        fn = getattr(L.lib(), name)
        values = [_p(a) if isinstance(a, torch.Tensor) else a for a in args]
        self.calls.append((fn, [t(v) if isinstance(v, (int, float)) else v
                                for t, v in zip(fn.argtypes, values)]))


def _run_calls(s):
    s.seq.value += 1
    for fn, args in s.calls:
        L.check(fn(*args))
    return s.outputs


# ------------------------------------------------ 64-bit restatement (torch)

def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, positions, freq, factors):
    """x [rows][heads][D], rotated in pairs (i, i + D / 2)."""
    angle = (positions.double()[:, None] * freq.double()[None, :])
    if factors is not None:
        angle = angle / factors.double()
    c, s = angle.cos()[:, None, :], angle.sin()[:, None, :]
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _half(x):
    return x.half().double()


def _attend(q, gate, keys, values, first_key, positions, window):
    """q [n][heads][D], gate [n][heads], keys and values [t][kv][D] of
    positions first_key.. (64-bit); causal, gated, grouped."""
    n, heads, dim = q.shape
    kv = keys.shape[1]
    at = first_key + torch.arange(keys.shape[0], device="cuda")
    seen = at[None, :] <= positions[:, None]
    if window:
        seen &= at[None, :] > positions[:, None] - window
    out = torch.empty_like(q)
    for h in range(heads):
        k = keys[:, h // (heads // kv)].contiguous()
        v = values[:, h // (heads // kv)].contiguous()
        s = (q[:, h].contiguous() @ k.t().contiguous()) / math.sqrt(dim)
        s = torch.softmax(s.masked_fill(~seen, -math.inf), -1)
        out[:, h] = s @ v
    return (out / (1 + torch.exp(-gate))[:, :, None]).reshape(n, heads * dim)


def _silu_mlp(x, gate, up, down):
    a, b = x @ _f64(gate).t(), x @ _f64(up).t()
    return (a / (1 + torch.exp(-a)) * b) @ _f64(down).t()


# --------------------------------------------------------------- MLP blocks

def _mlp_source(kind, seed, i, d):
    H, F = d.hidden, d.intermediate
    return {"gate": _matrix(kind, seed, f"gate{i}", F, H),
            "up": _matrix(kind, seed, f"up{i}", F, H),
            "down": _matrix(kind, seed, f"down{i}", H, F),
            "norm": _norm_weight(seed, f"norm{i}", H),
            "post": _norm_weight(seed, f"post{i}", H)}


def _prepare_decode_mlp(case, seed):
    """Rows embedded, then `layers` MLPs: each layer's norm in the launch of
    the gate/up product that reads it, its K parts added by the next norm.
    Each layer has flags of its own."""
    s, lib = State(case), L.lib()
    d, B, H, F = s.d, case["rows"], s.d.hidden, s.d.intermediate
    s.table = Tiled([_q8(seed, "embed", EMBED_ROWS, H)], H)
    s.tokens, s.final = _tokens(seed, B), _norm_weight(seed, "final", H)
    parts = lib.lfm3_q8_gemv_parts(H, F)
    s.x, s.z, s.hid, s.out = _zeros(B, H), _zeros(B, H), _zeros(B, F), _zeros(parts, B, H)
    s.image = _zeros(lib.lfm3_operand_image_bytes(H), dtype=torch.uint8)
    s.exps, s.error = _zeros(8, dtype=torch.int32), _zeros(1, dtype=torch.int32)
    s.call("lfm3_embed", s.table.codes, s.table.scales, EMBED_ROWS, H, s.tokens, B, s.x, None)
    s.layers, branch, post = [], None, None
    for i in range(case["layers"]):
        w = _mlp_source("q8", seed, i, d)
        ffn, down = Tiled([w["gate"], w["up"]], H, interleave=True), Tiled([w["down"]], F)
        flags = _zeros(lib.lfm3_norm_flags_bytes(), dtype=torch.uint8)
        s.layers.append((ffn, down, flags, w["norm"], w["post"]))
        s.call("lfm3_q8_gemv_image_norm", branch, parts if i else 1, B * H, post, s.x, w["norm"],
               d.eps, s.image, s.exps, flags, s.seq, s.error, ffn.codes, ffn.scales, F, H, 1, B,
               s.hid, F, None)
        s.call("lfm3_q8_gemv_partials", down.codes, down.scales, H, F, s.hid, F, s.out, H, B,
               parts, None)
        branch, post = s.out, w["post"]
    s.call("lfm3_residual_norm_parts", branch, parts, B * H, post, s.x, s.final, s.z, B, H, d.eps,
           None)
    s.outputs = {"x": s.x, "z": s.z, "hidden": s.hid}
    return s


def _exact_mlp(case, seed, kind, layers):
    d = DIMS[case["dims"]]
    x = _f64(_matrix(kind, seed, "embed", EMBED_ROWS, d.hidden))[
        _tokens(seed, case["rows"]).long()]
    for i in range(layers):
        w = _mlp_source(kind, seed, i, d)
        z = _rms(x, w["norm"], d.eps)
        a, b = z @ _f64(w["gate"]).t(), z @ _f64(w["up"]).t()
        hidden = a / (1 + torch.exp(-a)) * b
        x = x + _rms(hidden @ _f64(w["down"]).t(), w["post"], d.eps)
    return {"x": x, "z": _rms(x, _norm_weight(seed, "final", d.hidden), d.eps), "hidden": hidden}


class Chunk(State):
    """A prompt chunk through one layer: what every such case shares."""

    def __init__(self, case, seed):
        super().__init__(case)
        n, H = case["rows"], self.d.hidden
        self.table = Tiled([_q8(seed, "embed", EMBED_ROWS, H)], H)
        self.tokens = _tokens(seed, n)
        self.norm, self.post = _norm_weight(seed, "norm0", H), _norm_weight(seed, "post0", H)
        self.final = _norm_weight(seed, "final", H)
        self.lda = (H + 63) // 64 * 64
        self.x, self.z = _zeros(n, H), _zeros(n, H)
        self.a16, self.scale = _zeros(n, self.lda, dtype=torch.float16), _zeros(n)
        # Rows embedded and normed into the layer's FP16 input rows.
        self.call("lfm3_embed", self.table.codes, self.table.scales, EMBED_ROWS, H, self.tokens, n,
                  self.x, None)
        self.call("lfm3_residual_norm_half", None, 1, n * H, None, self.x, self.norm, None,
                  self.a16, self.lda, self.scale, n, H, self.d.eps, None)

    def project(self, m, rows, cols, a16, lda, scale, parts):
        """A projection's output in `parts` K parts."""
        n = self.case["rows"]
        out = _zeros(parts, n, rows)
        self.call("lfm3_q8_gemm_h16", m.halves, m.scales, rows, cols, a16, lda, scale, n, out,
                  rows, parts, None)
        return out

    def end(self, m, cols, a16, lda, scale, **outputs):
        """The layer's output projection, its K parts added to the residual
        rows, then the norm."""
        n, H = self.case["rows"], self.d.hidden
        parts = L.lib().lfm3_q8_gemm_parts(H, cols, n, 0)
        self.out = self.project(m, H, cols, a16, lda, scale, parts)
        self.call("lfm3_residual_norm_parts", self.out, parts, n * H, self.post, self.x, self.final,
                  self.z, n, H, self.d.eps, None)
        self.outputs = dict(outputs, x=self.x, z=self.z)
        return self


def _chunk_f64(case, seed):
    d = DIMS[case["dims"]]
    x = _q8_f64(_q8(seed, "embed", EMBED_ROWS, d.hidden))[_tokens(seed, case["rows"]).long()]
    return d, x, _rms(x, _norm_weight(seed, "norm0", d.hidden), d.eps)


def _chunk_end_f64(d, seed, x, branch):
    x = x + _rms(branch, _norm_weight(seed, "post0", d.hidden), d.eps)
    return {"x": x, "z": _rms(x, _norm_weight(seed, "final", d.hidden), d.eps)}


def _prepare_prompt_mlp(case, seed):
    s, lib = Chunk(case, seed), L.lib()
    n, H, F = case["rows"], s.d.hidden, s.d.intermediate
    w = _mlp_source("q8", seed, 0, s.d)
    s.ffn = Tiled([w["gate"], w["up"]], H, interleave=True, halves=True)
    s.down = Tiled([w["down"]], F, halves=True)
    hld = (F + 63) // 64 * 64
    s.hid = _zeros(n, F)
    s.row_max = _zeros(lib.lfm3_q8_gemm_swiglu_max_blocks(F) * n)
    s.h16, s.hscale = _zeros(n, hld, dtype=torch.float16), _zeros(n)
    s.flags = _zeros(lib.lfm3_q8_gemm_swiglu_flags_bytes(F, n), dtype=torch.uint8)
    s.error = _zeros(1, dtype=torch.int32)
    s.call("lfm3_q8_gemm_swiglu_h16_rows", s.ffn.halves, s.ffn.scales, F, H, s.a16, s.lda, s.scale,
           n, s.hid, F, s.row_max, s.h16, hld, s.hscale, s.flags, s.seq, s.error, None)
    return s.end(s.down, F, s.h16, hld, s.hscale, hidden=s.hid)


def _prepare_float_mlp(case, seed):
    s, lib = State(case), L.lib()
    d, n, H, F = s.d, case["rows"], s.d.hidden, s.d.intermediate
    w = _mlp_source(case["type"], seed, 0, d)
    s.table = Tiled([_matrix(case["type"], seed, "embed", EMBED_ROWS, H)], H)
    s.tokens = _tokens(seed, n)
    s.ffn = Tiled([w["gate"], w["up"]], H, interleave=True)
    s.down = Tiled([w["down"]], F)
    s.norm, s.post, s.final = w["norm"], w["post"], _norm_weight(seed, "final", H)
    parts, t = lib.lfm3_bf16_gemv_parts(H, F, n), s.ffn.type
    s.x, s.z, s.hid, s.out = _zeros(n, H), _zeros(n, H), _zeros(n, F), _zeros(parts, n, H)
    s.call("lfm3_float_embed", t, s.table.codes, EMBED_ROWS, H, s.tokens, None, n, s.x, None)
    s.call("lfm3_residual_norm_parts", None, 1, n * H, None, s.x, s.norm, s.z, n, H, d.eps, None)
    s.call("lfm3_float_gemv", t, s.ffn.codes, F, H, s.z, H, s.hid, F, n, 1, 1, None)
    s.call("lfm3_float_gemv", t, s.down.codes, H, F, s.hid, F, s.out, H, n, parts, 0, None)
    s.call("lfm3_residual_norm_parts", s.out, parts, n * H, s.post, s.x, s.final, s.z, n, H, d.eps,
           None)
    s.outputs = {"x": s.x, "z": s.z, "hidden": s.hid}
    return s


# -------------------------------------------------------- convolution block

def _conv_source(seed, d):
    H = d.hidden
    return {"in": _q8(seed, "in_proj", 3 * H, H), "out": _q8(seed, "out_proj", H, H),
            "taps": _normal(seed, "taps", H, d.conv_width, std=0.1),
            "history": _normal(seed, "history", H, d.conv_width - 1)}


def _prepare_prompt_conv(case, seed):
    s = Chunk(case, seed)
    n, H = case["rows"], s.d.hidden
    w = _conv_source(seed, s.d)
    s.in_proj = Tiled([w["in"]], H, halves=True)
    s.out_proj = Tiled([w["out"]], H, halves=True)
    s.taps, s.history = w["taps"], w["history"]
    s.y16, s.yscale = _zeros(n, H, dtype=torch.float16), _zeros(n)
    # One K part: the convolution reads each value once per tap.
    s.proj = s.project(s.in_proj, 3 * H, H, s.a16, s.lda, s.scale, 1)
    s.call("lfm3_conv_prompt_half", s.proj, 3 * H, s.taps, s.history, n, 0, s.y16, H, s.yscale, H,
           s.d.conv_width, 1, None)
    return s.end(s.out_proj, H, s.y16, H, s.yscale, history=s.history)


def _conv_f64(p, taps, history, d):
    """p [n][3 H] = B | C | X rows; returns y [n][H] and the new history."""
    H, W = d.hidden, d.conv_width
    n = p.shape[0]
    seq = torch.cat([history.double().t(), p[:, :H] * p[:, 2 * H:]], 0)
    y = sum(taps.double()[:, j] * seq[j:j + n] for j in range(W))
    return y * p[:, H:2 * H], seq[n:].t().contiguous()


def _exact_prompt_conv(case, seed):
    d, x, z = _chunk_f64(case, seed)
    w = _conv_source(seed, d)
    y, history = _conv_f64(z @ _f64(w["in"]).t(), w["taps"], w["history"], d)
    out = _chunk_end_f64(d, seed, x, y @ _f64(w["out"]).t())
    return dict(out, history=history)


# --------------------------------------------------------- attention blocks

def _ring(seed, name, capacity, live, d):
    """K or V rows [capacity][kv][D]: `live` slots filled, the rest zero."""
    t = _zeros(capacity, d.kv_heads, d.head_dim, dtype=torch.float16)
    t[:live] = _normal(seed, name, live, d.kv_heads, d.head_dim).half()
    return t


def _decode_rows(case, seed):
    d = DIMS[case["dims"]]
    ctx = _contexts(case, seed)
    # Sliding sessions hold a window's slots, others their context.
    caps = [min(int(c) + 1, d.window) if case["sliding"] else int(c) + 1 for c in ctx]
    live = [min(int(c), cap) for c, cap in zip(ctx, caps)]
    k = [_ring(seed, f"k{i}", cap, n, d) for i, (cap, n) in enumerate(zip(caps, live))]
    v = [_ring(seed, f"v{i}", cap, n, d) for i, (cap, n) in enumerate(zip(caps, live))]
    ld = (d.heads + 2 * d.kv_heads) * d.head_dim + (d.heads + 15) // 16 * 16
    return d, ctx, caps, k, v, _normal(seed, "qkvg", case["rows"], ld)


def _prepare_decode_attention(case, seed):
    d, ctx, caps, k, v, proj = _decode_rows(case, seed)
    s, lib, n, D, ld = State(case), L.lib(), case["rows"], d.head_dim, proj.shape[1]
    s.k, s.v, s.proj = k, v, proj
    s.q_norm, s.k_norm = (_norm_weight(seed, t, D) for t in ("q_norm", "k_norm"))
    s.freq, factors = _rope_tables(d, case["sliding"])
    s.factors = None if case["sliding"] else factors
    cap = lib.lfm3_attention_max_items(n, int(ctx.max()))
    items = np.zeros(cap * C.sizeof(L.AttentionItem), np.uint8)
    count = L.check(lib.lfm3_attention_plan(L.ptr(ctx), n, d.window if case["sliding"] else 0,
                                            L.ptr(items), cap))
    s.items = torch.from_numpy(items).cuda()
    s.kp, s.vp = _pointers(k), _pointers(v)
    s.positions = torch.from_numpy(ctx.astype(np.int32)).cuda()
    s.capacity = torch.tensor(caps, dtype=torch.int32, device="cuda")
    s.ws = _zeros(lib.lfm3_attention_workspace_bytes(count, n, d.heads, d.kv_heads, D),
                  dtype=torch.uint8)
    s.out = _zeros(n, d.heads * D)
    k_at, v_at, g_at = (_p(proj) + 4 * (d.heads + j * d.kv_heads) * D for j in range(3))
    s.call("lfm3_decode_heads_attention_ragged", proj, k_at, v_at, ld, g_at, ld, s.q_norm,
           s.k_norm, s.freq, s.factors, s.kp, s.vp, s.positions, s.capacity, s.items, count, s.out,
           d.heads * D, n, d.heads, d.kv_heads, D, d.eps, s.ws, s.ws.numel(), None)
    s.outputs = {"out": s.out, "slots": [(k[i][int(c) % caps[i]], v[i][int(c) % caps[i]])
                                         for i, c in enumerate(ctx)]}
    return s


def _heads_f64(d, proj, q_norm, k_norm, positions, sliding):
    """Normed, rotated q and k, v and gate of projection rows."""
    D, h, kv = d.head_dim, d.heads, d.kv_heads
    freq, factors = _rope_tables(d, sliding)
    factors = None if sliding else factors
    n, p = proj.shape[0], proj.double()
    q = _rms(p[:, :h * D].reshape(n, h, D), q_norm, d.eps)
    k = _rms(p[:, h * D:(h + kv) * D].reshape(n, kv, D), k_norm, d.eps)
    v = p[:, (h + kv) * D:(h + 2 * kv) * D].reshape(n, kv, D)
    gate = p[:, (h + 2 * kv) * D:(h + 2 * kv) * D + h]
    return (_rope(q, positions, freq, factors), _half(_rope(k, positions, freq, factors)),
            _half(v), gate)


def _exact_decode_attention(case, seed):
    d, ctx, caps, k, v, proj = _decode_rows(case, seed)
    q_norm, k_norm = (_norm_weight(seed, t, d.head_dim) for t in ("q_norm", "k_norm"))
    positions = torch.from_numpy(ctx.astype(np.int64)).cuda()
    q, nk, nv, gate = _heads_f64(d, proj, q_norm, k_norm, positions, case["sliding"])
    out, slots = [], []
    for i, c in enumerate(int(c) for c in ctx):
        first = max(0, c + 1 - d.window) if case["sliding"] else 0
        at = torch.arange(first, c, device="cuda") % caps[i]
        keys = torch.cat([k[i][at].double(), nk[i:i + 1]])
        values = torch.cat([v[i][at].double(), nv[i:i + 1]])
        out.append(_attend(q[i:i + 1], gate[i:i + 1], keys, values, first, positions[i:i + 1], 0))
        slots.append((nk[i], nv[i]))
    return {"out": torch.cat(out), "slots": slots}


def _prompt_attention_source(case, seed):
    d = DIMS[case["dims"]]
    H, D, n, at = d.hidden, d.head_dim, case["rows"], case["position"]
    cap = d.window if case["sliding"] else at + n
    live = min(at, cap)
    return d, {"q": _q8(seed, "q", d.heads * D, H), "k": _q8(seed, "k", d.kv_heads * D, H),
               "v": _q8(seed, "v", d.kv_heads * D, H), "g": _q8(seed, "g", d.heads, H),
               "o": _q8(seed, "o", H, d.heads * D), "q_norm": _norm_weight(seed, "q_norm", D),
               "k_norm": _norm_weight(seed, "k_norm", D), "ck": _ring(seed, "ck", cap, live, d),
               "cv": _ring(seed, "cv", cap, live, d)}


def _prepare_prompt_attention(case, seed):
    d, w = _prompt_attention_source(case, seed)
    s, lib = Chunk(case, seed), L.lib()
    n, H, D, at = case["rows"], d.hidden, d.head_dim, case["position"]
    window, cap, stride = d.window if case["sliding"] else 0, w["ck"].shape[0], d.kv_heads * D
    s.w = w
    s.qkvg = Tiled([w["q"], w["k"], w["v"], w["g"]], H, halves=True)
    s.o = Tiled([w["o"]], d.heads * D, halves=True)
    s.freq, factors = _rope_tables(d, case["sliding"])
    s.factors = None if case["sliding"] else factors
    ld = s.qkvg.rows
    parts = lib.lfm3_q8_gemm_parts(ld, H, n, 0)
    s.proj = s.project(s.qkvg, ld, H, s.a16, s.lda, s.scale, parts)
    if parts > 1:
        s.call("lfm3_sum_parts", s.proj, n * ld, n, ld, ld, parts, None)
    # Full-attention rows go straight into the cache; a sliding ring takes
    # the chunk's rows after the read.
    if window:
        s.k16, s.v16 = (_zeros(n, stride, dtype=torch.float16) for _ in range(2))
    else:
        s.k16, s.v16 = (t.view(-1, stride)[at:at + n] for t in (w["ck"], w["cv"]))
    q_at, k_at, v_at, g_at = (_p(s.proj) + 4 * o for o in s.qkvg.offsets)
    s.call("lfm3_prompt_heads", q_at, k_at, v_at, ld, w["q_norm"], w["k_norm"], s.freq, s.factors,
           s.k16, s.v16, n, d.heads, d.kv_heads, D, at, d.eps, None)
    s.y16, s.yscale = _zeros(n, d.heads * D, dtype=torch.float16), _zeros(n)
    s.ws = _zeros(lib.lfm3_prompt_attention_half_workspace_bytes(n, d.heads, D, at, window),
                  dtype=torch.uint8)
    s.call("lfm3_prompt_attention_half", q_at, ld, s.k16, s.v16, g_at, ld, w["ck"], w["cv"], s.y16,
           d.heads * D, s.yscale, n, d.heads, d.kv_heads, D, at, cap, window, s.ws, s.ws.numel(),
           None)
    if window:
        s.call("lfm3_store_kv", s.k16, s.v16, w["ck"], w["cv"], n, stride, at, cap, None)
    return s.end(s.o, d.heads * D, s.y16, d.heads * D, s.yscale, k=s.k16, v=s.v16)


def _exact_prompt_attention(case, seed):
    d, x, z = _chunk_f64(case, seed)
    _, w = _prompt_attention_source(case, seed)
    n, at = case["rows"], case["position"]
    positions = at + torch.arange(n, device="cuda")
    proj = torch.cat([z @ _f64(w[m]).t() for m in ("q", "k", "v", "g")], 1)
    q, k, v, gate = _heads_f64(d, proj, w["q_norm"], w["k_norm"], positions, case["sliding"])
    window = d.window if case["sliding"] else 0
    first = max(0, at + 1 - window) if window else 0
    slots = torch.arange(first, at, device="cuda") % w["ck"].shape[0]
    y = _attend(q, gate, torch.cat([w["ck"][slots].double(), k]),
                torch.cat([w["cv"][slots].double(), v]), first, positions, window)
    out = _chunk_end_f64(d, seed, x, y @ _f64(w["o"]).t())
    return dict(out, k=k.reshape(n, -1), v=v.reshape(n, -1))


# ------------------------------------------------------------- whole calls

def _layer_source(d, i):
    """Layer i of the checkpoint (a fixed file: only state and tokens follow
    a case's seed)."""
    c, H, D = CHECKPOINT_SEED, d.hidden, d.head_dim
    w = _mlp_source("q8", c, i, d)
    w["ffn_norm"], w["post_ffn"] = (_norm_weight(c, f"{t}{i}", H) for t in ("ffn_norm", "post_ffn"))
    if d.layer_type(i) == L.LAYER_CONV:
        w.update({"taps": _normal(c, f"taps{i}", H, d.conv_width, std=0.1),
                  "in": _q8(c, f"in{i}", 3 * H, H), "out": _q8(c, f"out{i}", H, H)})
    else:
        w.update({"q": _q8(c, f"q{i}", d.heads * D, H), "k": _q8(c, f"k{i}", d.kv_heads * D, H),
                  "v": _q8(c, f"v{i}", d.kv_heads * D, H), "g": _q8(c, f"g{i}", d.heads, H),
                  "o": _q8(c, f"o{i}", H, d.heads * D),
                  "q_norm": _norm_weight(c, f"q_norm{i}", D),
                  "k_norm": _norm_weight(c, f"k_norm{i}", D)})
    return w


def _embedding(d):
    return _q8(CHECKPOINT_SEED, "embedding", d.vocab, d.hidden)


@functools.lru_cache(maxsize=1)
def _model(name):
    """The loaded checkpoint, kept for the program's life as a server does."""
    d = DIMS[name]
    H, F, D = d.hidden, d.intermediate, d.head_dim

    def q8(t, cols):
        return (t.cpu().numpy(), L.TYPE_Q8_0, cols, t.shape[0])

    def f32(t, cols, rows=1):
        return (t.cpu().numpy(), L.TYPE_F32, cols, rows)

    w = L.Weights(d)
    w.globals = [q8(_embedding(d), H), None, f32(_norm_weight(CHECKPOINT_SEED, "output", H), H),
                 f32(_rope_tables(d, False)[1], D // 2)]
    for i in range(d.n_layers):
        s, t = _layer_source(d, i), [None] * L.LAYER_TENSORS
        t[0], t[1] = f32(s["norm"], H), f32(s["ffn_norm"], H)
        t[2], t[3] = f32(s["post"], H), f32(s["post_ffn"], H)
        t[4], t[5], t[6] = q8(s["gate"], H), q8(s["up"], H), q8(s["down"], F)
        if d.layer_type(i) == L.LAYER_CONV:
            t[7] = f32(s["taps"], d.conv_width, H)
            t[8], t[9] = q8(s["in"], H), q8(s["out"], H)
        else:
            t[10], t[11], t[12] = q8(s["q"], H), q8(s["k"], H), q8(s["v"], H)
            t[13], t[14] = f32(s["q_norm"], D), f32(s["k_norm"], D)
            t[15], t[16] = q8(s["g"], H), q8(s["o"], d.heads * D)
        w.layers.append(t)
    model = L.Model(w)
    # A prompt lays out what prompts keep: part of starting the program.
    s = model.session(64)
    s.forward(np.zeros(32, np.uint32), want_logits=False)
    s.close()
    return model


class _Session:
    """A session that is closed once nothing reads its buffers any more."""

    def __init__(self, model, context):
        self.session = model.session(context)

    def __del__(self):
        self.session.close()


class _Address:
    """A session's buffer as torch sees it; a tensor over it keeps this
    object, and so the session, alive."""

    def __init__(self, owner, address, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (address, False), "shape": shape,
                                         "typestr": kind, "version": 2, "strides": None}


def _view(owner, kind, layer, shape, half=False):
    address, nbytes = owner.session.state(kind, layer)
    assert nbytes >= math.prod(shape) * (2 if half else 4)
    return torch.as_tensor(_Address(owner, address, shape, "<f2" if half else "<f4"),
                           device="cuda")


def _history(seed, sid, layer, d):
    return _normal(seed, f"s{sid}.conv{layer}", d.hidden, d.conv_width - 1)


def _history_kv(seed, sid, layer, tag, rows, d):
    return _normal(seed, f"s{sid}.{tag}{layer}", rows, d.kv_heads, d.head_dim).half()


class Sessions(State):
    """Sessions of the loaded model with the state of past conversations."""

    def __init__(self, case, seed, positions, room):
        super().__init__(case)
        self.model = _model(case["dims"])
        self.positions = [int(p) for p in positions]
        self.owners = [_Session(self.model, p + room) for p in self.positions]
        self.sessions = [o.session for o in self.owners]
        d = self.d
        for sid, (p, o) in enumerate(zip(self.positions, self.owners)):
            s = o.session
            for i in range(d.n_layers):
                if d.layer_type(i) == L.LAYER_CONV:
                    _view(o, L.STATE_CONV, i, (d.hidden, d.conv_width - 1)).copy_(
                        _history(seed, sid, i, d))
                    continue
                live = min(p, s.capacity(i))
                for kind, tag in ((L.STATE_KEY, "k"), (L.STATE_VALUE, "v")):
                    if live:
                        _view(o, kind, i, (live, d.kv_heads, d.head_dim), True).copy_(
                            _history_kv(seed, sid, i, tag, live, d))
            s.set_position(p)
        torch.cuda.synchronize()

    def back(self):
        for s, p in zip(self.sessions, self.positions):
            s.set_position(p)


def _prepare_round(case, seed):
    s = Sessions(case, seed, _contexts(case, seed), ROUND_SPAN + 1)
    s.tokens = L.uniform_u32(seed & 0xffffffff, "tokens", case["rows"], 0, s.d.vocab - 1)
    s.fed, s.done = s.tokens, 0
    d = s.d
    last_conv = max(i for i in range(d.n_layers) if d.layer_type(i) == L.LAYER_CONV)
    s.state = [{"logits": _view(e, L.STATE_LOGITS, 0, (d.vocab,)),
                "hidden": _view(e, L.STATE_FRONTIER, 0, (d.hidden,)),
                "conv": _view(e, L.STATE_CONV, last_conv, (d.hidden, d.conv_width - 1))}
               for e in s.owners]
    s.rings = [_view(e, L.STATE_KEY, d.n_layers - 1,
                     (e.session.capacity(d.n_layers - 1), d.kv_heads, d.head_dim), True)
               for e in s.owners]
    return s


def _run_round(s):
    """One token of every session, the greedy ids fed back; after ROUND_SPAN
    tokens the sessions go back to where they began."""
    if s.done == ROUND_SPAN:
        s.back()
        s.done, s.fed = 0, s.tokens
    s.fed = s.model.forward_batch_greedy(s.sessions, s.fed)
    keys = [r[p + s.done] for r, p in zip(s.rings, s.positions)]
    s.done += 1
    return {"ids": s.fed, "state": s.state, "keys": keys}


def _prepare_prompt(case, seed):
    s = Sessions(case, seed, [case["position"]], case["rows"])
    d, n, p, e = s.d, case["rows"], case["position"], s.owners[0]
    s.tokens = L.uniform_u32(seed & 0xffffffff, "tokens", n, 0, d.vocab - 1)
    s.state = {"hidden": _view(e, L.STATE_FRONTIER, 0, (d.hidden,)), "layers": []}
    for i in range(d.n_layers):
        if d.layer_type(i) == L.LAYER_CONV:
            s.state["layers"].append(_view(e, L.STATE_CONV, i, (d.hidden, d.conv_width - 1)))
        elif d.layer_type(i) == L.LAYER_FULL:
            s.state["layers"].append([
                _view(e, kind, i, (p + n, d.kv_heads, d.head_dim), True)[p:]
                for kind in (L.STATE_KEY, L.STATE_VALUE)])
    return s


def _run_prompt(s):
    s.back()
    return dict(s.state, logits=s.sessions[0].forward(s.tokens))


def _whole_f64(d, x, positions, rows):
    """The model on residual rows x. rows: (session seed and id, its rows'
    slice, its position) runs of x. Returns the final normed rows and what
    each layer leaves behind (the new history, or the new K and V rows) per
    run."""
    left = []
    for i in range(d.n_layers):
        w, here = _layer_source(d, i), []
        z = _rms(x, w["norm"], d.eps)
        if d.layer_type(i) == L.LAYER_CONV:
            p, ys = z @ _f64(w["in"]).t(), []
            for seed, sid, part, _ in rows:
                y, history = _conv_f64(p[part], w["taps"], _history(seed, sid, i, d), d)
                ys.append(y)
                here.append(history)
            branch = torch.cat(ys) @ _f64(w["out"]).t()
        else:
            sliding = d.layer_type(i) == L.LAYER_SLIDING
            window, ys = d.window if sliding else 0, []
            proj = torch.cat([z @ _f64(w[m]).t() for m in ("q", "k", "v", "g")], 1)
            q, k, v, gate = _heads_f64(d, proj, w["q_norm"], w["k_norm"], positions, sliding)
            for seed, sid, part, at in rows:
                n = part.stop - part.start
                cap = min(d.window, at + max(n, ROUND_SPAN + 1)) if sliding else at + n
                first = max(0, at + 1 - window) if window else 0
                slots = torch.arange(first, at, device="cuda") % cap
                live = min(at, cap)
                ck, cv = (_history_kv(seed, sid, i, t, live, d)[slots].double() for t in "kv")
                ys.append(_attend(q[part], gate[part], torch.cat([ck, k[part]]),
                                  torch.cat([cv, v[part]]), first, positions[part], window))
                here.append((k[part], v[part]))
            branch = torch.cat(ys) @ _f64(w["o"]).t()
        x = x + _rms(branch, w["post"], d.eps)
        z = _rms(x, w["ffn_norm"], d.eps)
        x = x + _rms(_silu_mlp(z, w["gate"], w["up"], w["down"]), w["post_ffn"], d.eps)
        left.append(here)
    return _rms(x, _norm_weight(CHECKPOINT_SEED, "output", d.hidden), d.eps), left


def _exact_round(case, seed):
    d, ctx = DIMS[case["dims"]], [int(c) for c in _contexts(case, seed)]
    table = _q8_f64(_embedding(d))
    tokens = L.uniform_u32(seed & 0xffffffff, "tokens", case["rows"], 0, d.vocab - 1)
    positions = torch.tensor(ctx, device="cuda")
    rows = [(seed, i, slice(i, i + 1), c) for i, c in enumerate(ctx)]
    hidden, left = _whole_f64(d, table[torch.from_numpy(tokens.astype(np.int64)).cuda()],
                              positions, rows)
    logits = hidden @ table.t()
    last = max(i for i in range(d.n_layers) if d.layer_type(i) == L.LAYER_CONV)
    state = [{"logits": logits[i], "hidden": hidden[i], "conv": left[last][i]}
             for i in range(len(ctx))]
    return {"ids": None, "state": state, "keys": [left[-1][i][0][0] for i in range(len(ctx))]}


def _exact_prompt(case, seed):
    d, n, at = DIMS[case["dims"]], case["rows"], case["position"]
    tokens = L.uniform_u32(seed & 0xffffffff, "tokens", n, 0, d.vocab - 1)
    table = _q8_f64(_embedding(d))
    x = table[torch.from_numpy(tokens.astype(np.int64)).cuda()]
    hidden, left = _whole_f64(d, x, at + torch.arange(n, device="cuda"),
                              [(seed, 0, slice(0, n), at)])
    layers = [h[0] if d.layer_type(i) == L.LAYER_CONV else list(h[0])
              for i, h in enumerate(left) if d.layer_type(i) != L.LAYER_SLIDING]
    return {"hidden": hidden[-1], "layers": layers, "logits": hidden[-1] @ table.t()}


# ------------------------------------------------------------------ sampler

def _prepare_sample(case, seed):
    s, lib, n = State(case), L.lib(), case["rows"]
    cols = s.d.vocab
    s.logits = _normal(seed, "logits", n, cols, std=3.0)
    s.params = L.Sampling(case["temperature"], case["top_k"], case["repeat_penalty"])
    s.recent = torch.randint(0, cols, (n, case["recent"]), dtype=torch.int32, device="cuda",
                             generator=_generator(seed, "recent"))
    s.uniforms = torch.rand(n, device="cuda", generator=_generator(seed, "uniforms"))
    s.ids = _zeros(n, dtype=torch.int32)
    s.ws = _zeros(lib.lfm3_sample_workspace_bytes(n, cols, case["top_k"]), dtype=torch.uint8)
    s.call("lfm3_sample", s.logits, n, cols, cols, C.addressof(s.params), s.recent,
           case["recent"], s.uniforms, s.ids, s.ws, s.ws.numel(), None)
    s.outputs = {"ids": s.ids}
    return s


# ---------------------------------------------------------------- interface

_PREPARE = {"round": _prepare_round, "prompt": _prepare_prompt,
            "decode_mlp": _prepare_decode_mlp, "decode_attention": _prepare_decode_attention,
            "prompt_mlp": _prepare_prompt_mlp, "prompt_attention": _prepare_prompt_attention,
            "prompt_conv": _prepare_prompt_conv, "float_mlp": _prepare_float_mlp,
            "sample": _prepare_sample}
_RUN = {"round": _run_round, "prompt": _run_prompt}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    return _RUN.get(state.case["kind"], _run_calls)(state)


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode_mlp":
        return _exact_mlp(case, seed, "q8", case["layers"])
    if kind == "prompt_mlp":
        return _exact_mlp(case, seed, "q8", 1)
    if kind == "float_mlp":
        return _exact_mlp(case, seed, case["type"], 1)
    return {"round": _exact_round, "prompt": _exact_prompt,
            "decode_attention": _exact_decode_attention,
            "prompt_attention": _exact_prompt_attention, "prompt_conv": _exact_prompt_conv,
            "sample": lambda *_: None}[kind](case, seed)


def _weights_of(d):
    """Weights of one layer's parts, and of the vocabulary table."""
    H, D = d.hidden, d.head_dim
    return {"mlp": 3 * d.intermediate * H, "conv": 4 * H * H,
            "attention": 2 * d.heads * D * H + 2 * d.kv_heads * D * H + d.heads * H,
            "head": d.vocab * H}


def work(case):
    kind, d, n = case["kind"], DIMS[case["dims"]], case["rows"]
    H, F, D, W = d.hidden, d.intermediate, d.head_dim, _weights_of(d)
    q8 = 34 / 32  # bytes of a weight
    if kind == "sample":
        return {"bytes": 4 * n * (d.vocab + case["recent"] + 2), "flops": 2 * n * d.vocab}
    if kind == "float_mlp":
        b = 4 if case["type"] == "f32" else 2
        return {"bytes": W["mlp"] * b + n * H * (b + 8) + 12 * H, "flops": 2 * n * W["mlp"]}
    if kind in ("decode_mlp", "prompt_mlp"):
        layers = case.get("layers", 1)
        return {"bytes": layers * (W["mlp"] * q8 + 8 * H) + n * H * (q8 + 8) + 4 * H,
                "flops": 2 * n * layers * W["mlp"]}
    if kind == "prompt_conv":
        return {"bytes": W["conv"] * q8 + n * H * (q8 + 8) + H * (8 * d.conv_width + 4),
                "flops": 2 * n * W["conv"]}
    if kind == "prompt_attention":
        at, window = case["position"], d.window if case["sliding"] else 0
        seen = [min(window, p + 1) if window else p + 1 for p in range(at, at + n)]
        held = min(at, window) if window else at
        return {"bytes": W["attention"] * q8 + n * H * (q8 + 8) + 12 * H +
                4 * (held + n) * d.kv_heads * D,
                "flops": 2 * n * W["attention"] + 4 * d.heads * D * sum(seen)}
    if kind == "decode_attention":
        # The contexts' mean stands for the seed's.
        mean = (case["context_min"] + case["context_max"]) / 2 + 1
        keys = n * (min(mean, d.window) if case["sliding"] else mean)
        return {"bytes": 4 * keys * d.kv_heads * D + n * (2 * d.heads * D + 2 * d.kv_heads * D) * 4,
                "flops": 4 * d.heads * D * keys}
    types = [d.layer_type(i) for i in range(d.n_layers)]
    convs, full = types.count(L.LAYER_CONV), types.count(L.LAYER_FULL)
    sliding = types.count(L.LAYER_SLIDING)
    weights = d.n_layers * W["mlp"] + convs * W["conv"] + (full + sliding) * W["attention"]
    history = convs * H * (d.conv_width - 1) * 8
    if kind == "round":
        mean = (case["context_min"] + case["context_max"]) / 2 + 1
        keys = n * (full * mean + sliding * min(mean, d.window))
        return {"bytes": (weights + W["head"]) * q8 + 4 * keys * d.kv_heads * D + n * history +
                4 * n * d.vocab, "flops": 2 * n * (weights + W["head"]) + 4 * d.heads * D * keys}
    at = case["position"]
    seen = sum(range(at + 1, at + n + 1))
    near = sum(min(d.window, p + 1) for p in range(at, at + n))
    # The last layer's queries, its projections and its MLP: the last row's only.
    spared = (n - 1) * (W["mlp"] + 2 * d.heads * D * H)
    return {"bytes": (weights + W["head"]) * q8 + history +
            4 * d.kv_heads * D * (full * (at + n) + sliding * (min(at, d.window) + n)),
            "flops": 2 * (n * weights - spared + W["head"]) +
            4 * d.heads * D * ((full - 1) * seen + at + n + sliding * near)}


def tolerance(case):
    """About four times the largest distance of an output to its 64-bit
    value: FP32 sums for the decode and float blocks (their K and V rows are
    rounded to F16), FP16 activations for the prompt blocks, which a whole
    prompt carries through 24 layers. Sampled ids are whole numbers."""
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    return {"rel": {"round": 1e-3, "prompt": 1.6e-2, "decode_mlp": 4e-6,
                    "decode_attention": 5e-4, "prompt_mlp": 1.5e-3, "prompt_attention": 2.5e-3,
                    "prompt_conv": 1.6e-3, "float_mlp": 2e-6}[kind]}
