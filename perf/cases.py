"""The work this library is used for, as cases that can be timed and checked.

A case is one call, or one short chain of calls, through the public entry
points (``mote_amd.ops`` over the C ABI): quantized linears in each weight
format, the fused gate/up projection, RMSNorm, fused add + RMSNorm and RoPE,
from one decoded token to prompts of thousands of tokens.  Weights hold the
raw GGML blocks of the benchmark workloads (``mote_amd/workloads.py``: scales
|N(0, std)|, uniform quants), drawn on the GPU; activations are binary16.  In the chains the
scales are such that a projection of unit inputs has unit outputs, as trained
weights do.

``kind`` says what one pass is:

* ``linear``: y = x W^T in format ``fmt`` with output type ``out``.
* ``ffn``: the fused gate/up SiLU product, then the down projection.
* ``attention``: RMSNorm, the q / k / v projections, RoPE of q and k, the
  output projection of a given attention result, fused add + RMSNorm.
* ``layer``: ``attention`` followed by ``ffn`` on its normalised output.
"""

import math

import torch

from mote_amd import ops
from mote_amd.device import Stream

HEAD_DIM = 128
EPSILON = 1e-5
THETA = 500000.0

# fmt: (elements per block, bytes per block, std of the scales)
FORMATS = {
    "q4_0": (32, 18, 0.02),
    "q8_0": (32, 34, 0.02),
    "q4_k": (256, 144, 0.002),
    "q6_k": (256, 210, 0.0005),
}

_LINEAR = {
    ("q4_0", "f32"): ops.quantized_linear_q4_0_f32,
    ("q4_0", "f16"): ops.quantized_linear_q4_0_f16,
    ("q8_0", "f32"): ops.quantized_linear_q8_0_f32,
    ("q8_0", "f16"): ops.quantized_linear_q8_0_f16,
    ("q4_k", "f32"): ops.quantized_linear_q4_k_f32,
    ("q4_k", "f16"): ops.quantized_linear_q4_k_f16,
    ("q6_k", "f32"): ops.quantized_linear_q6_k_f32,
    ("q6_k", "f16"): ops.quantized_linear_q6_k_f16,
}


def _linear(name, fmt, m, k, n, out):
    return {"name": name, "kind": "linear", "fmt": fmt, "m": m, "k": k, "n": n, "out": out}


def _block(name, kind, m, hidden, heads, kv_heads, ffn):
    return {"name": name, "kind": kind, "m": m, "hidden": hidden, "heads": heads, "kv_heads": kv_heads, "ffn": ffn}


def listed():
    return [
        # one token through the benchmark's up projection: the latency of a
        # single weight-streaming call
        _linear("decode_up", "q4_0", 1, 4096, 14336, "f32"),
        # one token through every call of a decoder layer: nine short
        # launches, the smallest a few microseconds each
        _block("decode_layer", "layer", 1, 4096, 32, 8, 14336),
        # one token's logits: the vocabulary projection, kept in 6 bits
        _linear("decode_head", "q6_k", 1, 4096, 32000, "f32"),
        # one token through a down projection in 4-bit K-quants
        _linear("decode_down_k", "q4_k", 1, 14336, 4096, "f16"),
        # sixteen sequences decoded together: the MLP, split K in its down
        # projection
        _block("batch_ffn", "ffn", 16, 4096, 32, 8, 14336),
        # the ragged end of a prompt, wider model, binary16 result
        _linear("prompt_tail", "q4_0", 100, 5120, 13824, "f16"),
        # one chunk of a prompt through the benchmark's up projection
        _linear("prefill_up", "q4_0", 512, 4096, 14336, "f32"),
        # a prompt's MLP (the largest case)
        _block("prefill_ffn", "ffn", 1024, 4096, 32, 8, 14336),
        # a long prompt's attention block without the attention itself:
        # norms, four projections, RoPE
        _block("prefill_attention", "attention", 2048, 4096, 32, 8, 14336),
        # a ragged chunk with 8-bit weights
        _linear("prefill_q8_0", "q8_0", 300, 4096, 14336, "f16"),
        # a chunk of a prompt with K-quant weights: the up projection in 4
        # bits, the down projection in 6
        _linear("prefill_q4_k", "q4_k", 512, 4096, 14336, "f32"),
        _linear("prefill_q6_k", "q6_k", 256, 14336, 4096, "f16"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


# A drawn case's limits: at least a pass of several microseconds, at most the
# largest listed case.
_LEAST_BYTES = 8e6
_MOST_FLOPS = 3.4e11


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["bytes"] >= _LEAST_BYTES and w["flops"] <= _MOST_FLOPS:
            return case


def _draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "linear", "ffn", "attention", "layer"])
    # decode (one to a few tokens), batched decode, prompts
    m = rng.choice([1, _log_int(rng, 1, 8), _log_int(rng, 4, 64), _log_int(rng, 48, 512), _log_int(rng, 256, 2048)])
    if kind == "linear":
        fmt = rng.choice(["q4_0", "q4_0", "q8_0", "q4_k", "q6_k"])
        # K in whole blocks; most widths in use are multiples of 256
        step = 256 if fmt in ("q4_k", "q6_k") else rng.choice([256, 256, 128, 64, 32])
        k = max(1, _log_int(rng, 1024, 16384) // step) * step
        n = _log_int(rng, 1024, 32768)
        if rng.random() < 0.6:
            n = max(128, n // 128 * 128)  # most; the others are ragged
        return {"kind": kind, "fmt": fmt, "m": m, "k": k, "n": n, "out": rng.choice(["f32", "f16"])}
    heads = rng.choice([16, 24, 28, 32, 40, 64])
    kv_heads = heads // rng.choice([1, 2, 4])
    hidden = heads * HEAD_DIM
    ffn = max(1, int(hidden * rng.uniform(2.0, 5.5)) // 64) * 64
    return {"kind": kind, "m": m, "hidden": hidden, "heads": heads, "kv_heads": kv_heads, "ffn": ffn}


# --- inputs ---------------------------------------------------------------


def _weights(g, fmt, n, k, unit=False):
    elements, block_bytes, std = FORMATS[fmt]
    if unit:  # q4_0: sqrt(21.5) = 4.6 is the quants' root mean square
        std = 1.0 / (4.6 * math.sqrt(k))
    blocks = n * (k // elements)
    w = torch.randint(0, 256, (blocks, block_bytes), dtype=torch.uint8, device="cuda", generator=g)

    def scales():
        d = torch.randn(blocks, 1, device="cuda", generator=g).abs_().mul_(std)
        return d.to(torch.float16).view(torch.uint8)

    if fmt == "q6_k":
        w[:, 208:210] = scales()
    else:
        w[:, 0:2] = scales()
    if fmt == "q4_k":
        w[:, 2:4] = scales()
    return w.view(-1)


def _normal(g, *shape, mean=0.0, std=1.0):
    return torch.randn(*shape, device="cuda", generator=g).mul_(std).add_(mean).to(torch.float16)


def _inputs(case, seed):
    """The pass's inputs, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    m = case["m"]
    if case["kind"] == "linear":
        return {"x": _normal(g, m, case["k"]), "w": _weights(g, case["fmt"], case["n"], case["k"])}
    s = {}
    hidden, ffn = case["hidden"], case["ffn"]
    if case["kind"] in ("attention", "layer"):
        kv = case["kv_heads"] * HEAD_DIM
        s["x"] = _normal(g, m, hidden)
        s["attended"] = _normal(g, m, hidden)
        s["norm"] = _normal(g, hidden, mean=1.0, std=0.1)
        s["norm_ffn"] = _normal(g, hidden, mean=1.0, std=0.1)
        for name, n in (("q", hidden), ("k", kv), ("v", kv), ("o", hidden)):
            s["w" + name] = _weights(g, "q4_0", n, hidden, unit=True)
        start = int(torch.randint(0, 8192 - min(m, 8191), (1,), device="cuda", generator=g))
        pair = torch.arange(HEAD_DIM // 2, dtype=torch.float64, device="cuda")
        at = torch.arange(start, start + m, dtype=torch.float64, device="cuda")
        angle = at[:, None] * THETA ** (-2.0 * pair / HEAD_DIM)
        s["cos"], s["sin"] = angle.cos().float(), angle.sin().float()
    else:
        s["ffn_in"] = _normal(g, m, hidden)
    if case["kind"] in ("ffn", "layer"):
        s["wgate"] = _weights(g, "q4_0", ffn, hidden, unit=True)
        s["wup"] = _weights(g, "q4_0", ffn, hidden, unit=True)
        s["wdown"] = _weights(g, "q4_0", hidden, ffn, unit=True)
    return s


_stream = None


def prepare(case, seed):
    global _stream
    if _stream is None:
        _stream = Stream()  # a program keeps one
    s = _inputs(case, seed)
    m = case["m"]

    def out(*shape, dtype=torch.float16):
        return torch.empty(*shape, dtype=dtype, device="cuda")

    s["case"], s["stream"] = dict(case), _stream
    if case["kind"] == "linear":
        s["y"] = out(m, case["n"], dtype=torch.float32 if case["out"] == "f32" else torch.float16)
        return s
    hidden = case["hidden"]
    if case["kind"] in ("attention", "layer"):
        kv = case["kv_heads"] * HEAD_DIM
        for name, n in (("xn", hidden), ("q", hidden), ("k", kv), ("v", kv), ("o", hidden), ("ffn_in", hidden)):
            s[name] = out(m, n)
    if case["kind"] in ("ffn", "layer"):
        s["act"], s["y"] = out(m, case["ffn"]), out(m, hidden)
        s["dispatch"] = ops.Q4_0Dispatch()
    return s


# --- one pass -------------------------------------------------------------


def run(s):
    case, stream = s["case"], s["stream"]
    m = case["m"]
    if case["kind"] == "linear":
        _LINEAR[case["fmt"], case["out"]](
            s["x"].data_ptr(), s["w"].data_ptr(), s["y"].data_ptr(), m, case["n"], case["k"], stream)
        return s["y"]
    outputs = {}
    if case["kind"] in ("attention", "layer"):
        outputs.update(_attention(s, case, m, stream))
    if case["kind"] in ("ffn", "layer"):
        hidden, ffn = case["hidden"], case["ffn"]
        s["dispatch"].gate_up_silu(
            s["ffn_in"].data_ptr(), s["wgate"].data_ptr(), s["wup"].data_ptr(), s["act"].data_ptr(),
            m, ffn, hidden, stream, f16_out=True)
        ops.quantized_linear_q4_0_f16(
            s["act"].data_ptr(), s["wdown"].data_ptr(), s["y"].data_ptr(), m, hidden, ffn, stream)
        outputs["act"], outputs["y"] = s["act"], s["y"]
    return outputs


def _attention(s, case, m, stream):
    hidden, kv = case["hidden"], case["kv_heads"] * HEAD_DIM
    xn = s["xn"].data_ptr()
    q, k = s["q"].data_ptr(), s["k"].data_ptr()
    ops.rms_norm_f16(s["x"].data_ptr(), s["norm"].data_ptr(), xn, m, hidden, EPSILON, stream)
    ops.quantized_linear_q4_0_f16(xn, s["wq"].data_ptr(), q, m, hidden, hidden, stream)
    ops.quantized_linear_q4_0_f16(xn, s["wk"].data_ptr(), k, m, kv, hidden, stream)
    ops.quantized_linear_q4_0_f16(xn, s["wv"].data_ptr(), s["v"].data_ptr(), m, kv, hidden, stream)
    ops.rope_qk_f16(
        q, k, s["cos"].data_ptr(), s["sin"].data_ptr(), q, k,
        m, case["heads"], case["kv_heads"], HEAD_DIM, HEAD_DIM, ops.HALF_SPLIT, stream)
    ops.quantized_linear_q4_0_f16(
        s["attended"].data_ptr(), s["wo"].data_ptr(), s["o"].data_ptr(), m, hidden, hidden, stream)
    # the residual stream s["x"] takes the block's output in place
    ops.fused_add_rms_norm_f16(
        s["o"].data_ptr(), s["x"].data_ptr(), s["norm_ffn"].data_ptr(), s["ffn_in"].data_ptr(),
        m, hidden, EPSILON, stream)
    return {"q": s["q"], "k": s["k"], "v": s["v"], "residual": s["x"], "ffn_in": s["ffn_in"]}


# --- what a pass cannot do without ----------------------------------------


def _matrix(fmt, n, k):
    elements, block_bytes, _ = FORMATS[fmt]
    return n * (k // elements) * block_bytes


def work(case):
    m = case["m"]
    if case["kind"] == "linear":
        k, n = case["k"], case["n"]
        out = 4 if case["out"] == "f32" else 2
        return {"bytes": _matrix(case["fmt"], n, k) + 2 * m * k + out * m * n, "flops": 2 * m * n * k}
    hidden, ffn = case["hidden"], case["ffn"]
    total = flops = 0
    if case["kind"] in ("attention", "layer"):
        kv = case["kv_heads"] * HEAD_DIM
        rows = 2 * hidden + 2 * kv
        # weights; x, attended and the tables read; q, k, v, the residual and
        # the normalised output written
        total += _matrix("q4_0", rows, hidden) + 4 * hidden
        total += m * (2 * 2 * hidden + 4 * HEAD_DIM + 2 * (hidden + 2 * kv) + 2 * 2 * hidden)
        flops += 2 * m * rows * hidden
    if case["kind"] in ("ffn", "layer"):
        total += _matrix("q4_0", 3 * ffn, hidden) + m * (2 * ffn + 2 * hidden)
        total += 2 * m * hidden if case["kind"] == "ffn" else 0
        flops += 6 * m * ffn * hidden
    return {"bytes": total, "flops": flops}


def tolerance(case):
    # about four times what the paths differ by from exact(): binary16 results
    # 2.1e-4 from their own rounding, 2.8e-4 with weights rounded to binary16
    # (Q4_0 on the matrix cores, 1.8e-4 alone), 4e-4 along a chain; 32-bit sums
    # of exact products at most 4e-6
    if case["kind"] != "linear":
        return {"rel": 1.6e-3, "max": 1.6e-2}
    if case["out"] == "f16":
        return {"rel": 1.2e-3, "max": 1e-2}
    if case["fmt"] == "q4_0" and case["m"] > 2:
        return {"rel": 8e-4, "max": 8e-3}
    return {"rel": 2e-5, "max": 2e-4}


# --- the same in 64 bits ---------------------------------------------------


def _halves(b):
    return b.contiguous().view(torch.float16).double()


def _decoded(fmt, w, n, k):
    """The matrix [n, k] in binary64, from the blocks' definition."""
    elements, block_bytes, _ = FORMATS[fmt]
    b = w.view(-1, block_bytes)
    if fmt == "q4_0":
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double()
        v = (q - 8.0) * _halves(b[:, 0:2])
    elif fmt == "q8_0":
        v = b[:, 2:].contiguous().view(torch.int8).double() * _halves(b[:, 0:2])
    elif fmt == "q4_k":
        d, dmin, sc = _halves(b[:, 0:2]), _halves(b[:, 2:4]), b[:, 4:16]
        scale = torch.cat([sc[:, 0:4] & 63, (sc[:, 8:12] & 15) | ((sc[:, 0:4] >> 6) << 4)], 1).double()
        least = torch.cat([sc[:, 4:8] & 63, (sc[:, 8:12] >> 4) | ((sc[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        v = (d * scale)[:, :, None] * q - (dmin * least)[:, :, None]
    else:
        low = b[:, 0:128].reshape(-1, 2, 1, 2, 32)  # [half, nibble, 32-byte run, byte]
        low = torch.cat([low & 15, low >> 4], 2).reshape(-1, 2, 4, 32)
        high = b[:, 128:192].reshape(-1, 2, 1, 32)
        high = torch.cat([(high >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (low | (high << 4)).reshape(-1, 16, 16).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = _halves(b[:, 208:210])[:, :, None] * sc[:, :, None] * q
    return v.reshape(n, k)


def _product(x, fmt, w, n, k):
    return x.double() @ _decoded(fmt, w, n, k).t()


def _rms(x, weight):
    return x / (x.square().mean(1, keepdim=True) + EPSILON).sqrt() * weight.double()


def _rotated(x, cos, sin):
    m = x.shape[0]
    a, b = x.view(m, -1, 2, HEAD_DIM // 2).unbind(2)
    c, s = cos.double()[:, None], sin.double()[:, None]
    return torch.stack([a * c - b * s, b * c + a * s], 2).view(m, -1)


def exact(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "linear":
        return _product(s["x"], case["fmt"], s["w"], case["n"], case["k"])
    hidden, ffn = case["hidden"], case["ffn"]
    outputs = {}
    if case["kind"] in ("attention", "layer"):
        kv = case["kv_heads"] * HEAD_DIM
        x = s["x"].double()
        xn = _rms(x, s["norm"])
        outputs["q"] = _rotated(_product(xn, "q4_0", s["wq"], hidden, hidden), s["cos"], s["sin"])
        outputs["k"] = _rotated(_product(xn, "q4_0", s["wk"], kv, hidden), s["cos"], s["sin"])
        outputs["v"] = _product(xn, "q4_0", s["wv"], kv, hidden)
        outputs["residual"] = x + _product(s["attended"], "q4_0", s["wo"], hidden, hidden)
        outputs["ffn_in"] = s["ffn_in"] = _rms(outputs["residual"], s["norm_ffn"])
    if case["kind"] in ("ffn", "layer"):
        gate = _product(s["ffn_in"], "q4_0", s["wgate"], ffn, hidden)
        up = _product(s["ffn_in"], "q4_0", s["wup"], ffn, hidden)
        outputs["act"] = gate * torch.sigmoid(gate) * up
        outputs["y"] = _product(outputs["act"], "q4_0", s["wdown"], hidden, ffn)
    return outputs
