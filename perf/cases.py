"""The calls that a host engine makes of this library, as cases that can be timed.

A case is a dict of plain values.  `kind` names what the host does in one pass:

  linear   cml_matmul_f32: f32 activations through one resident weight
  decode   one token through decoder layers, replayed from a captured graph
  head     the end of a greedy decode step: norm, vocabulary projection, argmax, next embedding row
  ffn      a prompt through one dense feed-forward block, on quantized activations
  mixtral  routed experts from the router's logits (top-2 of 8, SwiGLU, Q4_K)
  gemma    routed experts, fused gate|up (top-8 of 128, GELU)
  seam     the host-slice entry point: activations and outputs in host memory

Weights are seeded N(0, 0.02) values in the named GGUF format, made on the GPU; activations are
seeded normal values whose channels differ in scale, as hidden states do.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from camelid_amd import binding as B
from camelid_amd.binding import Weight, check, lib

BLOCK = {"Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q6_K": (256, 210)}  # values, wire bytes
ACT_F32, ACT_Q8_0, ACT_Q8_K = 0, 1, 2
SILU, GELU_TANH = 0, 1
EPS = 1e-5


def listed():
    return [
        # the smallest call a decode loop makes: one token through a small attention projection, where the launch itself counts
        {"name": "linear_q8_0_2048x2048_t1", "kind": "linear", "fmt": "Q8_0", "rows": 2048, "cols": 2048, "tokens": 1},
        # a decode step of an 8B-class model in the usual mixed Q4_K / Q6_K file: two layers, one of each down-projection format
        {"name": "decode_q4k_4096x14336_2layers", "kind": "decode", "fmt": "Q4_K", "hidden": 4096, "ff": 14336, "kv": 1024, "layers": 2},
        # the end of a greedy step of a 3B-class model: final norm, Q6_K vocabulary projection, pick, embedding of the pick
        {"name": "head_q6k_128256x3072", "kind": "head", "fmt": "Q6_K", "rows": 128256, "cols": 3072},
        # a speculative-verify chunk through a gate / up projection
        {"name": "linear_q4k_14336x4096_t8", "kind": "linear", "fmt": "Q4_K", "rows": 14336, "cols": 4096, "tokens": 8},
        # a verify chunk through a vocabulary projection
        {"name": "linear_q4_0_128256x3072_t16", "kind": "linear", "fmt": "Q4_0", "rows": 128256, "cols": 3072, "tokens": 16},
        # a short, ragged prompt through a projection whose row count is no multiple of a large tile
        {"name": "linear_q6k_18944x3584_t37", "kind": "linear", "fmt": "Q6_K", "rows": 18944, "cols": 3584, "tokens": 37},
        # an ordinary ragged prompt in Q8_0
        {"name": "linear_q8_0_14336x4096_t200", "kind": "linear", "fmt": "Q8_0", "rows": 14336, "cols": 4096, "tokens": 200},
        # a prompt chunk of 512 tokens through a whole dense feed-forward block, the largest case
        {"name": "ffn_q4k_4096x14336_t512", "kind": "ffn", "fmt": "Q4_K", "down": "Q6_K", "hidden": 4096, "ff": 14336, "tokens": 512},
        # one token through a routed expert layer (decode)
        {"name": "mixtral_q4k_8x14336x4096_t1", "kind": "mixtral", "experts": 8, "k": 2, "hidden": 4096, "ff": 14336, "tokens": 1},
        # a prompt of 128 tokens through the same layer
        {"name": "mixtral_q4k_8x14336x4096_t128", "kind": "mixtral", "experts": 8, "k": 2, "hidden": 4096, "ff": 14336, "tokens": 128},
        # many small experts, a batch of 32 tokens
        {"name": "gemma_q4_0_128x704x2816_t32", "kind": "gemma", "fmt": "Q4_0", "experts": 128, "k": 8, "hidden": 2816, "ff": 704, "tokens": 32},
        # a host that holds everything in its own memory: one decode row through the compatibility entry point
        {"name": "seam_q8_0_8192x2048_t1", "kind": "seam", "fmt": "Q8_0", "rows": 8192, "cols": 2048, "tokens": 1},
    ]


def _spread(rng, lo, hi, step=1):
    """A multiple of `step` between lo and hi, uniform over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi // step * step, max(-(-lo // step) * step, round(v / step) * step)))


def draw(rng):
    kind = rng.choices(["linear", "decode", "head", "ffn", "mixtral", "gemma", "seam"], [10, 2, 2, 2, 2, 2, 1])[0]
    fmt = rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q8_0", "Q4_0"])
    if kind == "linear":
        cols = _spread(rng, 512, 16384, 256 if fmt in ("Q4_K", "Q6_K") or rng.random() < 0.7 else 32)
        rows = _spread(rng, 512, min(152064, 600_000_000 // cols), rng.choice([1, 8, 128]))
        tokens = _spread(rng, 1, max(1, min(512, 12_000_000_000 // (rows * cols))))
        return {"kind": kind, "fmt": fmt, "rows": rows, "cols": cols, "tokens": tokens}
    if kind == "decode":
        hidden = _spread(rng, 1024, 6144, 256)
        return {"kind": kind, "fmt": rng.choice(["Q4_K", "Q8_0"]), "hidden": hidden, "ff": _spread(rng, 2 * hidden, 4 * hidden, 256),
                "kv": max(256, hidden // rng.choice([1, 2, 4, 8]) // 64 * 64), "layers": rng.choice([1, 2, 3])}
    if kind == "head":
        return {"kind": kind, "fmt": fmt, "rows": _spread(rng, 32000, 152064, rng.choice([1, 64])), "cols": _spread(rng, 1024, 4096, 256)}
    if kind == "ffn":
        hidden = _spread(rng, 1024, 4096, 256)
        down, ff = rng.choice(["Q4_K", "Q6_K"]), _spread(rng, 2 * hidden, 14336 * 4096 // hidden if hidden > 3584 else 4 * hidden, 256)
        return {"kind": kind, "fmt": "Q4_K", "down": down, "hidden": hidden, "ff": ff, "tokens": _spread(rng, 17, 512)}
    if kind == "mixtral":
        return {"kind": kind, "experts": 8, "k": 2, "hidden": _spread(rng, 1024, 4096, 256), "ff": _spread(rng, 2048, 14336, 256),
                "tokens": _spread(rng, 1, 128)}
    if kind == "gemma":
        return {"kind": kind, "fmt": rng.choice(["Q4_0", "Q8_0"]), "experts": rng.choice([32, 64, 128]), "k": rng.choice([4, 8]),
                "hidden": _spread(rng, 1024, 2816, 256), "ff": _spread(rng, 512, 1408, 64), "tokens": _spread(rng, 1, 64)}
    cols = _spread(rng, 1024, 4096, 256)
    return {"kind": kind, "fmt": rng.choice(["Q8_0", "Q4_K"]), "rows": _spread(rng, 1024, 16384, 64), "cols": cols, "tokens": _spread(rng, 1, 16)}


# ---- seeded weights in wire form, on the GPU ------------------------------------------------------

def _bytes(x):
    return x.contiguous().view(torch.uint8).reshape(x.shape[0], -1)


def _wire_q8_0(w):
    d = (w.abs().amax(1, keepdim=True) / 127).half()
    q = (w / d.float().clamp_min(1e-20)).round().clamp(-127, 127).to(torch.int8)
    return torch.cat([_bytes(d), _bytes(q)], 1)


def _wire_q4_0(w):
    top = w.gather(1, w.abs().argmax(1, keepdim=True))
    d = (top / -8).half()
    inv = torch.where(d == 0, torch.zeros_like(top), 1 / d.float())
    q = (w * inv + 8.5).floor().clamp(0, 15).to(torch.uint8)
    return torch.cat([_bytes(d), q[:, :16] | q[:, 16:] << 4], 1)


def _wire_q4_k(w):
    s = w.reshape(-1, 8, 32)
    low = (-s.amin(2)).clamp_min(0)
    scale = (s.amax(2) + low) / 15
    d, dmin = (scale.amax(1, keepdim=True) / 63).half(), (low.amax(1, keepdim=True) / 63).half()
    sc = (scale / d.float().clamp_min(1e-20)).round().clamp(0, 63)
    m = (low / dmin.float().clamp_min(1e-20)).round().clamp(0, 63)
    step, off = (d.float() * sc).unsqueeze(2), (dmin.float() * m).unsqueeze(2)
    q = ((s + off) / step.clamp_min(1e-20)).round().clamp(0, 15).to(torch.uint8)
    sc, m = sc.to(torch.uint8), m.to(torch.uint8)
    head = torch.cat([sc[:, :4] | sc[:, 4:] >> 4 << 6, m[:, :4] | m[:, 4:] >> 4 << 6, sc[:, 4:] & 15 | (m[:, 4:] & 15) << 4], 1)
    q = q.reshape(-1, 4, 2, 32)
    return torch.cat([_bytes(d), _bytes(dmin), head, (q[:, :, 0] | q[:, :, 1] << 4).reshape(-1, 128)], 1)


def _wire_q6_k(w):
    s = w.reshape(-1, 16, 16)
    top = s.gather(2, s.abs().argmax(2, keepdim=True)).squeeze(2) / -32  # signed, so that both signs of a scale occur
    d = (top.abs().amax(1, keepdim=True) / 127).half()
    sc = (top / d.float().clamp_min(1e-20)).round().clamp(-127, 127)
    step = (d.float() * sc).unsqueeze(2)
    q = torch.where(step == 0, torch.zeros_like(s), s / step).round().clamp(-32, 31).add(32).to(torch.uint8).reshape(-1, 2, 4, 32)
    ql = torch.cat([q[:, :, 0] & 15 | (q[:, :, 2] & 15) << 4, q[:, :, 1] & 15 | (q[:, :, 3] & 15) << 4], 2).reshape(-1, 128)
    qh = (q[:, :, 0] >> 4 | q[:, :, 1] >> 4 << 2 | q[:, :, 2] >> 4 << 4 | q[:, :, 3] >> 4 << 6).reshape(-1, 64)
    return torch.cat([ql, qh, _bytes(sc.to(torch.int8)), _bytes(d)], 1)


_WIRE = {"Q8_0": _wire_q8_0, "Q4_0": _wire_q4_0, "Q4_K": _wire_q4_k, "Q6_K": _wire_q6_k}


def wire_bytes(fmt, rows, cols):
    values, nbytes = BLOCK[fmt]
    return rows * (cols // values) * nbytes


def _synth_wire(gen, fmt, rows, cols):
    values, nbytes = BLOCK[fmt]
    blocks = rows * (cols // values)
    out = torch.empty(blocks, nbytes, dtype=torch.uint8, device="cuda")
    step = (1 << 26) // values
    for at in range(0, blocks, step):
        n = min(step, blocks - at)
        out[at:at + n] = _WIRE[fmt](torch.randn(n, values, generator=gen, device="cuda") * 0.02)
    return out


def _weight(gen, fmt, rows, cols):
    wire, handle = _synth_wire(gen, fmt, rows, cols), C.c_void_p()
    check(lib().cml_weight_upload_dev(B.FORMATS[fmt], rows, cols, wire.data_ptr(), wire.numel(), None, C.byref(handle)))
    torch.cuda.synchronize()  # the wire bytes are freed on return
    return Weight(handle.value, B.FORMATS[fmt], rows, cols)


def _hidden(gen, *shape):
    channel = torch.exp(0.5 * torch.randn(shape[-1], generator=gen, device="cuda"))
    return torch.randn(*shape, generator=gen, device="cuda") * channel


def _norm_weight(gen, n):
    return 1 + 0.2 * torch.randn(n, generator=gen, device="cuda")


def _f32(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _workspace(nbytes):
    return torch.empty(max(256, int(nbytes)), dtype=torch.uint8, device="cuda")


def _quantized(fmt, tokens, cols):
    """Buffers for quantized activation rows of a weight family: (activation format, quants, scales)."""
    per = 256 if fmt in ("Q4_K", "Q6_K") else 32
    return (ACT_Q8_K if per == 256 else ACT_Q8_0, torch.empty(tokens, cols, dtype=torch.int8, device="cuda"), _f32(tokens, cols // per))


class _Graph:
    """A captured launch sequence, replayed on the default stream."""

    def __init__(self, sequence):
        L, stream = lib(), C.c_void_p()
        sequence(None)  # once outside the capture
        check(L.cml_stream_create(C.byref(stream)))
        check(L.cml_graph_begin_capture(stream))
        sequence(stream)
        graph = C.c_void_p()
        check(L.cml_graph_end_capture(stream, C.byref(graph)))
        check(L.cml_stream_destroy(stream))
        self.handle = graph.value

    def launch(self):
        check(lib().cml_graph_launch(self.handle, None))

    def __del__(self):
        lib().cml_graph_destroy(self.handle)


# ---- the kinds: what is in hand before the call, and the call -----------------------------------------

def _prepare_linear(case, gen):
    fmt, rows, cols, tokens = case["fmt"], case["rows"], case["cols"], case["tokens"]
    w, x, out = _weight(gen, fmt, rows, cols), _hidden(gen, tokens, cols), _f32(tokens, rows)
    ws = _workspace(lib().cml_matmul_workspace_bytes(w.fmt, cols, tokens))
    call = (w.handle, x.data_ptr(), tokens, out.data_ptr(), ws.data_ptr(), ws.numel(), None)
    return {"keep": (w, x, ws), "call": call, "out": out}


def _run_linear(s):
    check(lib().cml_matmul_f32(*s["call"]))
    return s["out"]


def _decode_formats(fmt, layer):
    """(v, down) of a layer: every second one of a Q4_K file keeps them in Q6_K."""
    return ("Q6_K", "Q6_K") if fmt == "Q4_K" and layer % 2 == 0 else (fmt, fmt)


def _prepare_decode(case, gen):
    L, fmt, hidden, ff, kv = lib(), case["fmt"], case["hidden"], case["ff"], case["kv"]
    x0 = _hidden(gen, hidden)
    layers, keep, outs, x = [], [x0], [], x0
    for i in range(case["layers"]):
        v_fmt, down_fmt = _decode_formats(fmt, i)
        q, k, v, o = _weight(gen, fmt, hidden, hidden), _weight(gen, fmt, kv, hidden), _weight(gen, v_fmt, kv, hidden), _weight(gen, fmt, hidden, hidden)
        gate, up, down = _weight(gen, fmt, ff, hidden), _weight(gen, fmt, ff, hidden), _weight(gen, down_fmt, hidden, ff)
        norm1, norm2 = _norm_weight(gen, hidden), _norm_weight(gen, hidden)
        normed, qo, ko, vo, mid, normed2, go, uo, y = _f32(hidden), _f32(hidden), _f32(kv), _f32(kv), _f32(hidden), _f32(hidden), _f32(ff), _f32(ff), _f32(hidden)
        _, aq, as_ = _quantized(fmt, 1, hidden)
        act, fq, fs = _quantized(down_fmt, 1, ff)
        ws = _workspace(max(L.cml_matmul_workspace_bytes(w.fmt, hidden, 1) for w in (q, v)))
        handles, targets = (C.c_void_p * 3)(q.handle, k.handle, v.handle), (C.c_void_p * 3)(qo.data_ptr(), ko.data_ptr(), vo.data_ptr())
        keep += [q, k, v, o, gate, up, down, norm1, norm2, normed, qo, mid, normed2, go, uo, aq, as_, fq, fs, ws, handles, targets, x]
        layers.append((x, norm1, normed, handles, targets, ws, qo, aq, as_, o, mid, norm2, normed2, gate, up, go, uo, act, fq, fs, down, y))
        outs += [ko, vo]
        x = y
    quantize = L.cml_quantize_q8_k if fmt in ("Q4_K", "Q6_K") else L.cml_quantize_q8_0

    def sequence(stream):
        for x, norm1, normed, handles, targets, ws, qo, aq, as_, o, mid, norm2, normed2, gate, up, go, uo, act, fq, fs, down, y in layers:
            check(L.cml_rms_norm_quantize(ACT_F32, x.data_ptr(), norm1.data_ptr(), EPS, 1, hidden, normed.data_ptr(), None, None, stream))
            check(L.cml_matmul_f32_multi(handles, 3, normed.data_ptr(), targets, ws.data_ptr(), ws.numel(), stream))
            # (attention itself is the host engine's: the q row stands in for its output)
            check(quantize(qo.data_ptr(), 1, hidden, aq.data_ptr(), as_.data_ptr(), stream))
            check(L.cml_gemv(o.handle, aq.data_ptr(), as_.data_ptr(), mid.data_ptr(), x.data_ptr(), stream))
            check(L.cml_rms_norm_quantize(ACT_F32, mid.data_ptr(), norm2.data_ptr(), EPS, 1, hidden, normed2.data_ptr(), None, None, stream))
            check(L.cml_matmul_f32_pair(gate.handle, up.handle, normed2.data_ptr(), go.data_ptr(), uo.data_ptr(), ws.data_ptr(), ws.numel(), stream))
            check(L.cml_glu_quantize(SILU, act, go.data_ptr(), uo.data_ptr(), 1, ff, fq.data_ptr(), fs.data_ptr(), stream))
            check(L.cml_gemv(down.handle, fq.data_ptr(), fs.data_ptr(), y.data_ptr(), mid.data_ptr(), stream))

    return {"keep": keep, "graph": _Graph(sequence), "out": [x] + outs}


def _run_decode(s):
    s["graph"].launch()
    return s["out"]


def _prepare_head(case, gen):
    fmt, rows, cols = case["fmt"], case["rows"], case["cols"]
    s = {"w": _weight(gen, fmt, rows, cols), "table": _weight(gen, fmt, rows, cols), "x": _hidden(gen, cols), "norm": _norm_weight(gen, cols),
         "normed": _f32(cols), "logits": _f32(rows), "token": torch.empty(1, dtype=torch.int32, device="cuda"), "row": _f32(cols)}
    s["ws"] = _workspace(lib().cml_matmul_workspace_bytes(s["w"].fmt, cols, 1))
    return s


def _run_head(s):
    L, w = lib(), s["w"]
    check(L.cml_rms_norm_quantize(ACT_F32, s["x"].data_ptr(), s["norm"].data_ptr(), EPS, 1, w.cols, s["normed"].data_ptr(), None, None, None))
    check(L.cml_matmul_f32(w.handle, s["normed"].data_ptr(), 1, s["logits"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(), None))
    check(L.cml_argmax_f32(s["logits"].data_ptr(), 1, w.rows, s["token"].data_ptr(), None))
    check(L.cml_embed_gather(s["table"].handle, s["token"].data_ptr(), 1, s["row"].data_ptr(), None))
    return [s["logits"], s["token"], s["row"]]


def _prepare_ffn(case, gen):
    fmt, hidden, ff, tokens = case["fmt"], case["hidden"], case["ff"], case["tokens"]
    return {"tokens": tokens, "hidden": hidden, "ff": ff, "x": _hidden(gen, tokens, hidden), "norm": _norm_weight(gen, hidden),
            "gate": _weight(gen, fmt, ff, hidden), "up": _weight(gen, fmt, ff, hidden), "down": _weight(gen, case["down"], hidden, ff),
            "in": _quantized(fmt, tokens, hidden), "mid": _quantized(case["down"], tokens, ff),
            "g": _f32(tokens, ff), "u": _f32(tokens, ff), "out": _f32(tokens, hidden)}


def _run_ffn(s):
    L, tokens = lib(), s["tokens"]
    act, q, d = s["in"]
    check(L.cml_rms_norm_quantize(act, s["x"].data_ptr(), s["norm"].data_ptr(), EPS, tokens, s["hidden"], None, q.data_ptr(), d.data_ptr(), None))
    check(L.cml_gemm(s["gate"].handle, q.data_ptr(), d.data_ptr(), tokens, s["g"].data_ptr(), None))
    check(L.cml_gemm(s["up"].handle, q.data_ptr(), d.data_ptr(), tokens, s["u"].data_ptr(), None))
    act, q, d = s["mid"]
    check(L.cml_glu_quantize(SILU, act, s["g"].data_ptr(), s["u"].data_ptr(), tokens, s["ff"], q.data_ptr(), d.data_ptr(), None))
    check(L.cml_gemm(s["down"].handle, q.data_ptr(), d.data_ptr(), tokens, s["out"].data_ptr(), None))
    return s["out"]


def _prepare_experts(case, gen, fmt, fused):
    experts, hidden, ff, tokens, k = case["experts"], case["hidden"], case["ff"], case["tokens"], case["k"]
    s = {"x": _hidden(gen, tokens, hidden), "logits": 1.5 * torch.randn(tokens, experts, generator=gen, device="cuda"), "out": _f32(tokens, hidden),
         "down": _weight(gen, fmt, experts * hidden, ff), "experts": experts, "k": k, "tokens": tokens,
         "gate": _weight(gen, fmt, experts * ff * (2 if fused else 1), hidden), "up": None if fused else _weight(gen, fmt, experts * ff, hidden)}
    s["ws"] = _workspace(lib().cml_moe_workspace_bytes(B.FORMATS[fmt], hidden, ff, tokens, k, experts))
    if fused:
        s["idx"], s["weight"] = torch.empty(tokens, k, dtype=torch.int32, device="cuda"), _f32(tokens, k)
        s["scale"] = torch.exp(0.1 * torch.randn(experts, generator=gen, device="cuda"))
    return s


def _run_mixtral(s):
    check(lib().cml_moe_ffn_logits(s["gate"].handle, s["up"].handle, s["down"].handle, s["experts"], s["k"], s["logits"].data_ptr(), s["x"].data_ptr(),
                                   s["tokens"], s["out"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(), None))
    return s["out"]


def _run_gemma(s):
    L = lib()
    check(L.cml_moe_route_softmax_top_k(s["logits"].data_ptr(), s["tokens"], s["experts"], s["k"], s["scale"].data_ptr(), s["idx"].data_ptr(),
                                        s["weight"].data_ptr(), None))
    check(L.cml_moe_ffn_ex(s["gate"].handle, None, s["down"].handle, s["experts"], s["k"], s["idx"].data_ptr(), s["weight"].data_ptr(), s["x"].data_ptr(),
                           s["tokens"], s["out"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(), GELU_TANH, None))
    return [s["idx"], s["weight"], s["out"]]


_host_weights = []  # the seam caches a weight by its host address: an address must not be used again for other bytes


def _prepare_seam(case, gen):
    B.init(0)
    fmt, rows, cols, tokens = case["fmt"], case["rows"], case["cols"], case["tokens"]
    wire = _synth_wire(gen, fmt, rows, cols).cpu().numpy()
    _host_weights.append(wire)
    per = 256 if fmt == "Q4_K" else 32
    x = _hidden(gen, tokens, cols).reshape(tokens, -1, per)
    scales = (x.abs().amax(2) / 127).half().float()
    q = (x / scales.unsqueeze(2)).round().clamp(-127, 127).to(torch.int8).cpu().numpy()
    scales, out = scales.cpu().numpy(), np.empty((tokens, rows), np.float32)
    call = (B.FORMATS[fmt], scales.ctypes.data, q.ctypes.data, wire.ctypes.data, wire.nbytes, tokens, rows, cols, out.ctypes.data)
    check(lib().cml_try_linear_rows(*call))  # the weight goes to the device when the model is loaded
    return {"keep": (wire, scales, q), "call": call, "out": out}


def _run_seam(s):
    check(lib().cml_try_linear_rows(*s["call"]))
    return s["out"]


_RUN = {"linear": _run_linear, "decode": _run_decode, "head": _run_head, "ffn": _run_ffn, "mixtral": _run_mixtral, "gemma": _run_gemma, "seam": _run_seam}


def prepare(case, seed):
    B.init(0)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "mixtral":
        state = _prepare_experts(case, gen, "Q4_K", False)
    elif kind == "gemma":
        state = _prepare_experts(case, gen, case["fmt"], True)
    else:
        make = {"linear": _prepare_linear, "decode": _prepare_decode, "head": _prepare_head, "ffn": _prepare_ffn, "seam": _prepare_seam}[kind]
        state = make(case, gen)
    state["run"] = _RUN[kind]
    return state


def run(state):
    return state["run"](state)


def work(case):
    kind = case["kind"]
    if kind in ("linear", "seam"):
        fmt, rows, cols, t = case["fmt"], case["rows"], case["cols"], case["tokens"]
        per_in = 4 if kind == "linear" else 1
        return {"bytes": wire_bytes(fmt, rows, cols) + t * (per_in * cols + 4 * rows), "flops": 2 * rows * cols * t}
    if kind == "decode":
        hidden, ff, kv, fmt = case["hidden"], case["ff"], case["kv"], case["fmt"]
        total = flops = 0
        for i in range(case["layers"]):
            v_fmt, down_fmt = _decode_formats(fmt, i)
            total += (2 * wire_bytes(fmt, hidden, hidden) + wire_bytes(fmt, kv, hidden) + wire_bytes(v_fmt, kv, hidden) + 2 * wire_bytes(fmt, ff, hidden) +
                      wire_bytes(down_fmt, hidden, ff) + 4 * (2 * hidden + 2 * kv))
            flops += 2 * (2 * hidden * hidden + 2 * kv * hidden + 3 * ff * hidden)
        return {"bytes": total + 8 * hidden, "flops": flops}
    if kind == "head":
        fmt, rows, cols = case["fmt"], case["rows"], case["cols"]
        return {"bytes": wire_bytes(fmt, rows, cols) + 4 * rows + 12 * cols, "flops": 2 * rows * cols}
    if kind == "ffn":
        hidden, ff, t = case["hidden"], case["ff"], case["tokens"]
        return {"bytes": 2 * wire_bytes(case["fmt"], ff, hidden) + wire_bytes(case["down"], hidden, ff) + 8 * t * hidden, "flops": 6 * hidden * ff * t}
    experts, k, hidden, ff, t = case["experts"], case["k"], case["hidden"], case["ff"], case["tokens"]
    touched = experts * (1 - (1 - k / experts) ** t)  # experts that the tokens are routed to, on average
    one = 3 * wire_bytes(case.get("fmt", "Q4_K"), ff, hidden)
    return {"bytes": touched * one + t * (8 * hidden + 4 * experts), "flops": 6 * hidden * ff * k * t}


def tolerance(case):
    # Four times what the same path gives with the f32 sums of a row taken in the reference's other orders.
    if case["kind"] in ("linear", "seam"):  # integer products are exact; the sums over the blocks of a row differ by rounding: 7.4e-7, at most 3.8e-6
        return {"rel": 3e-6, "max": 1.5e-5}
    if case["kind"] == "head":
        return {"rel": 3e-6, "max": 1.5e-5, "differ": 0.0}
    # several projections: a last-bit difference turns a few quants of the next activation by one (2.0e-4, at most 3.8e-3)
    return {"rel": 8e-4, "max": 1.6e-2}
