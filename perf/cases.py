"""The workloads this library's speed is judged on, as a program that serves GGUF models calls it.

Weights are raw GGUF blocks with the statistics of fak_amd/synth.py (drawn on the device),
repacked once into the tiled layout, as a program keeps them; activations are f32 N(0, 1). One pass
is one call of a public entry on the default stream. Shapes are the repository's own: SmolLM2-135M's
576 -> 1536 (Q8_0), Qwen2.5-7B's attention and FFN (hidden 3584, inter 18944) and the 27B FFN
(5120 x 25600).
"""
import math

import numpy as np
import torch

from fak_amd import fakhip

# Formats: raw bytes and weights of a block, and the ABI's prefix.
FORMATS = {
    "q4k": (144, 256, "fhip_q4k"),
    "q6k": (210, 256, "fhip_q6k"),
    "q8_0": (34, 32, "fhip_q8_0"),
}


def listed():
    return [
        # The smallest call: a SmolLM2-135M FFN projection of one decoded token.
        {"name": "q8_0_decode_576x1536", "kind": "q8_0", "out": 1536, "in": 576, "P": 1},
        # One decoded token of a 7B layer: q, k and v as one grouped call.
        {"name": "q4k_qkv_decode_7b", "kind": "group", "out": 3584, "out_kv": 512, "in": 3584, "P": 1},
        # One decoded token through a 7B gate or up projection.
        {"name": "q4k_decode_7b", "kind": "q4k", "out": 18944, "in": 3584, "P": 1},
        # One decoded token through the whole FFN of a q4_k_m file (Q6_K down projection).
        {"name": "mlp_q6down_decode_7b", "kind": "mlp", "out": 18944, "in": 3584, "P": 1},
        # Speculative verify of eight tokens, 27B gate or up projection.
        {"name": "q4k_verify8_27b", "kind": "q4k", "out": 25600, "in": 5120, "P": 8},
        # A short prompt (or the tail chunk of a long one): an odd number of tokens.
        {"name": "q4k_prefill77_7b", "kind": "q4k", "out": 18944, "in": 3584, "P": 77},
        # A prefill chunk.
        {"name": "q4k_prefill512_7b", "kind": "q4k", "out": 18944, "in": 3584, "P": 512},
        # The largest: a long prompt in one chunk.
        {"name": "q4k_prefill2048_7b", "kind": "q4k", "out": 18944, "in": 3584, "P": 2048},
        # A prefill chunk through the Q6_K down projection of a q4_k_m file.
        {"name": "q6k_prefill512_down_7b", "kind": "q6k", "out": 3584, "in": 18944, "P": 512},
        # A prompt of a Q8_0 model.
        {"name": "q8_0_prefill128", "kind": "q8_0", "out": 3584, "in": 3584, "P": 128},
        # A decoded token on the backend's own Q8 tensors (f32 weights narrowed at upload).
        {"name": "hal_q8_decode", "kind": "hal", "out": 3584, "in": 3584, "P": 1},
        # A decoded token on the opt-in int8 route (the CPU path's bits).
        {"name": "q4k_int8_decode_7b", "kind": "int8", "out": 18944, "in": 3584, "P": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another call of the same kinds: any output size (odd ones too), any reduction size the format
    takes, any width from decode to the longest chunk of its kind."""
    kind = rng.choice(["q4k", "q4k", "q4k", "q4k", "group", "mlp", "q6k", "q6k", "q8_0", "q8_0", "hal", "int8"])
    if kind in ("q8_0", "hal"):
        in_ = 32 * _log(rng, 18, 592)  # 576 .. 18944
    else:
        in_ = 256 * _log(rng, 4, 100)  # 1024 .. 25600
    out = _log(rng, 500, min(25600, 131072000 // in_))
    case = {"kind": kind, "out": out, "in": in_}
    if kind == "mlp":  # out: the intermediate size
        case["out"] = max(256, out // 256 * 256)
        case["P"] = rng.randint(1, 4)
    elif kind == "group":
        case["out_kv"] = _log(rng, 128, 2048)
        case["P"] = _log(rng, 1, 16)
    elif kind in ("hal", "int8"):
        case["P"] = _log(rng, 1, 64)
    elif kind == "q8_0":
        case["P"] = _log(rng, 1, 512)
    else:
        case["P"] = _log(rng, 1, 2048)
    return case


def _generator(seed, part):
    g = torch.Generator("cuda")
    g.manual_seed(1000003 * (seed + 1) + part)
    return g


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).view(v.shape + (2,))


def _raw(fmt, out, in_, g):
    """Raw row-major GGUF blocks on the device, [out * in / block, block bytes] uint8."""
    size, block, _ = FORMATS[fmt]
    n = out * (in_ // block)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda").abs()

    raw = torch.randint(0, 256, (n, size), generator=g, device="cuda", dtype=torch.uint8)
    if fmt == "q4k":  # d, dmin, then uniform 6-bit scales and mins and uniform nibbles
        raw[:, 0:4] = _f16_bytes(normal(n, 2) * 1e-3).view(n, 4)
    elif fmt == "q6k":
        raw[:, 208:210] = _f16_bytes(normal(n) * 1e-3)
    else:
        raw[:, 0:2] = _f16_bytes(normal(n) * 0.002)
        raw[:, 2:] = raw[:, 2:].clamp(1).add(128)  # int8 codes -127 .. 127
    return raw


def _weights(case, seed):
    """The raw weights of a case, as (format, out, in, blocks), in call order."""
    kind, out, in_ = case["kind"], case["out"], case["in"]
    if kind == "group":
        shapes = [("q4k", out, in_), ("q4k", case["out_kv"], in_), ("q4k", case["out_kv"], in_)]
    elif kind == "mlp":
        shapes = [("q4k", out, in_), ("q4k", out, in_), ("q6k", in_, out)]
    else:
        shapes = [("q4k" if kind == "int8" else kind, out, in_)]
    for i, (fmt, o, k) in enumerate(shapes):
        yield fmt, o, k, _raw(fmt, o, k, _generator(seed, i))


def _hal_weights(case, seed):
    """HAL Q8 codes [out][in] and f32 scales per 32 values."""
    g = _generator(seed, 0)
    codes = torch.randint(-127, 128, (case["out"], case["in"]), generator=g, device="cuda", dtype=torch.int8)
    scales = torch.randn(case["out"], case["in"] // 32, generator=g, device="cuda").abs() * 0.002
    return codes, scales


def _activations(case, seed):
    return torch.randn(case["P"], case["in"], generator=_generator(seed, 100), device="cuda")


class Weight:
    """A tiled weight in the library's own memory."""

    def __init__(self, fmt, out, in_, raw):
        prefix = FORMATS[fmt][2]
        self.ptr = fakhip.alloc_call("fhip_malloc", getattr(fakhip.load(), prefix + "_packed_bytes")(out, in_))
        fakhip.call(prefix + "_repack", self.ptr, raw.data_ptr(), out, in_)

    def __del__(self):
        if getattr(self, "ptr", 0):
            fakhip.load().fhip_free(self.ptr)


_ready = []


def prepare(case, seed):
    if not _ready:
        _ready.append(fakhip.init())
    kind, out, in_, P = case["kind"], case["out"], case["in"], case["P"]
    x = _activations(case, seed)
    state = {"x": x}
    if kind == "hal":
        w = _hal_weights(case, seed)
        outs = [out]
        args = ("fhip_q8_matmul_f32", w[0].data_ptr(), w[1].data_ptr(), x.data_ptr(), None, out, in_, P, 32)
    else:
        w = [Weight(*v) for v in _weights(case, seed)]
        torch.cuda.synchronize()
        if kind == "group":
            outs = [out, case["out_kv"], case["out_kv"]]
            args = None
        elif kind == "mlp":
            outs = [in_]
            args = ("fhip_q4k_mlp_q6down_f32", w[0].ptr, w[1].ptr, w[2].ptr, x.data_ptr(), None, in_, out, P)
        else:
            outs = [out]
            entry = {"int8": "fhip_q4k_matmul_int8_f32"}.get(kind, "fhip_%s_matmul_f32" % kind)
            args = (entry, w[0].ptr, x.data_ptr(), None, out, in_, P)
    y = [torch.zeros(P, o, device="cuda") for o in outs]
    if kind == "group":
        n = len(outs)
        ptrs = (fakhip.C.c_void_p * n)(*[v.ptr for v in w])
        ys = (fakhip.C.c_void_p * n)(*[v.data_ptr() for v in y])
        args = ("fhip_q4k_matmul_group_f32", ptrs, ys, (fakhip.C.c_int * n)(*outs), n, x.data_ptr(), in_, P)
    else:
        args = tuple(y[0].data_ptr() if a is None else a for a in args)
    state.update(w=w, y=y, args=args)
    return state


def run(state):
    fakhip.call(*state["args"])
    return state["y"]


def _weight_bytes(case):
    kind, out, in_ = case["kind"], case["out"], case["in"]
    if kind == "group":
        return (out + 2 * case["out_kv"]) * (in_ // 256) * 144
    if kind == "mlp":
        return 2 * out * (in_ // 256) * 144 + in_ * (out // 256) * 210
    if kind == "hal":
        return out * in_ + out * (in_ // 32) * 4
    size, block, _ = FORMATS["q4k" if kind == "int8" else kind]
    return out * (in_ // block) * size


def work(case):
    kind, out, in_, P = case["kind"], case["out"], case["in"], case["P"]
    rows = out + 2 * case["out_kv"] if kind == "group" else in_ if kind == "mlp" else out
    macs = 3 * out * in_ if kind == "mlp" else rows * in_
    return {"bytes": _weight_bytes(case) + 4 * P * (in_ + rows), "flops": 2 * P * macs}


def tolerance(case):
    """About four times the error against 64 bits that each route shows (in brackets): decode and
    verify carry 22 and more bits of an activation (Q4_K 1.4e-7, Q8_0 1.8e-6), the Q6_K decode two
    int8 digits of it (6e-5), wider Q4_K and Q6_K calls f16 activations and f16-rounded weights
    (3.7e-4). The HAL and int8 routes are the CPU path's bits."""
    kind, P = case["kind"], case["P"]
    if kind in ("hal", "int8"):
        return "exact"
    if kind == "mlp" or (kind == "q6k" and P == 1):
        return {"rel": 2.5e-4, "max": 2.5e-3}
    if kind == "q8_0":
        return {"rel": 8e-6, "max": 8e-5}
    if P <= 16:
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 1.5e-3, "max": 1e-2}


def _dequant(fmt, out, in_, raw):
    """The weight in 64 bits, [out, in]."""
    n = raw.shape[0]

    def f16(a):
        return a.contiguous().view(torch.float16).double()

    if fmt == "q8_0":
        w = f16(raw[:, 0:2]) * raw[:, 2:].contiguous().view(torch.int8).double()
        return w.view(out, in_)
    if fmt == "q4k":
        s = raw[:, 4:16].long()
        scale, low = torch.empty(n, 8, device="cuda").double(), torch.empty(n, 8, device="cuda").double()
        for j in range(8):  # 6-bit scales and mins in 12 bytes
            if j < 4:
                scale[:, j], low[:, j] = s[:, j] & 63, s[:, j + 4] & 63
            else:
                scale[:, j] = (s[:, j + 4] & 15) | (s[:, j - 4] >> 6) << 4
                low[:, j] = (s[:, j + 4] >> 4) | (s[:, j] >> 6) << 4
        d, dmin = f16(raw[:, 0:2]), f16(raw[:, 2:4])
        q = raw[:, 16:].view(n, 4, 32)
        q = torch.stack((q & 15, q >> 4), 2).view(n, 8, 32).double()
        w = (d * scale).unsqueeze(2) * q - (dmin * low).unsqueeze(2)
        return w.view(out, in_)
    ql, qh = raw[:, 0:128].view(n, 2, 64), raw[:, 128:192].view(n, 2, 32)
    parts = []
    for i in range(4):  # quarter i of each half: 32 low nibbles and a 2-bit field of qh
        lo = ql[:, :, 32 * (i & 1):32 * (i & 1) + 32]
        lo = lo >> 4 if i >= 2 else lo & 15
        parts.append(lo | ((qh >> (2 * i)) & 3) << 4)
    q = torch.stack(parts, 2).view(n, 16, 16).double() - 32.0
    scale = raw[:, 192:208].contiguous().view(torch.int8).double()
    return (f16(raw[:, 208:210]).unsqueeze(2) * scale.unsqueeze(2) * q).view(out, in_)


def _quantized(x):
    """The activation as the int8 routes see it: codes times f32 scales per 32 values, in 64 bits."""
    v = x.cpu().numpy().reshape(x.shape[0], -1, 32)
    d = np.abs(v).max(2, keepdims=True) / np.float32(127)
    s = v * (np.float32(1) / d)
    t = np.trunc(s)
    f = s - t
    t = np.clip(t + (f >= 0.5) - (f <= -0.5), -127, 127)
    return torch.from_numpy((t.astype(np.float64) * d.astype(np.float64)).reshape(x.shape)).cuda()


def exact(case, seed):
    kind = case["kind"]
    x = _activations(case, seed)
    x = _quantized(x) if kind in ("hal", "int8") else x.double()
    if kind == "hal":
        codes, scales = _hal_weights(case, seed)
        w = codes.double().view(case["out"], -1, 32) * scales.double().unsqueeze(2)
        return [x @ w.view(case["out"], -1).T]
    w = [_dequant(*v) for v in _weights(case, seed)]
    if kind == "mlp":
        gate, up = x @ w[0].T, x @ w[1].T
        return [(gate * torch.sigmoid(gate) * up) @ w[2].T]
    return [x @ v.T for v in w]
