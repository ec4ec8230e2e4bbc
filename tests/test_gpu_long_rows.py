"""Rows far longer than a model's: every route's operand offsets must hold there too. Activations are zero
but for a few super-blocks, so the reference (64 bits, the weights decoded on the host) needs those only.

Tolerances, max|d|/RMS of a token's 16 outputs: f16 activations and f16-rounded weights (prefill GEMM),
rounding errors independent: 3.7e-4 RMS of an output, and the largest of 80 under 4 times that: 2e-3. Up
to 32 tokens hi and lo operands (22 bits) and exact weights: 1e-5."""
import ctypes as C
import time

import numpy as np
import pytest

from fak_amd import fakhip, synth
from tests import test_gpu_q4k_mid as q4k, test_gpu_q6k_mid as q6k, test_gpu_q8_0_gemm as q8_0
from tests.gpu_util import Dev, rel_err_rows

pytestmark = pytest.mark.gpu

ENTRY = {"q4k": ("fhip_q4k", 144, 256, q4k.exact, lambda o, i: synth.q4k_weights(o, i, 5)),
         "q8_0": ("fhip_q8_0", 34, 32, q8_0.exact, lambda o, i: synth.q8_0_weights(o, i, 5)),
         "q6k": ("fhip_q6k", 210, 256, q6k.exact, lambda o, i: q6k.weights(o, i, 5))}


def check(fmt, out, in_, P, tokens, blocks, tol):
    """Tokens `tokens` are N(0, 1) in the blocks (of the format: 256 or 32 values) `blocks`, all else is zero."""
    prefix, size, block, exact, weights = ENTRY[fmt]
    lib = fakhip.load()
    nb, n = in_ // block, len(blocks)
    few = weights(out, n * block)
    raw = np.zeros((out, nb, size), np.uint8)
    raw[:, blocks] = few.reshape(out, n, size)
    X = synth.activations(len(tokens), n * block, 7)
    w = fakhip.alloc_call(prefix + "_upload", raw.ctypes.data, out, in_)
    try:
        with Dev(P * in_ * 4) as dx, Dev(P * out * 4) as dy:
            fakhip.call("fhip_memset_async", dx.ptr, 0, dx.nbytes)
            fakhip.call("fhip_sync")
            for i, t in enumerate(tokens):
                for j, b in enumerate(blocks):
                    part = np.ascontiguousarray(X[i, j * block:(j + 1) * block])
                    fakhip.call("fhip_h2d", dx.ptr + 4 * (t * in_ + b * block), part.ctypes.data, part.nbytes)
            fakhip.call(prefix + "_matmul_f32", w, dx.ptr, dy.ptr, out, in_, P)
            Y = dy.to_host(np.float32).reshape(P, out)
    finally:
        lib.fhip_free(w)
        lib.fhip_trim_pool(0)
    assert rel_err_rows(Y[tokens], exact(few, out, n * block, X)) <= tol
    rest = np.setdiff1d(np.arange(P), tokens)
    assert not Y[rest].any()


@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
@pytest.mark.parametrize("in_,P", [((1 << 24) + 512, 100), ((1 << 23) + 256, 897)])
def test_prefill_gemm(hip, fmt, in_, P):
    """A 128-token tile's operands past 4 and past 2 GiB, its last token tile's last super-blocks; one
    token tile and (256-row workgroups) eight."""
    print(f"[case] long rows, prefill GEMM {fmt} in={in_} P={P}", flush=True)
    nb = in_ // 256
    check(fmt, 16, in_, P, [0, 3, 40, 99, P - 1] if P > 100 else [0, 3, 40, 99],
          [0, 1, nb // 2, nb - 2, nb - 1], 2e-3)


@pytest.mark.parametrize("fmt,out,in_,P", [("q4k", 16, 262400, 17), ("q4k", 300, 262400, 32), ("q4k", 130, 1048832, 23),
                                           ("q6k", 130, 262400, 18), ("q6k", 511, 262400, 31),
                                           ("q6k", 530, 262400, 32), ("q6k", 600, 1048576, 17),
                                           ("q6k", 513, 1048832, 20)])
def test_17_to_32_tokens(hip, fmt, out, in_, P):
    """Rows too long for the few-token kernel's f16 form: both sixteens of tokens, every range."""
    print(f"[case] long rows {fmt} out={out} in={in_} P={P}", flush=True)
    nb = in_ // 256
    check(fmt, out, in_, P, sorted({0, 1, 15, 16, P - 1}), [0, 1, 2, 5, nb // 2, nb // 2 + 1, nb - 1], 1e-5)


@pytest.mark.parametrize("out,in_,P", [(33, 1 << 21, 40), (33, (1 << 21) + 32, 2), (17, (1 << 21) + 64, 16),
                                       (50, (1 << 21) + 32, 35)])
def test_q8_0(hip, out, in_, P):
    """The longest row of the GEMM, and rows past it: the GEMV in slices of sixteen tokens."""
    print(f"[case] long rows q8_0 out={out} in={in_} P={P}", flush=True)
    nb = in_ // 32
    check("q8_0", out, in_, P, sorted({0, 1, P - 1}), [0, 1, 7, 8, nb // 2, nb // 2 + 1, nb - 2, nb - 1], 1e-5)


@pytest.mark.parametrize("in_,P", [(1 << 20, 130), ((1 << 19) + 32, 300), (65536, 1000)])
def test_q8_0_scratch(hip, in_, P):
    """A wide call of a long row keeps its scratch within 256 MiB (and the workspace's quarter over it)."""
    print(f"[case] long rows q8_0 scratch in={in_} P={P}", flush=True)
    lib, free, total = fakhip.load(), C.c_size_t(), C.c_size_t()
    raw = np.zeros(40 * (in_ // 32) * 34, np.uint8)
    w = fakhip.alloc_call("fhip_q8_0_upload", raw.ctypes.data, 40, in_)
    st = C.c_void_p()  # a stream of its own: its workspace starts empty
    fakhip.call("fhip_stream_create", C.byref(st))
    fakhip.call("fhip_set_stream", st)
    try:
        with Dev(P * in_ * 4) as dx, Dev(P * 40 * 4) as dy:
            fakhip.call("fhip_mem_info", C.byref(free), C.byref(total))
            before = free.value
            fakhip.call("fhip_q8_0_matmul_f32", w, dx.ptr, dy.ptr, 40, in_, P)
            fakhip.call("fhip_sync")
            fakhip.call("fhip_mem_info", C.byref(free), C.byref(total))
    finally:
        fakhip.call("fhip_set_stream", None)
        fakhip.call("fhip_stream_destroy", st)
        lib.fhip_free(w)
        lib.fhip_trim_pool(0)
    # scales and the partial sums of the K ranges, at most 32 MiB, come on top
    assert before - free.value <= 1.25 * (288 << 20)


def seconds(prefix, w, out, in_, P):
    with Dev(P * in_ * 4) as dx, Dev(P * out * 4) as dy:
        fakhip.call("fhip_memset_async", dx.ptr, 0, dx.nbytes)
        best = 1e9
        for _ in range(6):
            fakhip.call("fhip_sync")
            t = time.perf_counter()
            for _ in range(8):
                fakhip.call(prefix + "_matmul_f32", w, dx.ptr, dy.ptr, out, in_, P)
            fakhip.call("fhip_sync")
            best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("fmt,out,in_,few,many,bound", [("q4k", 40, 262400, 16, 32, 1.65),
                                                        ("q6k", 40, 262400, 16, 32, 1.65),
                                                        ("q8_0", 16, 2097184, 1, 16, 6)])
def test_many_tokens_read_the_rows_together(hip, fmt, out, in_, few, many, bound):
    """Tokens one after the other, or in groups one after the other, would take `many` / `few` times as long."""
    print(f"[case] long rows, time of {many} tokens against {few}, {fmt} in={in_}", flush=True)
    prefix, size, block = ENTRY[fmt][:3]
    lib = fakhip.load()
    raw = np.zeros(out * (in_ // block) * size, np.uint8)
    w = fakhip.alloc_call(prefix + "_upload", raw.ctypes.data, out, in_)
    try:
        seconds(prefix, w, out, in_, many)  # workspaces, clocks
        assert seconds(prefix, w, out, in_, many) < bound * seconds(prefix, w, out, in_, few)
    finally:
        lib.fhip_free(w)
