"""Rows far longer than a model's: every route's operand offsets must hold there too. Activations are zero
but for a few super-blocks, so the reference (64 bits, the weights decoded on the host) needs those only.

Tolerances, max|d|/RMS of a token's 16 outputs: f16 activations and f16-rounded weights (prefill GEMM),
rounding errors independent: 3.7e-4 RMS of an output, and the largest of 80 under 4 times that: 2e-3."""
import numpy as np
import pytest

from fak_amd import fakhip, synth
from tests import test_gpu_q4k_mid as q4k, test_gpu_q6k_mid as q6k
from tests.gpu_util import Dev, rel_err_rows

pytestmark = pytest.mark.gpu

ENTRY = {"q4k": ("fhip_q4k", 144, 256, q4k.exact, lambda o, i: synth.q4k_weights(o, i, 5)),
         "q6k": ("fhip_q6k", 210, 256, q6k.exact, lambda o, i: q6k.weights(o, i, 5))}


def check(fmt, out, in_, P, tokens, blocks, tol):
    """Tokens `tokens` are N(0, 1) in the blocks (of the format's 256 values) `blocks`, all else is zero."""
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
