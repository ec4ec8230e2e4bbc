"""The Q4_K kernel for a few tokens to a few tens (quant_mid_kernel) at the edges of its tiles: rows
around a workgroup's 128, one super-block to ranges that are no multiple of its three-stage passes,
hi and lo rows up to 16 tokens, tiles of 32 above, several groups of tokens, against the weights
dequantized on the host in 64 bits. (Two operand tiles, 256 rows: test_gpu_mid_forms.py.)

Tolerances, max|d|/RMS: up to 16 tokens an activation carries 22 bits below its range's largest
magnitude and every product is exact, so the error is a few 2^-22: 1e-5. Above, activations are f16
(2^-11 of each, rounding errors independent): about 2.2e-4 RMS of an output, and the largest of 1e5
outputs under 6 times that: 2e-3."""
import numpy as np
import pytest

from fak_amd import synth
from tests.gpu_util import (Dev, q4k_matmul, q4k_matmul_group, rel_err_rows, scaled_activations,
                            spread_rows)

pytestmark = pytest.mark.gpu


def exact(raw, out, in_, X):
    blk = raw.reshape(-1, 144)
    d = blk[:, 0:4].copy().view(np.float16).astype(np.float64)
    s = blk[:, 4:16].astype(np.int64)
    sc, mn = np.empty((len(blk), 8)), np.empty((len(blk), 8))
    for j in range(4):
        sc[:, j], mn[:, j] = s[:, j] & 63, s[:, j + 4] & 63
        sc[:, j + 4] = (s[:, j + 8] & 15) | (s[:, j] >> 6) << 4
        mn[:, j + 4] = (s[:, j + 8] >> 4) | (s[:, j + 4] >> 6) << 4
    q = blk[:, 16:].reshape(-1, 4, 32)
    q = np.stack((q & 15, q >> 4), 2).reshape(-1, 8, 32).astype(np.float64)
    w = (d[:, 0:1] * sc)[:, :, None] * q - (d[:, 1:2] * mn)[:, :, None]
    return X.astype(np.float64) @ w.reshape(out, in_).T


def tol(P):
    return 1e-5 if P <= 16 else 2e-3


@pytest.mark.parametrize("out,in_,P", [(1, 256, 5), (127, 256, 16), (129, 512, 17), (260, 768, 32),
                                       (257, 1024, 33), (3584, 3584, 8), (300, 18944, 12),
                                       (5000, 4096, 64), (9000, 2560, 50), (640, 1792, 65),
                                       (1100, 5376, 128)])
def test_shapes(hip, out, in_, P):
    print(f"[case] q4k mid out={out} in={in_} P={P}", flush=True)
    raw = synth.q4k_weights(out, in_, seed=out + in_)
    X = synth.activations(P, in_, P)
    assert rel_err_rows(q4k_matmul(raw, out, in_, X, P), exact(raw, out, in_, X)) <= tol(P)


@pytest.mark.parametrize("P", [9, 40])
@pytest.mark.parametrize("pattern", ["all", "wee"])
def test_scales_and_special_values(hip, pattern, P):
    """Any finite activation scale; a NaN or an infinity stays in its own token."""
    out, in_ = 200, 2048
    print(f"[case] q4k mid {pattern} P={P}", flush=True)
    raw = synth.q4k_weights(out, in_, seed=3)
    X = scaled_activations(P, in_, 5, pattern)
    ref = exact(raw, out, in_, X)
    X[2, 100], X[P - 1, 2047] = np.nan, -np.inf
    Y = q4k_matmul(raw, out, in_, X, P)
    assert np.isnan(Y[[2, P - 1]]).all()
    keep = [t for t in range(P) if t not in (2, P - 1)]
    assert rel_err_rows(Y[keep], ref[keep]) <= tol(P)


def test_group_members(hip):
    outs, in_, P = [520, 130, 64], 1536, 11
    print("[case] q4k mid group", flush=True)
    raws = [synth.q4k_weights(o, in_, seed=o) for o in outs]
    X = synth.activations(P, in_, 1)
    for raw, o, y in zip(raws, outs, q4k_matmul_group(raws, outs, in_, X, P)):
        assert rel_err_rows(y, exact(raw, o, in_, X)) <= 1e-5


@pytest.mark.parametrize("out,in_,P", [(78848, 2560, 64), (2048, 65536, 64), (40, 262144, 32)])
def test_scratch_stays_small(hip, out, in_, P):
    """Operands and partial results fit the no-allocation entry's 64 MiB at tall and at long weights; both
    entries give the same bits, right on rows of every 128."""
    lib = hip.load()
    print(f"[case] q4k mid scratch out={out} in={in_} P={P}", flush=True)
    raw = synth.q4k_weights(out, in_, seed=1)
    w = hip.alloc_call("fhip_q4k_upload", np.ascontiguousarray(raw).ctypes.data, out, in_)
    try:
        X = synth.activations(P, in_, 1)
        with Dev.from_host(X) as dx, Dev(P * out * 4) as dy:
            hip.call("fhip_q4k_matmul_noalloc_f32", w, dx.ptr, dy.ptr, out, in_, P)
            Y = dy.to_host(np.float32).reshape(P, out)
            hip.call("fhip_q4k_matmul_f32", w, dx.ptr, dy.ptr, out, in_, P)
            np.testing.assert_array_equal(Y, dy.to_host(np.float32).reshape(P, out))
            rows = spread_rows(out, per_block=1)
            sub = raw.reshape(out, -1)[rows].reshape(-1)
            assert rel_err_rows(Y[:, rows], exact(sub, len(rows), in_, X)) <= tol(P)
    finally:
        lib.fhip_free(w)
