"""The Q6_K kernel for a few tokens to a few tens (quant_mid_kernel) at the edges of its tiles: rows around
a workgroup's 128, one super-block to ranges that are no multiple of its three-stage passes, grids that
the 8 XCDs divide unevenly, hi and lo rows up to 16 tokens, tiles of 32 above, several groups of tokens,
against the weights decoded from the layout, summed in 64 bits. (Two operand tiles, 256 rows:
test_gpu_mid_forms.py.)

Tolerances, max|d|/RMS: up to 16 tokens an activation carries 22 bits below its range's largest magnitude
and every weight operand is exact, so the error is a few 2^-22: 1e-5. Above, activations are f16 (2^-11
of each, rounding errors independent): about 2.2e-4 RMS of an output, and the largest of 1e5 outputs
under 6 times that: 2e-3."""
import numpy as np
import pytest

from fak_amd import synth
from tests import q6k_cases as qc
from tests.gpu_util import rel_err_rows, scaled_activations
from tests.test_gpu_q6k import dev_matmul

pytestmark = pytest.mark.gpu


def weights(out, in_, seed):
    rng = np.random.default_rng(seed)
    return qc.pin_d(rng.integers(0, 256, size=out * (in_ // 256) * 210, dtype=np.uint8), 0x1400)


def exact(raw, out, in_, X):
    w = qc.numpy_decode(raw).reshape(out, in_)
    return X.astype(np.float64) @ w.astype(np.float64).T


def tol(P):
    return 1e-5 if P <= 16 else 2e-3


@pytest.mark.parametrize("out,in_,P", [(9, 256, 2), (127, 256, 16), (129, 512, 17), (260, 768, 32),
                                       (257, 1024, 33), (3584, 3584, 4), (300, 18944, 12),
                                       (3100, 24832, 3), (3000, 4096, 64), (2600, 2560, 50),
                                       (640, 1792, 65), (1100, 5376, 128), (127, 768, 16),
                                       (129, 768, 17), (129, 512, 9), (130, 512, 32)])
def test_shapes(hip, out, in_, P):
    print(f"[case] q6k mid out={out} in={in_} P={P}", flush=True)
    raw = weights(out, in_, seed=out + in_)
    X = synth.activations(P, in_, P)
    assert rel_err_rows(dev_matmul(raw, out, in_, X, P), exact(raw, out, in_, X)) <= tol(P)


@pytest.mark.parametrize("P", [2, 9, 40])
@pytest.mark.parametrize("pattern", ["all", "wee"])
def test_scales_and_special_values(hip, pattern, P):
    """Any finite activation scale; a NaN or an infinity stays in its own token."""
    out, in_ = 200, 2048
    print(f"[case] q6k mid {pattern} P={P}", flush=True)
    raw = weights(out, in_, seed=3)
    X = scaled_activations(P, in_, 5, pattern)
    ref = exact(raw, out, in_, X)
    X[0, 100], X[P - 1, 2047] = np.nan, -np.inf
    Y = dev_matmul(raw, out, in_, X, P)
    assert np.isnan(Y[[0, P - 1]]).all()
    if P > 2:
        assert rel_err_rows(Y[1:P - 1], ref[1:P - 1]) <= tol(P)


def test_extreme_codes_and_scales(hip):
    """Every (code, scale) product is exact in its two operands: all 64 codes under scales -128 and 127."""
    out, in_, P = 64, 1024, 5
    print("[case] q6k mid extremes", flush=True)
    raw = weights(out, in_, seed=9).reshape(-1, 210)
    raw[:, 192:208] = np.tile(np.array([128, 127], np.uint8), (len(raw), 8))
    raw = raw.reshape(-1)
    X = synth.activations(P, in_, 2)
    assert rel_err_rows(dev_matmul(raw, out, in_, X, P), exact(raw, out, in_, X)) <= 1e-5


@pytest.mark.parametrize("P", [16, 17, 31])
def test_rows_too_long_for_it(hip, P):
    out, in_ = 40, 262144 + 256
    print(f"[case] q6k long rows P={P}", flush=True)
    raw = weights(out, in_, seed=4)
    X = synth.activations(P, in_, 8)
    assert rel_err_rows(dev_matmul(raw, out, in_, X, P), exact(raw, out, in_, X)) <= 1e-5
