"""Super-blocks far below their K range's largest magnitude are all an output of Q4_K or Q6_K sees where the
larger super-blocks meet zero weights: up to 32 tokens they keep the bits of their route, at every ratio, in
ranges of one super-block to eighteen, in the tokens that have them and in ordinary tokens beside them.

Most rows are zero: the reference (64 bits) takes the others. Tolerances, max|d|/RMS of a token's outputs: hi
and lo operands (up to 16 tokens, and rows of more than 262144 values) 1e-5; one f16 operand, 2^-11 of each
value, rounding errors independent: 2.2e-4 RMS, and the largest of 4e3 under 5 times that: 2e-3."""
import numpy as np
import pytest

from fak_amd import synth
from tests import test_gpu_q4k_mid as q4k, test_gpu_q6k_mid as q6k
from tests.gpu_util import q4k_matmul, rel_err_rows
from tests.test_gpu_q6k import dev_matmul as q6k_matmul

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,out,in_,P", [("q4k", 200, 2048, 7), ("q4k", 3072, 32512, 16), ("q4k", 257, 768, 17),
                                           ("q4k", 30000, 9216, 24),
                                           ("q6k", 200, 2048, 2), ("q6k", 3100, 34816, 9), ("q6k", 129, 1280, 32),
                                           ("q6k", 20000, 9216, 30), ("q6k", 520, 262400, 19)])
def test_small_beside_large(hip, fmt, out, in_, P):
    print(f"[case] small beside large {fmt} out={out} in={in_} P={P}", flush=True)
    nb, size = in_ // 256, 144 if fmt == "q4k" else 210
    rows = np.unique(np.linspace(0, out - 1, 64).astype(int))
    big = np.arange(nb) % 3 == 1
    few = (synth.q4k_weights if fmt == "q4k" else q6k.weights)(len(rows), in_, seed=out + in_)
    few = few.reshape(len(rows), nb, size).copy()
    few[:, big] = 0
    raw = np.zeros((out, nb, size), np.uint8)
    raw[rows] = few
    X = synth.activations(P, in_, P).reshape(P, nb, 256)
    ratios = [1.0, 2.0 ** 12, 2.0 ** 16, 1e6, 1e24, 1e30]
    for t in range(P):
        X[t, big] *= np.float32(ratios[t % 6])
        X[t] *= np.float32([1.0, 1e-3, 1.0, 1e-20, 1e-20, 1e-34][t % 6])
    X[1, 0] = 0.0
    X = X.reshape(P, in_)
    Y = (q4k_matmul if fmt == "q4k" else q6k_matmul)(raw.reshape(-1), out, in_, X, P)
    exact = (q4k if fmt == "q4k" else q6k).exact
    tol = 1e-5 if P <= 16 or in_ > 262144 else 2e-3
    assert rel_err_rows(Y[:, rows], exact(few.reshape(-1), len(rows), in_, X)) <= tol
    Y[:, rows] = 0
    assert not Y.any()
