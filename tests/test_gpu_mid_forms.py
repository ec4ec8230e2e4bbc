"""Every form the few-token kernel and its operand launch plan for Q4_K and Q6_K, on the shapes that take
them: one or two operand tiles (four or eight waves), hi and lo rows or f16 ones, one K range or several,
ranges whose units a thread of the operand launch holds in one or two registers or reads twice, ragged
rows, several groups of tokens.

Two or three rows of every 128 hold weights (at offsets that reach every lane over the blocks), the others
zeros: the reference, in 64 bits, takes those rows only. Tolerances as in the kernel's other tests: 1e-5 for
hi and lo operands, 2e-3 for f16 ones."""
import numpy as np
import pytest

from fak_amd import synth
from tests import test_gpu_q4k_mid as q4k, test_gpu_q6k_mid as q6k
from tests.gpu_util import q4k_matmul, rel_err_rows, spread_rows
from tests.test_gpu_q6k import dev_matmul as q6k_matmul

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,out,in_,P", [
    # two operand tiles: the 7B and 27B shapes at 33..64 tokens, two groups, long ranges with and without a split
    ("q4k", 18900, 3584, 33), ("q4k", 18900, 3584, 61), ("q4k", 3500, 18944, 64), ("q4k", 5001, 4352, 65),
    ("q4k", 45000, 1024, 40), ("q4k", 45003, 2560, 33), ("q4k", 45000, 4352, 33), ("q4k", 20000, 12800, 48),
    ("q6k", 18900, 3584, 33), ("q6k", 18900, 3584, 61), ("q6k", 3500, 18944, 64), ("q6k", 5001, 2560, 100),
    ("q6k", 45000, 1024, 40), ("q6k", 45003, 2560, 33), ("q6k", 45000, 4352, 33), ("q6k", 20000, 12800, 48),
    # one operand tile
    ("q4k", 16001, 4352, 64), ("q4k", 300, 262144, 33), ("q4k", 3100, 1024, 50), ("q4k", 5000, 2560, 100),
    ("q4k", 20, 262144, 17), ("q6k", 16001, 4352, 64), ("q6k", 300, 262144, 33), ("q6k", 3100, 1024, 100),
    ("q6k", 12301, 2560, 64), ("q6k", 20, 262144, 17),
    # hi and lo rows
    ("q4k", 9001, 1024, 16), ("q4k", 30001, 2560, 9), ("q6k", 30000, 4352, 16), ("q6k", 20003, 12800, 2),
    ("q6k", 20000, 1024, 2), ("q6k", 30001, 2560, 5), ("q6k", 30000, 4352, 2)])
def test_forms(hip, fmt, out, in_, P):
    print(f"[case] mid forms {fmt} out={out} in={in_} P={P}", flush=True)
    nb, size = in_ // 256, 144 if fmt == "q4k" else 210
    rows = spread_rows(out, per_block=3 if out > 1000 else 20)
    few = (synth.q4k_weights if fmt == "q4k" else q6k.weights)(len(rows), in_, seed=out + in_)
    raw = np.zeros((out, nb * size), np.uint8)
    raw[rows] = few.reshape(len(rows), nb * size)
    X = synth.activations(P, in_, P)
    Y = (q4k_matmul if fmt == "q4k" else q6k_matmul)(raw.reshape(-1), out, in_, X, P)
    exact = (q4k if fmt == "q4k" else q6k).exact(few, len(rows), in_, X)
    assert rel_err_rows(Y[:, rows], exact) <= (1e-5 if P <= 16 else 2e-3)
    Y[:, rows] = 0
    assert not Y.any()
