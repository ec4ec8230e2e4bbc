"""The Q8_0 GEMM (q8_gemm_kernel) at the edges of its tiles: rows around the workgroup's 128, one
block to an odd number of them, ranges shorter than its three-pair passes, 17 tokens (two where the
operands do not fit in the GEMV's LDS) to more than a slice of 1024, against the weights dequantized on the host in 64 bits.

Tolerance: an activation enters as two f16 operands, 22 bits below the largest magnitude of its
range (4 to 5 RMS here), so an output's error is about 1e-6 RMS, and its f32 sums add a few 2^-24 per
block: 1e-5 max|d|/RMS is several times both."""
import numpy as np
import pytest

from fak_amd import synth
from tests.gpu_util import knobs, q8_0_matmul, rel_err_rows, scaled_activations, spread_rows

pytestmark = pytest.mark.gpu


def exact(raw, out, in_, X):
    blk = raw.reshape(out, in_ // 32, 34)
    d = blk[:, :, 0:2].copy().view(np.float16).astype(np.float64)
    w = (blk[:, :, 2:].view(np.int8).astype(np.float64) * d).reshape(out, in_)
    return X.astype(np.float64) @ w.T


@pytest.mark.parametrize("out,in_,P", [(1, 32, 17), (127, 64, 32), (129, 96, 33), (260, 544, 64),
                                       (1536, 576, 65), (513, 3584, 200), (40, 18944, 96),
                                       (3584, 1056, 128), (48, 1024, 1061), (2100, 4096, 150),
                                       (16, 18944, 2), (300, 9216, 5), (65, 3584, 12)])
def test_shapes(hip, out, in_, P):
    print(f"[case] q8_0 gemm out={out} in={in_} P={P}", flush=True)
    raw = synth.q8_0_weights(out, in_, seed=out + in_)
    X = synth.activations(P, in_, P)
    assert rel_err_rows(q8_0_matmul(raw, out, in_, X, P), exact(raw, out, in_, X)) <= 1e-5


@pytest.mark.parametrize("out,in_,P", [
    # ranges of 33, 65 and 129 pairs of blocks (two, four units per thread of the operand launch, and a range
    # read twice), the last half padding, K unsplit; one token tile per workgroup, then two
    (2001, 2080, 510), (2001, 4128, 500), (1001, 8224, 1020), (4040, 2080, 500), (3601, 4128, 515),
    (3601, 8224, 520),
    # the same, K in ranges: the 7B shapes, and odd counts of blocks
    (18944, 3584, 512), (2048, 18944, 512), (3584, 18944, 512), (2100, 5152, 150), (700, 19008, 1024)])
def test_range_lengths(hip, out, in_, P):
    print(f"[case] q8_0 gemm ranges out={out} in={in_} P={P}", flush=True)
    rows = spread_rows(out)
    raw = synth.q8_0_weights(out, in_, seed=out + in_)
    X = synth.activations(P, in_, P)
    Y = q8_0_matmul(raw, out, in_, X, P)
    sub = raw.reshape(out, -1)[rows].reshape(-1)
    assert rel_err_rows(Y[:, rows], exact(sub, len(rows), in_, X)) <= 1e-5


@pytest.mark.parametrize("out,in_,P", [(16208, 6784, 3), (16208, 6784, 5), (31248, 5120, 4), (30700, 3584, 6),
                                       (39056, 4096, 5), (16650, 9600, 3), (33200, 1024, 8), (18944, 3584, 8),
                                       (40000, 1056, 8), (40000, 1056, 9)])
def test_few_tokens_of_a_large_matrix(hip, out, in_, P):
    """Three to eight tokens of 32 M weights and more, on either side of the rule that picks the GEMV or the
    GEMM, and nine."""
    print(f"[case] q8_0 few tokens out={out} in={in_} P={P}", flush=True)
    rows = spread_rows(out)
    few = synth.q8_0_weights(len(rows), in_, seed=out + in_)
    raw = np.zeros((out, in_ // 32 * 34), np.uint8)
    raw[rows] = few.reshape(len(rows), -1)
    X = synth.activations(P, in_, P)
    Y = q8_0_matmul(raw.reshape(-1), out, in_, X, P)
    assert rel_err_rows(Y[:, rows], exact(few, len(rows), in_, X)) <= 1e-5
    Y[:, rows] = 0
    assert not Y.any()


def test_three_tokens_cost_little_more_than_two(hip):
    """Where both kernels run at memory's pace, the GEMM's three launches cost a third more than the GEMV's one."""
    from tests.test_gpu_long_rows import seconds
    out, in_ = 16208, 6784
    print("[case] q8_0 time of 3 tokens against 2", flush=True)
    lib = hip.load()
    raw = np.zeros(out * (in_ // 32) * 34, np.uint8)
    w = hip.alloc_call("fhip_q8_0_upload", raw.ctypes.data, out, in_)
    try:
        seconds("fhip_q8_0", w, out, in_, 3)
        assert seconds("fhip_q8_0", w, out, in_, 3) < 1.25 * seconds("fhip_q8_0", w, out, in_, 2)
    finally:
        lib.fhip_free(w)


@pytest.mark.parametrize("pattern", ["all", "wee"])
def test_scales_and_special_values(hip, pattern):
    """Any finite activation scale, and a NaN or an infinity stays in its own token."""
    out, in_, P = 200, 2048, 40
    print(f"[case] q8_0 gemm {pattern}", flush=True)
    raw = synth.q8_0_weights(out, in_, seed=3)
    X = scaled_activations(P, in_, 5, pattern)
    ref = exact(raw, out, in_, X)
    X[7, 100], X[20, 2047] = np.nan, -np.inf
    Y = q8_0_matmul(raw, out, in_, X, P)
    assert np.isnan(Y[[7, 20]]).all()
    keep = [t for t in range(P) if t not in (7, 20)]
    # a row of one huge value is held to its RMS: 22 bits below it
    assert rel_err_rows(Y[keep], ref[keep]) <= 1e-5


@pytest.mark.parametrize("out,in_,P", [(200, 2048, 40), (129, 96, 33), (2100, 4096, 150), (40, 18944, 96),
                                       (513, 3616, 200)])
def test_small_blocks_beside_large_ones(hip, out, in_, P):
    """Blocks far below their range's largest magnitude are all an output sees where the larger blocks
    meet zero weights: they keep their 22 bits, at every ratio, in the tokens that have them and in
    ordinary tokens of the same tile."""
    print(f"[case] q8_0 gemm small beside large out={out} in={in_} P={P}", flush=True)
    raw = synth.q8_0_weights(out, in_, seed=out + in_).reshape(out, in_ // 32, 34)
    big = np.arange(in_ // 32) % 3 == 1
    raw[:, big, 2:] = 0
    X = synth.activations(P, in_, P).reshape(P, in_ // 32, 32)
    ratios = [1.0, 2.0 ** 12, 2.0 ** 16, 1e6, 1e24, 1e30]
    for t in range(P):
        X[t, big] *= np.float32(ratios[t % 6])
        X[t] *= np.float32([1.0, 1e-3, 1.0, 1e-20, 1e-20, 1e-34][t % 6])
    X[3, 0, :] = 0.0
    X = X.reshape(P, in_)
    raw = raw.reshape(-1)
    assert rel_err_rows(q8_0_matmul(raw, out, in_, X, P), exact(raw, out, in_, X)) <= 1e-5


@pytest.mark.parametrize("out,in_,P", [(200, 2048, 8), (33, 1056, 16), (3584, 3584, 3)])
def test_gemv_global_operands_forced(hip, monkeypatch, out, in_, P):
    """FAK_HIP_GEMV_GLOBALX=1: the GEMV with its operands in global memory, up to 16 tokens."""
    print(f"[case] q8_0 gemv global operands out={out} in={in_} P={P}", flush=True)
    raw = synth.q8_0_weights(out, in_, seed=out + in_)
    X = synth.activations(P, in_, P)
    with knobs(monkeypatch, FAK_HIP_GEMV_GLOBALX=1):
        Y = q8_0_matmul(raw, out, in_, X, P)
    assert rel_err_rows(Y, exact(raw, out, in_, X)) <= 1e-5


@pytest.mark.parametrize("out,in_,P", [(1536, 576, 1), (3584, 3584, 1), (300, 20000, 1), (2048, 2048, 8), (512, 1056, 16)])
def test_gemv_error(hip, out, in_, P):
    """The GEMV's operands are the codes themselves and 22 bits of the activations: 2-norm error against 64
    bits a few 2^-24 (with 1152 + code, less 1152 times the block's sum, it was 1.5e-6 to 2e-6)."""
    print(f"[case] q8_0 gemv error out={out} in={in_} P={P}", flush=True)
    raw = synth.q8_0_weights(out, in_, seed=out + in_)
    X = synth.activations(P, in_, P)
    ref = exact(raw, out, in_, X)
    assert np.linalg.norm(q8_0_matmul(raw, out, in_, X, P) - ref) <= 4e-7 * np.linalg.norm(ref)
