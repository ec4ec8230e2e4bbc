"""The HAL Q8 kernels for 32-code blocks (q8_hal_gemv32_kernel, q8_hal_gemm32_kernel) at the edges
of their tiles, against the oracle's qdot8scalar / qgemm8cell, bit for bit: rows around the
workgroup's 16 or 32, activations around the 4096 values a workgroup holds in registers, chunks of
one to four blocks, every token tile, and the calls that keep the general kernels (codes that are
not 16-byte aligned, an output written over its input)."""
import numpy as np
import pytest

from fak_amd import fakhip
from tests.gpu_util import Dev
from tests.test_gpu_hal_q8 import dev_matmul, edge_rows, rand_hal_weight

pytestmark = pytest.mark.gpu


def assert_bits(y, ref):
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    ok = ~np.isnan(ref)
    np.testing.assert_array_equal(y[ok].view(np.uint32), ref[ok].view(np.uint32))


def hal_case(out, in_, P):
    rng = np.random.default_rng(7 * out + in_ + P)
    codes, scales = rand_hal_weight(rng, out, in_, 32)
    codes[rng.integers(0, codes.size, 8)] = -128
    scales[rng.integers(0, scales.size, 4)] *= -1
    X = rng.standard_normal((P, in_)).astype(np.float32)
    E = edge_rows(in_, 32, rng)
    for t in range(0, P, 2):
        X[t] = E[(t // 2) % len(E)]
    if P > 3:
        X[3, in_ // 2] = np.inf
        X[1, 0] = np.nan
    return codes, scales, X


@pytest.mark.parametrize("out,in_", [(1, 32), (15, 64), (16, 2048), (33, 4064), (17, 4128),
                                     (35, 18944), (40, 51200)])
def test_decode(hip, oracle_mod, out, in_):
    print(f"[case] hal decode out={out} in={in_}", flush=True)
    codes, scales, X = hal_case(out, in_, 6)
    for t in range(6):
        y = dev_matmul(codes, scales, X[t], out, in_, 1, 32)[0]
        assert_bits(y, oracle_mod.hal_q8_matmul(codes, scales, X[t], out, in_, 32))


@pytest.mark.parametrize("out,in_,P", [(1, 32, 2), (17, 96, 3), (50, 160, 4), (31, 128, 5),
                                       (33, 3584, 15), (16, 288, 17), (3233, 64, 33),
                                       (1601, 224, 129)])
def test_batched(hip, oracle_mod, out, in_, P):
    print(f"[case] hal batched out={out} in={in_} P={P}", flush=True)
    codes, scales, X = hal_case(out, in_, P)
    Y = dev_matmul(codes, scales, X, out, in_, P, 32)
    assert_bits(Y, oracle_mod.hal_q8_batched_matmul(codes, scales, X, out, in_, P, 32))


@pytest.mark.parametrize("P", [1, 5])
def test_general_kernels_stay(hip, oracle_mod, P):
    out = in_ = 96
    codes, scales, X = hal_case(out, in_, P)
    ref = (oracle_mod.hal_q8_matmul(codes, scales, X[0], out, in_, 32)[None] if P == 1 else
           oracle_mod.hal_q8_batched_matmul(codes, scales, X, out, in_, P, 32))
    with Dev.from_host(np.concatenate([np.zeros(4, np.int8), codes])) as dc, \
            Dev.from_host(scales) as ds, Dev.from_host(X) as dx, Dev.from_host(codes) as da, \
            Dev(P * out * 4) as dy:
        print(f"[case] hal unaligned codes P={P}", flush=True)
        fakhip.call("fhip_q8_matmul_f32", dc.ptr + 4, ds.ptr, dx.ptr, dy.ptr, out, in_, P, 32)
        assert_bits(dy.to_host(np.float32).reshape(P, out), ref)
        print(f"[case] hal output over input P={P}", flush=True)
        fakhip.call("fhip_q8_matmul_f32", da.ptr, ds.ptr, dx.ptr, dx.ptr, out, in_, P, 32)
        assert_bits(dx.to_host(np.float32).reshape(P, out), ref)
