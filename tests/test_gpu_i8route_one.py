"""The int8 route's one-token kernel (q4k_i8route1_kernel) at the edges of its shapes, bit for bit
against the oracle: rows around a 16-row tile, fewer records than waves, a wave split of every size,
several tiles per workgroup, rows longer than the activations a workgroup holds in registers, the
longest row whose terms fit in LDS and one past it (the general kernel), the last tile count it takes on
long rows and the next, zero, subnormal and
non-finite activation blocks."""
import numpy as np
import pytest

from fak_amd import synth
from tests.gpu_util import q4k_matmul_int8
from tests.test_gpu_i8route import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out,in_", [(1, 256), (15, 512), (17, 768), (100, 3584), (520, 4352),
                                     (8200, 256), (16500, 1280), (48, 18944), (33, 30976),
                                     (33, 31232), (16368, 4352), (16384, 4352)])
def test_shapes(hip, oracle_mod, out, in_):
    print(f"[case] int8 one token out={out} in={in_}", flush=True)
    raw = synth.q4k_weights(out, in_, out + in_)
    x = synth.activations(1, in_, in_)
    x[0, 32:64] = 0.0
    x[0, 100] *= 1e30
    sel = np.arange(out) if out <= 1000 else np.r_[0:70, out - 300:out]
    rb = (in_ // 256) * 144
    sub = np.concatenate([raw[o * rb:(o + 1) * rb] for o in sel])
    same_bits(q4k_matmul_int8(raw, out, in_, x, 1)[0][sel],
              oracle_mod.q4k_matrows_int8(sub, len(sel), in_, x[0]))


def test_non_finite(hip, oracle_mod):
    out, in_ = 40, 1024
    print("[case] int8 one token non-finite", flush=True)
    raw = synth.q4k_weights(out, in_, 9)
    for t in range(3):
        x = synth.activations(1, in_, 9 + t)
        if t == 0:
            x[0, 5] = np.nan
        elif t == 1:
            x[0, 300] = -np.inf
        else:
            x[0, 672:704] = 0.0
            x[0, 700] = np.float32(1e-40)
        same_bits(q4k_matmul_int8(raw, out, in_, x, 1)[0],
                  oracle_mod.q4k_matrows_int8(raw, out, in_, x[0]))
