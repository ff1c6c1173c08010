"""The expert-major v_dot4 phases (k_moe_ax, k_moe_bx) at every segment width
and around the eight pairs they stage at a time: segments of 8 to 64 lanes,
whose lanes keep a pair's sums each.  Bars: those of the stage-wise parity
(_check_moe)."""

import numpy as np
import pytest

import oracle as O
from tests.test_gpu_parity import _check_moe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,I", [(256, 256), (512, 768), (1024, 1280), (2048, 768), (4096, 256)])
@pytest.mark.parametrize("k", [1, 8, 9, 16])
def test_expert_major_segments(tg, orc, D, I, k):
    rng = np.random.default_rng(D + I + k)
    n = 3
    rw = np.zeros((n, k), np.float32)
    rw[0, :] = 0.5
    rw[1, k // 2:] = 0.3
    rw[2, 0] = 0.2
    x = rng.standard_normal((k, D)).astype(np.float32)
    base = rng.standard_normal((k, D)).astype(np.float32)
    print(f"expert-major segments: D={D} I={I} k={k}", flush=True)
    _check_moe(tg, orc, n, k, D, I, O.FMT_Q4K, [O.FMT_Q6K] * n, O.ACT_SILU, True, rw, x, base)
