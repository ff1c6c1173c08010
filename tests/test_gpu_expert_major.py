"""The expert-major v_dot4 phases (k_moe_ax, k_moe_bx) at every segment width
and around the eight pairs they stage at a time: segments of 8 to 64 lanes,
whose lanes keep a pair's sums each.  Bars: those of the stage-wise parity
(_check_moe)."""

import numpy as np
import pytest

import oracle as O
from tests.test_gpu_parity import _check_moe, _experts, close

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


@pytest.mark.parametrize("fmt,down,act", [(O.FMT_Q4K, O.FMT_Q6K, O.ACT_SILU), (O.FMT_MXFP4, O.FMT_MXFP4, O.ACT_GPTOSS)])
@pytest.mark.parametrize("k", [1, 3, 9])
def test_expert_major_null_biases(tg, orc, fmt, down, act, k):
    """Experts without biases beside experts with them: null entries count as
    no bias, in the v_dot4 phases and (MXFP4, nine rows) the MFMA ones."""
    print(f"expert-major null biases: fmt {fmt}, {k} rows", flush=True)
    n, D, I = 4, 512, 256
    rng = np.random.default_rng(fmt + k)
    rw = rng.uniform(0.1, 1.0, (n, k)).astype(np.float32) / n
    x = rng.standard_normal((k, D)).astype(np.float32)
    g, u, d = _experts(n, D, I, fmt, [down] * n, 97)
    b = [[rng.uniform(-0.5, 0.5, w).astype(np.float32) for _ in range(n)] for w in (I, I, D)]
    for t in b[:2]:
        t[0] = t[2] = None
    b[2][1] = b[2][2] = None
    h_ref, h_gpu = np.zeros((n * k, I), np.float32), np.zeros((n * k, I), np.float32)
    args = (g, u, d, fmt, [down] * n, *b, act, rw, x)
    orc.moe_v2(*args, np.zeros((k, D), np.float32), I, hidden_out=h_ref)
    got = tg.moe_forward_rows_v2(*args, np.zeros((k, D), np.float32), I, hidden_out=h_gpu)
    assert tg.last_error() == ""
    for p in range(n * k):
        ok, rel = close(h_gpu[p], h_ref[p], tol=1e-4)
        assert ok, ("hidden", p, rel)
    ok, rel = close(got, orc.moe_v2(*args, np.zeros((k, D), np.float32), I, hidden_in=h_gpu))
    assert ok, rel
