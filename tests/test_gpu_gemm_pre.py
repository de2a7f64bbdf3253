"""The MFMA GEMM with a norm ahead of the product (pre=1) on the GPU: against
the norm kernel and the GEMM in two launches, and what it refuses.
"""
import numpy as np
import pytest

import _oracle as O
from test_gpu_dsv2 import DT_BF16, DT_F16, DT_F32, DT_FP8, fp8_rows, say, up
from test_gpu_kernels import NP_STORE, rand_store

pytestmark = pytest.mark.gpu

# M, N, K, weight type, x type, norm (1 RMSNorm, 2 LayerNorm), tiled weights:
# row pairs of a wave, one to 32 K steps (fewer than the waves, whole and
# ragged slices), 1 and 2 tiles a block (one grid of more than a round), a ragged
# last tile
CASES = [(5, 48, 64, DT_F16, DT_F16, 2, 0), (8, 4800, 1600, DT_F16, DT_F16, 2, 1), (8, 6400, 1600, DT_F16, DT_F16, 2, 0),
         (9, 33, 576, DT_BF16, DT_BF16, 2, 1), (16, 12288, 256, DT_BF16, DT_BF16, 2, 0), (16, 200, 2048, DT_F16, DT_F16, 2, 1),
         (7, 4112, 1088, DT_F16, DT_F16, 1, 0), (13, 3000, 2048, DT_FP8, DT_F16, 1, 1), (6, 9000, 640, DT_FP8, DT_BF16, 2, 0)]


@pytest.mark.parametrize("M,N,K,wdt,xdt,norm,tiled", CASES)
def test_norm_ahead_of_gemm(hip, M, N, K, wdt, xdt, norm, tiled):
    say(f"case: gemm pre M={M} N={N} K={K} wt={wdt} xt={xdt} norm={norm} tiled={tiled}")
    rng = np.random.default_rng(M + N + K + norm)
    xs, xf = rand_store(rng, (M, K), xdt)
    if norm == 2:                               # a mean that dwarfs the spread, rows of other scales
        xf = xf * np.linspace(0.1, 4, M)[:, None].astype(np.float32) + 8.0
        xs = O.encode(xf.astype(np.float32), xdt)
        xf = O.decode(xs, xdt)
    scale = []
    if wdt == DT_FP8:
        ws, sc, wf = fp8_rows(rng, N, K)
        scale = [up(hip, sc)]
    else:
        ws, wf = rand_store(rng, (N, K), wdt, 0.02)
    g = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    b = (0.1 * rng.standard_normal(K)).astype(np.float32)
    es = 1 if wdt == DT_FP8 else 2
    w = up(hip, ws)
    if tiled:
        wt = hip.Buffer((N + 15) // 16 * 16 * K * es)
        hip.builtin("tile_w", [wt, w], n=N, k=K, wt=wdt)
        w = wt
    x, gb = up(hip, xs), [up(hip, g)] + ([up(hip, b)] if norm == 2 else [])
    y, xn, y2 = hip.Buffer(M * N * 4), hip.Buffer(M * K * 2), hip.Buffer(M * N * 4)
    geo = dict(m=M, n=N, k=K, wt=wdt, xt=xdt, yt=DT_F32, epi=0, tiled=tiled)
    hip.builtin("gemv", [y, x, w] + scale + gb, norm=norm, eps=1e-5, pre=1, **geo)
    hip.builtin("norm", [xn, x] + gb, m=M, k=K, xt=xdt, yt=xdt, eps=1e-5, ln=norm == 2, bias=norm == 2)
    hip.builtin("gemv", [y2, xn, w] + scale, **geo)
    got, two = y.read(np.float32).reshape(M, N), y2.read(np.float32).reshape(M, N)
    # the two differ where the statistics' sum orders put a normalised value
    # on the other side of a rounding: at most one rounding of x a product
    nx = O.decode(xn.read(NP_STORE[xdt]), xdt).reshape(M, K).astype(np.float64)
    ulp = 2.0 ** (-10 if xdt == DT_F16 else -7)
    floor = np.abs(nx) @ np.abs(wf.astype(np.float64)).T
    assert np.all(np.abs(got - two) <= (ulp + K * 2.0 ** -23) * floor)
    # and against the whole in float64: half a rounding of x a product, the
    # statistics' error (K roundings, doubled by the square root's argument)
    x64 = xf.astype(np.float64)
    mean = x64.mean(1, keepdims=True) if norm == 2 else 0.0
    n64 = (x64 - mean) / np.sqrt(((x64 - mean) ** 2).mean(1, keepdims=True) + 1e-5) * g + (b if norm == 2 else 0.0)
    want = n64 @ wf.astype(np.float64).T
    assert np.all(np.abs(got - want) <= (ulp / 2 + K * 2.0 ** -22) * (np.abs(n64) @ np.abs(wf.astype(np.float64)).T + floor))
    err, err2 = np.sqrt(((got - want) ** 2).mean()), np.sqrt(((two - want) ** 2).mean())
    say(f"  rms error {err:.3e}, in two launches {err2:.3e}")
    assert err <= 1.02 * err2


def test_norm_ahead_refusals(hip):
    big = [hip.Buffer(1 << 20) for _ in range(5)]
    ok = dict(m=8, n=64, k=256, wt=DT_F16, xt=DT_F16, yt=DT_F32, epi=0, norm=2, eps=1e-5, pre=1)
    hip.builtin("gemv", big, **ok)
    for kw in (dict(m=17), dict(k=4096, m=8, n=32), dict(norm=0), dict(path=1), dict(m=4), dict(r=4), dict(k=232),
               dict(xt=DT_F32, wt=DT_F32)):
        with pytest.raises(hip.ThvmHipError, match="pre=1"):
            hip.builtin("gemv", big, **dict(ok, **kw))
