"""The GEMV at two to four x rows stages all rows at once, in an instance per
fused norm (a LayerNorm's ahead of the weights): every row must still be the
one-row launch's bits, with no norm and each fused norm, over row lengths from
one vector per thread to the most a fused norm takes and weight rows of every
chunk remainder."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

DT_FP8, DT_F16, DT_BF16, DT_F32 = 9, 11, 12, 13


def up(hip, a):
    return hip.Buffer.from_numpy(np.ascontiguousarray(a))


@pytest.mark.parametrize("wdt,xdt", [(DT_FP8, DT_BF16), (DT_BF16, DT_BF16), (DT_F16, DT_F16), (DT_F32, DT_F32),
                                     (DT_FP8, DT_F32), (DT_FP8, DT_F16)])
@pytest.mark.parametrize("N,K", [(37, 64), (2050, 1600), (130, 4096), (64, 8192), (70, 10224)])
@pytest.mark.parametrize("norm", [0, 1, 2])
def test_gemv_rows_equal_one_row(hip, wdt, xdt, N, K, norm):
    if norm and K > 8192:
        K = 8176     # the longest ragged row a fused norm takes
    print(f"case: gemv rows wdt={wdt} xdt={xdt} N={N} K={K} norm={norm}", flush=True)
    rng = np.random.default_rng(N + K + norm)
    x = rng.standard_normal((4, K)).astype(np.float32) * 2 + 0.3
    x = x if xdt == DT_F32 else O.encode(x, xdt)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float32)
    sc = (np.abs(w).max(1) / 448).astype(np.float32)
    w = w if wdt == DT_F32 else O.encode(w / sc[:, None], wdt) if wdt == DT_FP8 else O.encode(w, wdt)
    args = [up(hip, w)] + ([up(hip, sc)] if wdt == DT_FP8 else [])
    if norm:
        args.append(up(hip, (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)))
    if norm == 2:
        args.append(up(hip, rng.standard_normal(K).astype(np.float32)))
    kw = dict(n=N, k=K, wt=wdt, xt=xdt, yt=DT_F32, norm=norm, eps=1e-5)
    one = []
    for r in range(4):
        y = hip.Buffer(N * 4)
        # (8 waves: a LayerNorm's sum is in the order of its block, which one row may take smaller)
        hip.builtin("gemv", [y, up(hip, x[r]), *args], m=1, waves=8, **kw)
        one.append(y.read(np.uint32))
    for M in (2, 3, 4):
        y = hip.Buffer(M * N * 4)
        hip.builtin("gemv", [y, up(hip, x[:M]), *args], m=M, **kw)
        got = y.read(np.uint32).reshape(M, N)
        for r in range(M):
            assert np.array_equal(got[r], one[r]), (M, r)


@pytest.mark.parametrize("wdt,xdt", [(DT_FP8, DT_BF16), (DT_F16, DT_F16)])
@pytest.mark.parametrize("M,K", [(4, 20416), (4, 20480), (4, 20544), (2, 40960), (1, 81920)])
def test_gemv_rows_at_the_lds_limit(hip, wdt, xdt, M, K):
    """Rows that just do not fit the GEMV's LDS (160 KiB with its reserve: M K 2
    = 163840 bytes exactly, and a step to each side) take the MFMA GEMM."""
    N = 48
    print(f"case: gemv rows at the LDS limit wdt={wdt} M={M} K={K}", flush=True)
    rng = np.random.default_rng(M + K)
    x = O.encode(rng.standard_normal((M, K)).astype(np.float32), xdt)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float32)
    sc = (np.abs(w).max(1) / 448).astype(np.float32) if wdt == DT_FP8 else None
    ws = O.encode(w / sc[:, None] if sc is not None else w, wdt)
    wf = O.decode(ws, wdt).astype(np.float64) * (sc[:, None] if sc is not None else 1.0)
    xf = O.decode(x, xdt).astype(np.float64)
    y = hip.Buffer(M * N * 4)
    hip.builtin("gemv", [y, up(hip, x), up(hip, ws), *([up(hip, sc)] if sc is not None else [])], m=M, n=N, k=K, wt=wdt,
                xt=xdt, yt=DT_F32)
    got = y.read(np.float32).reshape(M, N)
    # f32 sums of K products in any order: well inside 2^-24 sqrt(K) of the absolute sum
    assert np.all(np.abs(got - xf @ wf.T) <= 1e-5 * (np.abs(xf) @ np.abs(wf).T))


@pytest.mark.parametrize("wdt,xdt,K", [(DT_FP8, DT_BF16, 1024), (DT_F16, DT_F16, 768), (DT_F32, DT_F32, 192), (DT_FP8, DT_BF16, 12288)])
@pytest.mark.parametrize("N", [2048, 2050, 4096, 4098, 8190, 8192, 16382, 16384])
def test_gemv_rows_per_wave_keep_the_bits(hip, wdt, xdt, K, N):
    """One or two weight rows a wave, as the shape picks it on each side of its
    lines, are the same sums."""
    print(f"case: gemv rows per wave wdt={wdt} N={N} K={K}", flush=True)
    rng = np.random.default_rng(N + K)
    x = rng.standard_normal((4, K)).astype(np.float32)
    x = x if xdt == DT_F32 else O.encode(x, xdt)
    wn = {DT_FP8: 1, DT_F16: 2, DT_F32: 4}[wdt]
    w = O.encode((rng.standard_normal((256, K)) * 0.05).astype(np.float32), wdt) if wdt != DT_F32 else \
        (rng.standard_normal((256, K)) * 0.05).astype(np.float32)
    w = np.tile(w, (N // 256 + 1, 1))[:N]
    assert w.itemsize == wn
    args = [up(hip, w)] + ([up(hip, rng.random(N).astype(np.float32))] if wdt == DT_FP8 else [])
    g, b = (up(hip, rng.standard_normal(K).astype(np.float32)) for _ in range(2))
    for norm in (0, 1, 2) if K <= 8192 else (0,):
        for M in (1, 2, 3, 4):
            out = []
            for kw in ({}, dict(r=1)):
                y = hip.Buffer(M * N * 4)
                hip.builtin("gemv", [y, up(hip, x[:M]), *args, *[g, b][:norm]], m=M, n=N, k=K, wt=wdt, xt=xdt, yt=DT_F32,
                            norm=norm, eps=1e-5, waves=8, **kw)
                out.append(y.read(np.uint32))
                y.free()
            assert np.array_equal(*out), (norm, M)
