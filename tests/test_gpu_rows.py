"""The GEMV at two to four x rows stages all rows at once and keeps fewer chunks
in flight than at one: every row must still be the one-row launch's bits, with
no norm and each fused norm, over row lengths from one vector per thread to the
most a fused norm takes and weight rows of every chunk remainder."""
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
