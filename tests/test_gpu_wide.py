"""The wide MFMA GEMM (gemv builtin with ws=1: batches above 16 rows where it
is picked, prompt chunks above 64) against float64 dot products of the stored
operands: tile edges and remainders of every dimension, every weight / x type,
row-major and tiled weights, split and unsplit K on one shared workspace, every
epilogue by its vector and its scalar form."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

DT_FP8, DT_F16, DT_BF16, DT_F32 = 9, 11, 12, 13
WS = 64 << 20


def say(*a):
    print(*a, flush=True)


def up(hip, a):
    return hip.Buffer.from_numpy(np.ascontiguousarray(a))


def case(rng, wdt, xdt, M, N, K):
    """stored x, W and scales, the float64 product and the rows' absolute sums"""
    x = O.encode(rng.standard_normal((M, K)).astype(np.float32), xdt)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float32)
    scale = None
    if wdt == DT_FP8:
        scale = (np.abs(w).max(1) / 448.0).astype(np.float32)
        ws = O.encode(w / scale[:, None], DT_FP8)
        wf = O.decode(ws, DT_FP8).astype(np.float64) * scale[:, None]
    else:
        ws = O.encode(w, wdt)
        wf = O.decode(ws, wdt).astype(np.float64)
    xf = O.decode(x, xdt).astype(np.float64)
    return x, ws, scale, xf, wf


def rnd(v, dt):
    return O.decode(O.encode(np.asarray(v, np.float32), dt), dt).astype(np.float64)


def near(got, want, floor, dt):
    """within one storage rounding of dt and 1e-5 of the row's absolute sum"""
    ulp = {DT_F32: 0.0, DT_BF16: 2.0 ** -7, DT_F16: 2.0 ** -10}[dt]
    return np.all(np.abs(got - want) <= ulp * np.abs(want) + 2e-5 * floor + 1e-6)


# (M, N, K): one and two row tiles at <= 32 and <= 64 rows, past 64 rows with a
# ragged last tile; N off the 4-row lanes, the 16-row tile, the 64-row block;
# K of one step, of an odd step count, and long enough for several splits
SHAPES = [(17, 100, 6144), (32, 97, 6208), (33, 64, 6144), (64, 10241, 64), (65, 97, 64), (66, 130, 192),
          (129, 64, 1600), (150, 260, 1088), (299, 192, 256)]


@pytest.mark.parametrize("wx", [(DT_FP8, DT_BF16), (DT_FP8, DT_F16), (DT_BF16, DT_BF16), (DT_F16, DT_F16)])
@pytest.mark.parametrize("shape", SHAPES)
def test_wide_gemm_store(hip, wx, shape):
    (wdt, xdt), (M, N, K) = wx, shape
    say(f"case: wide gemm wdt={wdt} xdt={xdt} M={M} N={N} K={K}")
    rng = np.random.default_rng(M * 31 + N + K)
    x, w, scale, xf, wf = case(rng, wdt, xdt, M, N, K)
    ref, floor = xf @ wf.T, np.abs(xf) @ np.abs(wf).T
    wb, xb, sb = up(hip, w), up(hip, x), [up(hip, scale)] if scale is not None else []
    tb = hip.Buffer((N + 15) // 16 * 16 * K * (1 if wdt == DT_FP8 else 2))
    hip.builtin("tile_w", [tb, wb], n=N, k=K, wt=wdt)
    ws = hip.Buffer(WS)
    for tiled in (0, 1):
        first = None
        # the picked tile and splits, then every tile count unsplit and in 3 splits, on one workspace
        for kw in ({}, {}, *[dict(r=r, blocks=s) for r in (1, 2, 4) for s in (1, 3)]):
            y = hip.Buffer(M * N * 4)
            hip.builtin("gemv", [y, xb, tb if tiled else wb, *sb, ws], m=M, n=N, k=K, wt=wdt, xt=xdt,
                        yt=DT_F32, ws=1, tiled=tiled, **kw)
            got = y.read(np.float32).reshape(M, N)
            y.free()
            assert np.all(np.abs(got - ref) <= 1e-5 * floor + 1e-30), (tiled, kw)
            if not kw:   # and the same bits from one run to the next
                assert first is None or np.array_equal(first.view(np.uint32), got.view(np.uint32))
                first = got
    for b in (wb, xb, tb, ws, *sb):
        b.free()


@pytest.mark.parametrize("wdt", [DT_FP8, DT_BF16])
@pytest.mark.parametrize("shape", [(20, 96, 6144), (64, 97, 6208), (70, 130, 320)])
def test_wide_gemm_fused_rmsnorm(hip, wdt, shape):
    """rnd(x g) is multiplied and the row sums scaled by 1/rms: within two
    half-ulps (2^-8 each) per element of the exact normed product."""
    M, N, K = shape
    say(f"case: wide gemm fused norm wdt={wdt} M={M} N={N} K={K}")
    rng = np.random.default_rng(77 + M)
    x, w, scale, xf, wf = case(rng, wdt, DT_BF16, M, N, K)
    g = (1 + 0.2 * rng.standard_normal(K)).astype(np.float32)
    xn = xf / np.sqrt((xf * xf).mean(1, keepdims=True) + 1e-5) * g
    ref, floor = xn @ wf.T, np.abs(xn) @ np.abs(wf).T
    ws = hip.Buffer(WS)
    sb = [up(hip, scale)] if scale is not None else []
    for kw in ({}, dict(r=2, blocks=3), dict(r=1, blocks=1)):
        y = hip.Buffer(M * N * 4)
        hip.builtin("gemv", [y, up(hip, x), up(hip, w), *sb, up(hip, g), ws], m=M, n=N, k=K, wt=wdt,
                    xt=DT_BF16, yt=DT_F32, norm=1, eps=1e-5, ws=1, **kw)
        got = y.read(np.float32).reshape(M, N)
        assert np.all(np.abs(got - ref) <= (1e-5 + 2.0 ** -7) * floor + 1e-6), kw


@pytest.mark.parametrize("dt", [DT_BF16, DT_F16])
@pytest.mark.parametrize("M,N,K,kw", [(70, 256, 320, {}), (70, 256, 512, dict(r=1, blocks=2)),
                                      (70, 250, 320, {}), (21, 192, 6144, {})])
def test_wide_gemm_epilogues(hip, dt, M, N, K, kw):
    """Residual in place, SwiGLU and GELU + bias; N = 250 takes the scalar form
    (rows not a multiple of four)."""
    say(f"case: wide gemm epilogues dt={dt} M={M} N={N} K={K} {kw}")
    rng = np.random.default_rng(M + N + dt)
    x, w, _, xf, wf = case(rng, dt, dt, M, N, K)
    ref, floor = xf @ wf.T, np.abs(xf) @ np.abs(wf).T
    xb, wb, ws = up(hip, x), up(hip, w), hip.Buffer(WS)
    base = dict(m=M, n=N, k=K, wt=dt, xt=dt, yt=dt, ws=1, **kw)
    res = O.encode(rng.standard_normal((M, N)).astype(np.float32), dt)
    y = up(hip, res)
    hip.builtin("gemv", [y, xb, wb, y, ws], epi=1, **base)
    rf = O.decode(res, dt)
    got = O.decode(y.read(np.uint16), dt).reshape(M, N)
    assert near(got, rnd(rf + rnd(ref, dt), dt), floor + np.abs(rf), dt)
    y = hip.Buffer(M * (N // 2) * 2)
    hip.builtin("gemv", [y, xb, wb, ws], epi=2, **base)
    gt, u = rnd(ref[:, 0::2], dt), rnd(ref[:, 1::2], dt)
    got = O.decode(y.read(np.uint16), dt).reshape(M, N // 2)
    assert near(got, gt / (1 + np.exp(-gt)) * u, (floor[:, 0::2] + floor[:, 1::2]) * (1 + np.abs(u)), dt)
    b = O.encode((rng.standard_normal(N) * 0.1).astype(np.float32), dt)
    y = hip.Buffer(M * N * 2)
    hip.builtin("gemv", [y, xb, wb, up(hip, b), ws], epi=3, bias=1, **base)
    v = rnd(ref + O.decode(b, dt), dt)
    got = O.decode(y.read(np.uint16), dt).reshape(M, N)
    want = 0.5 * v * (1 + np.tanh(0.7978845608 * (v + 0.044715 * v ** 3)))
    ulp = 2.0 ** -7 if dt == DT_BF16 else 2.0 ** -10
    # a rounding of v that falls the other way moves the GELU by up to 1.13 of it
    assert np.all(np.abs(got - want) <= 1.2 * ulp * np.abs(v) + ulp * np.abs(want) + 2e-5 * floor + 1e-4)


@pytest.mark.parametrize("rope", [0, 1])
@pytest.mark.parametrize("B,T,kw", [(70, 0, {}), (2, 40, {}), (1, 77, dict(r=1, blocks=2)), (5, 15, {})])
def test_wide_gemm_qkv_append(hip, rope, B, T, kw):
    """q, and k / v into the caches: one position of M sequences (T = 0), or T
    positions of each of B (seq=T) with the last ones past the cache's end."""
    H, Hkv, hd, ms, K, dt = 4, 2, 64, 48, 256, DT_BF16
    M, step, pos = (B * T, T, 9) if T else (B, 1, 9)
    N = (H + 2 * Hkv) * hd
    say(f"case: wide gemm qkv rope={rope} B={B} T={T} {kw}")
    rng = np.random.default_rng(B * 100 + T)
    x, w, scale, xf, wf = case(rng, DT_FP8, dt, M, N, K)
    ref, floor = rnd(xf @ wf.T, dt), np.abs(xf) @ np.abs(wf).T
    f = 1.0 / (10000.0 ** (np.arange(hd // 2) * 2.0 / hd))
    ang = np.arange(ms)[:, None] * f[None, :]
    cs, sn = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
    q = hip.Buffer(M * H * hd * 2)
    kc, vc = (hip.Buffer(B * Hkv * ms * hd * 2) for _ in range(2))
    tabs = [up(hip, cs), up(hip, sn)] if rope else []
    hip.builtin("gemv", [q, up(hip, x), up(hip, w), up(hip, scale), *tabs, up(hip, np.array([pos + 1], np.int32)),
                         kc, vc, hip.Buffer(WS)], m=M, n=N, k=K, wt=DT_FP8, xt=dt, yt=dt, epi=4 if rope else 5,
                h=H, hkv=Hkv, hd=hd, maxseq=ms, ws=1, **(dict(seq=T) if T else {}), **kw)
    p = pos + np.arange(M) % step
    v = ref.reshape(M, H + 2 * Hkv, hd).copy()
    if rope:
        c, s = cs[np.minimum(p, ms - 1)][:, None], sn[np.minimum(p, ms - 1)][:, None]
        e, o = v[:, :H + Hkv, 0::2].copy(), v[:, :H + Hkv, 1::2].copy()
        v[:, :H + Hkv, 0::2], v[:, :H + Hkv, 1::2] = e * c - o * s, o * c + e * s
    fl = np.maximum(floor.reshape(M, H + 2 * Hkv, hd), np.abs(v))
    fl = fl.reshape(M, -1, hd // 2, 2).max(-1, keepdims=True).repeat(2, -1).reshape(fl.shape)
    ok = p < ms   # rows past the cache's end write nothing
    got = O.decode(q.read(np.uint16), dt).reshape(M, H, hd)
    assert np.all(np.abs(got - v[:, :H])[ok] <= (2.0 ** -7 * np.abs(v[:, :H]) + 2.0 ** -8 * fl[:, :H])[ok])
    for buf, h0 in ((kc, H), (vc, H + Hkv)):
        got = O.decode(buf.read(np.uint16), dt).reshape(B, Hkv, ms, hd)
        want, bar = np.zeros((B, Hkv, ms, hd)), np.zeros((B, Hkv, ms, hd))
        for m in range(M):
            if ok[m]:
                want[m // step, :, p[m]] = v[m, h0:h0 + Hkv]
                bar[m // step, :, p[m]] = (2.0 ** -7 * np.abs(v) + 2.0 ** -8 * fl)[m, h0:h0 + Hkv]
        assert np.all(np.abs(got - want) <= bar)


@pytest.mark.parametrize("rope", [0, 1])
@pytest.mark.parametrize("M,ms,K", [(20, 40, 6144), (64, 40, 6144), (40, 64, 8192)])
def test_wide_gemm_spec_append(hip, rope, M, ms, K):
    """spec=1: the M rows are consecutive positions of one sequence, in the
    wide GEMM as in k_gemm (the same call without ws), up to the order of the
    sums; rows past the cache's end write nothing, and nothing is written
    beside the one sequence's caches (views amid a larger buffer)."""
    H, Hkv, hd, dt, pos = 4, 2, 64, DT_BF16, 9
    N = (H + 2 * Hkv) * hd
    say(f"case: wide gemm spec rope={rope} M={M} max_seq={ms} K={K}")
    rng = np.random.default_rng(M + K)
    x, w, scale, xf, wf = case(rng, DT_FP8, dt, M, N, K)
    floor = (np.abs(xf) @ np.abs(wf).T).max()
    ang = np.arange(ms)[:, None] * (1.0 / 10000.0 ** (np.arange(hd // 2) * 2.0 / hd))[None, :]
    tabs = [up(hip, np.cos(ang).astype(np.float32)), up(hip, np.sin(ang).astype(np.float32))] if rope else []
    one = Hkv * ms * hd * 2                                   # bytes of one sequence's cache
    outs = []
    for ws in (0, 1):
        q, big = hip.Buffer(M * H * hd * 2), hip.Buffer(4 * M * one)
        kc, vc = (hip.lib().thvm_hip_buf_view(big.id, o * one, one) for o in (M, 2 * M))
        hip.builtin("gemv", [q, up(hip, x), up(hip, w), up(hip, scale), *tabs, up(hip, np.array([pos + 1], np.int32)),
                             kc, vc, *([hip.Buffer(WS)] if ws else [])], m=M, n=N, k=K, wt=DT_FP8, xt=dt, yt=dt,
                    epi=4 if rope else 5, h=H, hkv=Hkv, hd=hd, maxseq=ms, spec=1, **(dict(ws=1) if ws else {}))
        raw = big.read(np.uint16).reshape(4 * M, one // 2)
        rest = np.delete(raw, [M, 2 * M], 0)
        assert not rest.any(), ws
        outs.append([O.decode(a, dt).astype(np.float64) for a in (q.read(np.uint16), raw[M], raw[2 * M])])
    live = min(M, ms - pos)
    for a, b, rows in zip(outs[0], outs[1], (None, ms, ms)):
        if rows:                                              # positions pos .. pos + live - 1 of each head
            a, b = a.reshape(Hkv, ms, hd), b.reshape(Hkv, ms, hd)
            assert b[:, pos:pos + live].any(-1).all() and not b[:, :pos].any() and not b[:, pos + live:].any()
        # a sum that rounds the other way moves a value by an ulp (2^-7 of it at most);
        # the rotation mixes the two of its pair, and rounds once more
        pair = np.hypot(a[..., 0::2], a[..., 1::2]).repeat(2, -1)
        assert np.all(np.abs(a - b) <= 2.5 * 2.0 ** -7 * pair + 2e-5 * floor)


def test_wide_gemm_refusals(hip):
    say("case: wide gemm refusals")
    b = hip.Buffer(1 << 22)
    kw = dict(n=256, k=1024, wt=DT_BF16, xt=DT_BF16, yt=DT_BF16)
    with pytest.raises(hip.ThvmHipError, match="out of range"):
        hip.builtin("gemv", [b, b, b], m=65, **kw)
    with pytest.raises(hip.ThvmHipError, match="needs"):      # the splits' workspace too small
        hip.builtin("gemv", [b, b, b, hip.Buffer(64)], m=65, ws=1, blocks=2, **kw)
    with pytest.raises(hip.ThvmHipError, match="ws=1 takes"):  # operands the MFMA path does not take
        hip.builtin("gemv", [b, b, b, b], m=65, n=256, k=256, wt=DT_F32, xt=DT_F32, yt=DT_F32, ws=1)
    with pytest.raises(hip.ThvmHipError, match="rows a sequence"):
        hip.builtin("gemv", [b, b, b, b, b, b, b], m=70, n=256, k=256, wt=DT_BF16, xt=DT_BF16, yt=DT_BF16,
                    epi=5, h=2, hkv=1, hd=64, maxseq=8, ws=1, seq=33)


@pytest.mark.parametrize("m,extra", [(2, dict(path=1)), (4, dict(path=1)), (6, dict(pre=1, norm=2)), (16, dict(pre=1, norm=2)),
                                     (4, dict(spec=1)), (70, dict(spec=1)), (6, None)])
def test_wide_gemm_seq_refusals(hip, m, extra):
    """seq= on a QKV call that another kernel would run (one position a row),
    or beside spec, is refused before anything is launched: the caches hold
    m / seq sequences only."""
    say(f"case: wide gemm seq refusal m={m} {extra}")
    H, Hkv, hd, ms, K, dt = 2, 1, 64, 16, 256, DT_BF16
    N = (H + 2 * Hkv) * hd
    q, x, w = hip.Buffer(m * H * hd * 2), hip.Buffer(m * K * 2), hip.Buffer(N * K * 2)
    norm = [hip.Buffer(K * 4), hip.Buffer(K * 4)] if extra and extra.get("norm") else []
    kc, vc = (hip.Buffer(m // 2 * Hkv * ms * hd * 2) for _ in range(2))
    tail = [hip.Buffer(4), kc, vc] + ([hip.Buffer(WS)] if extra is not None else [])
    with pytest.raises(hip.ThvmHipError, match="rows a sequence"):
        hip.builtin("gemv", [q, x, w, *norm, *tail], m=m, n=N, k=K, wt=dt, xt=dt, yt=dt, epi=5, h=H, hkv=Hkv, hd=hd,
                    maxseq=ms, seq=2, **(dict(ws=1, **extra) if extra is not None else {}))


def test_wide_gemm_empty_and_huge_shapes_refused(hip):
    """No columns or rows, and counts whose tile arithmetic would leave 32 bits,
    are errors (the workspace is sized before the launcher's range checks)."""
    say("case: wide gemm empty and huge shapes")
    b = hip.Buffer(1 << 16)
    for m, n, k in ((65, 0, 64), (0, 64, 64), (65, 64, 0), (2 ** 32 - 1, 64, 64), (65, 2 ** 32 - 1, 64), (2 ** 32 - 1, 2 ** 32 - 1, 64)):
        with pytest.raises(hip.ThvmHipError):
            hip.builtin("gemv", [b, b, b, b], m=m, n=n, k=k, wt=DT_BF16, xt=DT_BF16, yt=DT_BF16, ws=1)


@pytest.mark.parametrize("wx", [(DT_FP8, DT_BF16), (DT_BF16, DT_BF16), (DT_F16, DT_F16)])
@pytest.mark.parametrize("K", [1024, 1600, 4096, 14336])
def test_wide_gemm_sums_as_exact_as_k_gemm(hip, wx, K):
    """The f32 sums' error against float64 (2-norm over the result's) is no
    larger than that of k_gemm, whose place the wide GEMM takes above 16 rows
    and whose waves each sum an eighth of K: at every tile, K unsplit, where a
    wave's slice is longest, and split."""
    (wdt, xdt), M, N = wx, 60, 256
    say(f"case: wide gemm sums wdt={wdt} K={K}")
    x, w, scale, xf, wf = case(np.random.default_rng(N + K), wdt, xdt, M, N, K)
    ref = xf @ wf.T
    args, ws = [up(hip, x), up(hip, w), *([up(hip, scale)] if scale is not None else [])], hip.Buffer(WS)

    def err(extra, **kw):
        y = hip.Buffer(M * N * 4)
        hip.builtin("gemv", [y, *args, *extra], m=M, n=N, k=K, wt=wdt, xt=xdt, yt=DT_F32, **kw)
        return np.linalg.norm(y.read(np.float32).reshape(M, N) - ref) / np.linalg.norm(ref)

    # (seq, which the plain store does not read, takes the wide GEMM at any shape)
    bar = err([])
    for r in (1, 2, 4):
        for blocks in (1, 2):
            e = err([ws], ws=1, seq=1, r=r, blocks=blocks)
            assert e <= bar, (r, blocks, e, bar)
