"""mla_prep on the GPU at the edges of its two absorption kernels: d_nope from
one 16-value piece to several 128-wide steps, batches around the 16-row MFMA
tile, and the q rows that 16-byte loads cannot read (which take the VALU
form), against the oracle and the products in float64.
"""
import numpy as np
import pytest

import _oracle as O
from test_gpu_dsv2 import DT_BF16, DT_FP8, bf, close_bf16, say, unbf, up, weights

pytestmark = pytest.mark.gpu

# H, dn, dr, kv, B, extra columns of a q row, weight type
CASES = [(16, 128, 64, 512, 1, 0, DT_FP8), (16, 128, 64, 512, 15, 0, DT_FP8), (16, 128, 64, 512, 32, 0, DT_FP8),
         (3, 16, 8, 64, 16, 0, DT_FP8), (5, 32, 16, 128, 17, 8, DT_FP8), (1, 256, 64, 256, 33, 0, DT_FP8),
         (2, 512, 8, 64, 4, 0, DT_FP8), (4, 128, 64, 512, 32, 0, DT_BF16), (3, 16, 8, 64, 18, 0, DT_BF16),
         (2, 256, 32, 128, 5, 16, DT_BF16),
         # the VALU form: d_nope 8, rope widths and row strides off the 16-byte grid
         (4, 8, 8, 64, 9, 0, DT_BF16), (4, 128, 2, 128, 9, 0, DT_FP8), (4, 64, 64, 512, 17, 1, DT_FP8),
         (2, 64, 12, 64, 3, 0, DT_BF16)]


@pytest.mark.parametrize("H,dn,dr,kv,B,extra,wdt", CASES)
def test_mla_prep_edges(hip, H, dn, dr, kv, B, extra, wdt):
    say(f"case: mla_prep H={H} dn={dn} dr={dr} kv={kv} B={B} extra={extra} wdt={wdt}")
    rng = np.random.default_rng(H + dn + dr + kv + B + extra + wdt)
    ldq, ms, pos = H * (dn + dr) + kv + dr + extra, 40, 38
    qkv = bf(rng.standard_normal((B, ldq)))
    wuk, suk, wukf = weights(rng, H * kv, dn, wdt)
    wkvn = (1 + 0.1 * rng.standard_normal(kv)).astype(np.float32)
    ang = rng.uniform(0, 6.3, (ms, dr // 2))
    cs, sn = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
    ckv0, kpe0 = bf(rng.standard_normal((B, ms, kv))), bf(rng.standard_normal((B, ms, dr)))
    ckv, kpe = up(hip, ckv0), up(hip, kpe0)
    qlat, qpe = hip.Buffer(B * H * kv * 4), hip.Buffer(B * H * dr * 2)
    f8 = wdt == DT_FP8
    args = [up(hip, qkv), up(hip, wuk)] + ([up(hip, suk)] if f8 else []) + [
        up(hip, wkvn), up(hip, cs), up(hip, sn), up(hip, np.array([pos + 1], np.int32)), ckv, kpe, qlat, qpe]
    hip.builtin("mla_prep", args, b=B, h=H, dn=dn, dr=dr, kv=kv, dv=64, maxseq=ms, ldq=ldq, wt=wdt,
                eps=1e-6)
    g_qlat = qlat.read(np.float32).reshape(B, H, kv)
    g_qpe = qpe.read(np.uint16).reshape(B, H, dr)
    g_ckv = ckv.read(np.uint16).reshape(B, ms, kv)
    g_kpe = kpe.read(np.uint16).reshape(B, ms, dr)
    keep = np.arange(ms) != pos
    w64 = wukf.astype(np.float64).reshape(H, kv, dn)
    for b in range(B):
        w_qpe, w_qlat = np.empty((H, dr), np.uint16), np.empty((H, kv), np.float32)
        w_crow, w_prow = np.empty(kv, np.uint16), np.empty(dr, np.uint16)
        O.oracle().or_mla_prep(w_qpe.ctypes.data, w_qlat.ctypes.data, w_crow.ctypes.data, w_prow.ctypes.data,
                               np.ascontiguousarray(qkv[b]).ctypes.data, wuk.ctypes.data, wdt,
                               suk.ctypes.data if f8 else None, wkvn.ctypes.data,
                               np.ascontiguousarray(cs[pos]).ctypes.data, np.ascontiguousarray(sn[pos]).ctypes.data,
                               H, dn, dr, kv, 1e-6)
        assert np.all(close_bf16(unbf(g_qpe[b]), unbf(w_qpe)))
        assert np.all(close_bf16(unbf(g_ckv[b, pos]), unbf(w_crow)))
        assert np.all(close_bf16(unbf(g_kpe[b, pos]), unbf(w_prow)))
        qn = unbf(qkv[b, :H * (dn + dr)].reshape(H, dn + dr)[:, :dn]).astype(np.float64)
        want, floor = (w64 @ qn[:, :, None])[..., 0], (np.abs(w64) @ np.abs(qn)[:, :, None])[..., 0]
        # products are exact in f32; dn sums and the scale round at 2^-24 each
        # (weights() gives the scaled rows in f32: one more)
        assert np.all(np.abs(g_qlat[b] - want) <= (dn + 2) * 2.0 ** -24 * floor)
        assert np.array_equal(g_ckv[b, keep], ckv0[b, keep]) and np.array_equal(g_kpe[b, keep], kpe0[b, keep])
