"""One-launch forms of the decode step on the GPU at the edges of their
ranges: attention whose blocks take a whole cache row and write the output
themselves, and the greedy argmax that also advances the length.
"""
import numpy as np
import pytest

import _oracle as O
from test_gpu_dsv2 import DT_BF16, DT_F16, DT_F32, say, up
from test_gpu_kernels import NP_STORE, SZ, attn_close, rand_store

pytestmark = pytest.mark.gpu

# H, Hkv, hd, chunks, B, cache type: each side of the lines in (row, kv head)
# pairs (96), chunks (8, 16) and a block's work (768, 1536), the three head groups
ATTN = [(4, 4, 64, 1, 2, DT_F32), (4, 4, 64, 8, 2, DT_F32), (12, 12, 64, 8, 1, DT_F16), (3, 3, 128, 8, 1, DT_BF16),
        (12, 12, 64, 9, 1, DT_F16), (2, 2, 64, 12, 3, DT_BF16), (2, 2, 64, 13, 3, DT_BF16),
        (4, 4, 64, 9, 1, DT_F32), (26, 26, 64, 16, 5, DT_F16), (16, 16, 64, 16, 8, DT_F32), (16, 16, 128, 9, 8, DT_BF16),
        (8, 4, 128, 6, 2, DT_BF16), (8, 4, 128, 7, 2, DT_BF16), (8, 2, 128, 3, 1, DT_BF16), (8, 2, 128, 4, 1, DT_F16),
        (64, 16, 128, 8, 8, DT_BF16), (8, 1, 64, 3, 2, DT_BF16),
        (12, 12, 64, 2, 16, DT_F32), (38, 38, 64, 8, 5, DT_F16), (48, 24, 128, 5, 8, DT_BF16), (64, 16, 64, 3, 12, DT_F16),
        (12, 12, 64, 11, 8, DT_F16), (19, 19, 128, 9, 5, DT_BF16), (3, 3, 64, 10, 1, DT_F16), (3, 3, 64, 11, 1, DT_F16),
        (76, 19, 128, 8, 5, DT_BF16), (64, 16, 128, 8, 6, DT_BF16), (38, 19, 128, 7, 5, DT_F32), (32, 16, 128, 7, 6, DT_F32)]


@pytest.mark.parametrize("H,Hkv,hd,ns,B,cdt", ATTN)
def test_attention_picked_launch(hip, H, Hkv, hd, ns, B, cdt):
    """fused=2 with the chunks per block picked from the shape, and with all
    of them in one block, against the oracle."""
    ms = 64 * ns - 3
    rng = np.random.default_rng(H + hd + ns + B + cdt)
    qs, _ = rand_store(rng, (B, H, hd), cdt)
    ks, _ = rand_store(rng, (B, Hkv, ms, hd), cdt)
    vs, _ = rand_store(rng, (B, Hkv, ms, hd), cdt)
    q, k, v = up(hip, qs), up(hip, ks), up(hip, vs)
    scale = float(np.float32(1.0 / np.sqrt(hd)))
    geo = dict(b=B, h=H, hkv=Hkv, hd=hd, maxseq=ms, chunk=64, nsplit=ns, qt=cdt, ct=cdt, ot=cdt, scale=scale)
    for L in sorted({1, min(64, ms), min(65, ms), ms // 2 + 1, ms}):
        say(f"case: attn H={H} Hkv={Hkv} hd={hd} chunks={ns} B={B} dt={cdt} L={L}")
        ln = up(hip, np.array([L], np.int32))

        def run(**kw):
            out = hip.Buffer(B * H * hd * SZ[cdt])
            part = hip.Buffer(B * H * ns * (hd + 2) * 4 + B * Hkv * 4)
            hip.builtin("attn", [out, q, k, v, ln, part], **geo, **kw)
            return out.read(NP_STORE[cdt])

        got = run(fused=2)
        want = np.empty(B * H * hd, NP_STORE[cdt])
        O.oracle().or_attn_decode(want.ctypes.data, cdt, qs.ctypes.data, cdt, ks.ctypes.data, vs.ctypes.data, cdt, B, H,
                                  Hkv, hd, ms, L, scale)
        assert attn_close(O.decode(got, cdt), O.decode(want, cdt), cdt)
        if H // Hkv <= 4:
            one = run(fused=2, cpb=ns, mf=2)
            assert attn_close(O.decode(one, cdt), O.decode(want, cdt), cdt)


@pytest.mark.parametrize("B,V,nb", [(1, 1, 256), (1, 50257, 256), (4, 63, 8), (17, 1001, 64), (64, 777, 256)])
def test_argmax_advances_length(hip, B, V, nb):
    """bump=1: the ids and history of the two-op form (argmax, then len_bump),
    and the length advanced once whatever the batch."""
    say(f"case: argmax bump B={B} V={V} nb={nb}")
    rng = np.random.default_rng(B + V)
    lg = rng.standard_normal((B, V)).astype(np.float32)
    lg[0, :] = -np.inf                        # all equal: the lowest index
    if B > 1:
        lg[1, [V // 2, V - 1]] = 50.0         # tie
        lg[B - 1, V // 3] = np.inf
    nb, stride = min(nb, V), 5
    for L in (0, stride - 1, stride):         # past the history: no id is kept
        outs = []
        for bump in (0, 1):
            tok, pv, pi = hip.Buffer(B * 4), hip.Buffer(B * nb * 4), hip.Buffer(B * nb * 4)
            hist, ln = up(hip, np.full((B, stride), -7, np.int32)), up(hip, np.array([L], np.int32))
            hip.builtin("argmax", [tok, up(hip, lg), pv, pi, hist, ln], b=B, v=V, nb=nb, hist=1, hstride=stride, bump=bump)
            if not bump:
                hip.builtin("len_bump", [ln], delta=1)
            outs.append((tok.read(np.int32), hist.read(np.int32).reshape(B, stride), ln.read(np.int32)[0]))
        (t0, h0, l0), (t1, h1, l1) = outs
        assert np.array_equal(t0, t1) and np.array_equal(h0, h1) and l0 == l1 == L + 1
        assert list(t1) == [int(np.argmax(r)) for r in lg]
        assert np.all(h1 == -7) if L == stride else np.array_equal(h1[:, L], t1)


def test_argmax_bump_refusals(hip):
    tok, lg, pv, pi = (hip.Buffer(4096) for _ in range(4))
    hist, ln = hip.Buffer(64), hip.Buffer(4)
    for kw in (dict(bump=1), dict(bump=1, hist=1, hstride=4, temp=0.5)):
        with pytest.raises(hip.ThvmHipError, match="bump"):
            hip.builtin("argmax", [tok, lg, pv, pi, hist, ln], b=1, v=64, nb=8, **kw)


@pytest.mark.parametrize("bump", [0, 1])
@pytest.mark.parametrize("B", [17, 64, 70, 1000])
def test_argmax_over_many_rows(hip, B, bump):
    """Each row a block of its own, or (bump) one block whose waves take several."""
    say(f"case: argmax rows B={B} bump={bump}")
    V, nb, stride, L = 300, 7, 12, 5
    lg = np.random.default_rng(B).standard_normal((B, V)).astype(np.float32)
    lg[:, 250] = lg[:, 31] = 9.0                        # ties: the lowest index
    tok, pv, pi, hist = (hip.Buffer(n) for n in (B * 4, B * nb * 4, B * nb * 4, B * stride * 4))
    ln = up(hip, np.array([L], np.int32))
    hip.builtin("argmax", [tok, up(hip, lg), pv, pi, hist, ln], b=B, v=V, nb=nb, hist=1, hstride=stride, bump=bump)
    assert np.all(tok.read(np.int32) == 31)
    h = hist.read(np.int32).reshape(B, stride)
    assert np.all(h[:, L] == 31) and not np.delete(h, L, 1).any() and ln.read(np.int32)[0] == L + bump
