"""Prompt ingestion in chunks (generate over two positions or more): the causal
chunk attention against float64 softmax attention at every edge of its tiles,
and generate() against the same prompt fed a step at a time, over the model
forms it takes and those it leaves to the step."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

DT_FP8, DT_F16, DT_BF16, DT_F32 = 9, 11, 12, 13


def say(*a):
    print(*a, flush=True)


def up(hip, a):
    return hip.Buffer.from_numpy(np.ascontiguousarray(a))


@pytest.mark.parametrize("dt", [DT_BF16, DT_F16])
@pytest.mark.parametrize("H,Hkv,hd", [(4, 2, 64), (3, 3, 64), (8, 2, 128), (6, 2, 128), (16, 1, 128)])
@pytest.mark.parametrize("B,T,pos", [(1, 1, 0), (2, 15, 0), (1, 16, 1), (1, 17, 62), (3, 33, 15), (1, 130, 300)])
def test_attn_prompt(hip, dt, H, Hkv, hd, B, T, pos):
    """Position t sees rows [0, pos + t]; rows after the chunk hold NaN and
    must not reach a result."""
    say(f"case: attn_prompt dt={dt} H={H} Hkv={Hkv} hd={hd} B={B} T={T} pos={pos}")
    rng = np.random.default_rng(H * 1000 + hd + T + pos)
    ms = pos + T + 5
    q, k, v = (O.encode(rng.standard_normal(s).astype(np.float32), dt)
               for s in ((B, T, H, hd), (B, Hkv, ms, hd), (B, Hkv, ms, hd)))
    k[:, :, pos + T:] = v[:, :, pos + T:] = 0x7FFF
    out = hip.Buffer(B * T * H * hd * 2)
    scale = 1.0 / np.sqrt(hd)
    hip.builtin("attn_prompt", [out, up(hip, q), up(hip, k), up(hip, v), up(hip, np.array([pos + 1], np.int32))],
                b=B, t=T, h=H, hkv=Hkv, hd=hd, maxseq=ms, dt=dt, scale=float(scale))
    got = O.decode(out.read(np.uint16), dt).reshape(B, T, H, hd).astype(np.float64)
    qf, kf, vf = (O.decode(a, dt).astype(np.float64) for a in (q, k[:, :, :pos + T], v[:, :, :pos + T]))
    g = H // Hkv
    for h in range(H):
        s = np.einsum("btd,bjd->btj", qf[:, :, h], kf[:, h // g]) * scale
        s = np.where(np.arange(pos + T)[None, None] <= pos + np.arange(T)[None, :, None], s, -np.inf)
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        want = np.einsum("btj,bjd->btd", p, vf[:, h // g])
        floor = np.einsum("btj,bjd->btd", p, np.abs(vf[:, h // g]))
        ulp = 2.0 ** -8 if dt == DT_BF16 else 2.0 ** -11
        assert np.all(np.abs(got[:, :, h] - want) <= ulp * np.abs(want) + 1e-4 * floor), h


LLAMA = dict(arch=1, n_layers=2, dim=256, n_heads=4, n_kv_heads=2, head_dim=64, ffn=512, vocab=600, max_seq=640,
             batch=1, eps=1e-5, rope_theta=500000.0, init_std=0.05, wdtype=DT_FP8, adtype=DT_BF16)
GPT2 = dict(arch=2, n_layers=2, dim=256, n_heads=4, n_kv_heads=4, head_dim=64, ffn=1024, vocab=600, max_seq=640,
            batch=1, eps=1e-5, init_std=0.05, wdtype=DT_F16, adtype=DT_F16)
FORMS = {"fp8": dict(LLAMA), "bf16": dict(LLAMA, wdtype=DT_BF16), "fp8-fp16": dict(LLAMA, adtype=DT_F16),
         "fp16-b3": dict(LLAMA, wdtype=DT_F16, adtype=DT_F16, batch=3), "fp8-b8": dict(LLAMA, batch=8),
         "gqa4-hd128": dict(LLAMA, dim=512, n_heads=4, n_kv_heads=1, head_dim=128, batch=2),
         "gpt2-fp16": dict(GPT2), "gpt2-bf16-b5": dict(GPT2, wdtype=DT_BF16, adtype=DT_BF16, batch=5),
         "sampled": dict(LLAMA, temperature=0.8, sample_seed_lo=3),
         # forms the chunk kernels do not take: the step, bit for bit
         "f32": dict(LLAMA, wdtype=DT_F32, adtype=DT_F32), "bf16-w-fp16-x": dict(LLAMA, wdtype=DT_BF16, adtype=DT_F16),
         "persistent": dict(LLAMA, dim=512, n_heads=8, n_kv_heads=4, step_mode=1)}
STEPPED = ("f32", "bf16-w-fp16-x", "persistent")


def stepped(hip, cfg, prompt):
    """The prompt a step at a time: caches, logits, next ids, position."""
    dec = hip.Decoder(seed=11, **cfg)
    try:
        for i in range(prompt.shape[1]):
            dec.set_state(prompt[:, i], i)
            dec.step()
        return state(dec, cfg, prompt.shape[1])
    finally:
        dec.close()


def state(dec, cfg, n):
    c = {}
    for l in range(cfg["n_layers"]):
        for k in ("kcache", "vcache"):
            a = dec.read_tensor(f"l{l}.{k}")
            c[f"l{l}.{k}"] = (a if a.dtype == np.float32 else O.decode(a, cfg["adtype"])).reshape(
                cfg["batch"], -1, cfg["max_seq"], cfg["head_dim"]).astype(np.float64)
    return c, dec.logits().astype(np.float64), dec.tokens(n + 1), dec.position


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# 515 ids: a second chunk at one sequence (the stepped forms have no chunks)
@pytest.mark.parametrize("n,form", [(n, f) for n in (1, 2, 17, 70, 515) for f in FORMS if n < 515 or f not in STEPPED])
def test_generate_prompt_equals_steps(hip, n, form):
    cfg = FORMS[form]
    say(f"case: prompt of {n} ids, {form}")
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], (cfg["batch"], n)).astype(np.int32)
    wc, wl, wt, wp = stepped(hip, cfg, prompt)
    for captured in (False, True):
        dec = hip.Decoder(seed=11, **cfg)
        try:
            if captured:
                dec.set_state(prompt[:, 0], 0)
                dec.capture()
            ids, cnt = dec.generate(prompt, 1)
            gc, gl, gt, gp = state(dec, cfg, n)
        finally:
            dec.close()
        exact = form in STEPPED or n == 1
        assert gp == wp == n and np.array_equal(gt[:, :n], prompt) and np.all(cnt == 1)
        assert np.array_equal(ids[:, 0], gt[:, n])
        # two correct orders of every sum through two layers of 16-bit activations
        bar = 0.0 if exact else 4e-3 if cfg["adtype"] == DT_F16 else 2.5e-2
        for k in wc:
            assert rel(gc[k], wc[k]) <= bar, k
            assert not gc[k][:, :, n:].any() or captured, k
        assert rel(gl, wl) <= bar, rel(gl, wl)
        if exact:
            assert np.array_equal(gt, wt)
        elif not cfg.get("temperature"):   # greedy: the largest logit, up to the bar
            for b in range(cfg["batch"]):
                assert wl[b, gt[b, n]] >= wl[b].max() - 4 * bar * wl[b].std()


def test_generate_continues_after_a_chunked_prompt(hip):
    """Ids after a chunked prompt equal steps from the state it left, with the
    step captured before or during the call, and eos stops a row."""
    cfg = dict(LLAMA, batch=2)
    prompt = np.random.default_rng(2).integers(0, cfg["vocab"], (2, 40)).astype(np.int32)
    say("case: generate past a chunked prompt")
    dec = hip.Decoder(seed=11, **cfg)
    try:
        first, n1 = dec.generate(prompt, 20)          # captures its step on the way
        again, n2 = dec.generate(prompt, 20)
        assert np.array_equal(first, again) and np.all(n1 == 20) and np.all(n2 == 20)
        one, _ = dec.generate(prompt, 1)
        for _ in range(19):
            dec.step()
        assert np.array_equal(dec.tokens(60)[:, 40:], first)
        eos = int(first[0, 5])
        out, cnt = dec.generate(prompt, 20, eos=eos)
        stop = int(np.argmax(first[0] == eos))
        assert cnt[0] == stop and np.array_equal(out[0, :stop], first[0, :stop]) and np.all(out[0, stop:] == -1)
        with pytest.raises(hip.ThvmHipError, match="outside"):
            dec.generate(np.where(np.arange(40) == 20, cfg["vocab"], prompt), 1)
    finally:
        dec.close()


@pytest.mark.parametrize("new", [0, 1])
def test_replay_after_a_chunked_prompt(hip, new):
    """A fresh decoder's generate() leaves a step to replay, also where the
    request ends before any step ran; without a request replay stays refused."""
    prompt = np.random.default_rng(3).integers(0, LLAMA["vocab"], (1, 20)).astype(np.int32)
    say("case: replay after a chunked prompt", new)
    ids = []
    for replay in (False, True):
        dec = hip.Decoder(seed=11, **LLAMA)
        try:
            if replay:
                with pytest.raises(hip.ThvmHipError, match="no captured step"):
                    dec.replay(1)
                dec.generate(prompt, new)
                dec.replay(9)
                assert dec.position == 20 + 9
            else:
                dec.generate(prompt, 10)
            ids.append(dec.tokens(30))
        finally:
            dec.close()
    assert np.array_equal(ids[0], ids[1])


@pytest.mark.parametrize("n,new", [(2, 24), (50, 24), (50, 0), (50, 1)])
def test_speculative_generate_after_a_chunked_prompt(hip, n, new):
    """A speculative request reads its prompt in the plain request's chunks: the
    caches and the first id are the same bits, whatever the row count does to
    the order of the GEMM's sums."""
    prompt = np.random.default_rng(5).integers(0, LLAMA["vocab"], (1, n)).astype(np.int32)
    out, caches = [], []
    for spec in (0, 4):
        say("case: speculative generate past a chunked prompt", n, new, spec)
        dec = hip.Decoder(seed=11, **dict(LLAMA, spec_rows=spec))
        try:
            out.append(dec.generate(prompt, new)[0])
            caches.append(dec.read_tensor(f"l{LLAMA['n_layers'] - 1}.kcache")
                          .reshape(LLAMA["n_kv_heads"], LLAMA["max_seq"], -1)[:, :n].copy())
        finally:
            dec.close()
    assert np.array_equal(caches[0], caches[1])
    assert np.array_equal(out[0], out[1])          # a verify row is the one-row step, bit for bit


@pytest.mark.parametrize("n", [3, 4, 5])
def test_prompt_over_a_long_ffn_row(hip, n):
    """ffn = 20480: four positions' rows of the down projection fill the GEMV's
    LDS to the byte, so its chunk of four ids runs on the MFMA GEMM."""
    cfg = dict(LLAMA, n_layers=1, dim=128, n_heads=2, n_kv_heads=1, ffn=20480, max_seq=64, wdtype=DT_BF16)
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], (1, n)).astype(np.int32)
    say("case: prompt over a long ffn row", n)
    wc, wl, _, _ = stepped(hip, cfg, prompt)
    dec = hip.Decoder(seed=11, **cfg)
    try:
        dec.generate(prompt, 1)
        gc, gl, _, gp = state(dec, cfg, n)
    finally:
        dec.close()
    # (the bar of test_generate_prompt_equals_steps for bf16)
    assert gp == n and rel(gl, wl) <= 2.5e-2 and all(rel(gc[k], wc[k]) <= 2.5e-2 for k in wc)


def test_generate_after_a_pool_rollback(hip):
    """The chunk workspace, made inside the first request, outlives a rollback
    to a watermark taken before that request, and the same ids come back."""
    cfg = dict(LLAMA, batch=2)
    prompt = np.random.default_rng(7).integers(0, cfg["vocab"], (2, 40)).astype(np.int32)
    say("case: generate, pool rollback, generate")
    L = hip.lib()
    dec = hip.Decoder(seed=11, **cfg)
    try:
        wm = L.thvm_hip_buf_pool_begin()
        first, _ = dec.generate(prompt, 6)
        L.thvm_hip_buf_pool_rollback_with_preserve(wm)
        L.thvm_hip_buf_clear_preserved(wm)
        again, _ = dec.generate(prompt, 6)
        assert np.array_equal(first, again)
    finally:
        dec.close()


_SWEPT_CHILD = """
import sys
sys.path[:0] = [{root!r}, {tests!r}]
import numpy as np
import thvm_amd
import test_gpu_prompt as T
thvm_amd.init()
prompt = np.random.default_rng(8).integers(0, T.LLAMA["vocab"], (1, 40)).astype(np.int32)
dec = thvm_amd.Decoder(seed=11, **T.LLAMA)
want, _ = dec.generate(prompt, 6)
dec.close()
dec = thvm_amd.Decoder(seed=11, **T.LLAMA)
dec.generate(prompt, 1)                        # ends before any step is captured
thvm_amd.lib().thvm_hip_buf_free_unpreserved_all()
got, _ = dec.generate(prompt, 6)
assert np.array_equal(got, want)
dec.close()
thvm_amd.shutdown()
print("swept child ok", flush=True)
"""


def test_generate_holds_the_step_against_a_sweep(hip):
    """A request that ends with its prompt holds the step's buffers as one that
    captured the step does: the table-wide sweep leaves the decoder whole (in a
    process of its own, the sweep would take other tests' buffers)."""
    import subprocess
    import sys
    from pathlib import Path
    root = Path(__file__).resolve().parents[1]
    say("case: generate, table-wide sweep, generate (child process)")
    r = subprocess.run([sys.executable, "-c", _SWEPT_CHILD.format(root=str(root), tests=str(root / "tests"))],
                       capture_output=True, text=True, timeout=100)
    say(r.stdout[-2000:], r.stderr[-2000:])
    assert r.returncode == 0 and "swept child ok" in r.stdout


@pytest.mark.parametrize("H,Hkv,hd", [(8, 4, 64), (3, 3, 128)])
def test_attn_prompt_keeps_p_in_f32(hip, H, Hkv, hd):
    """Over hundreds of near-equal probabilities an output is the nearest bf16 of
    the float64 result except where that lies within the f32 sums' error of a
    midpoint: about c 2^-24 / 2^-8 of the values for an error of c f32 ulps (4 of
    them give 2.5e-4; p cut to 16 bits gave 2e-3)."""
    T, ms, dt = 500, 512, DT_BF16
    say(f"case: attn_prompt p in f32 H={H} hd={hd}")
    rng = np.random.default_rng(hd)
    q = O.encode((0.2 * rng.standard_normal((1, T, H, hd))).astype(np.float32), dt)
    k, v = (O.encode(rng.standard_normal((1, Hkv, ms, hd)).astype(np.float32), dt) for _ in range(2))
    out, scale = hip.Buffer(T * H * hd * 2), float(np.float32(1 / np.sqrt(hd)))
    hip.builtin("attn_prompt", [out, up(hip, q), up(hip, k), up(hip, v), up(hip, np.array([1], np.int32))],
                b=1, t=T, h=H, hkv=Hkv, hd=hd, maxseq=ms, dt=dt, scale=scale)
    got = out.read(np.uint16).reshape(T, H, hd)
    qf, kf, vf = (O.decode(a, dt).astype(np.float64)[0] for a in (q, k, v))
    off = 0
    for h in range(H):
        s = qf[:, h] @ kf[h * Hkv // H].T * scale
        s = np.where(np.arange(ms)[None] <= np.arange(T)[:, None], s, -np.inf)
        p = np.exp(s - s.max(-1, keepdims=True))
        want = (p / p.sum(-1, keepdims=True)) @ vf[h * Hkv // H]
        off += (O.encode(want.astype(np.float32), dt) != got[:, h]).sum()
    assert off <= 5e-4 * got.size, off / got.size


@pytest.mark.parametrize("dt,bits", [(DT_BF16, 0x7F80), (DT_BF16, 0xFFC0), (DT_F16, 0x7C00), (DT_F16, 0xFC00), (DT_F16, 0x7E01)])
@pytest.mark.parametrize("H,Hkv,hd", [(4, 2, 64), (3, 3, 128)])
@pytest.mark.parametrize("T,pos,at", [(40, 0, 7), (33, 21, 15), (48, 16, 47), (5, 14, 0)])
def test_attn_prompt_later_v_not_finite(hip, dt, bits, H, Hkv, hd, T, pos, at):
    """An infinity or NaN in one value of a chunk row's V reaches that row's
    position and the ones after it, in that value alone; the positions before
    it, which share its tile of rows, keep their bits."""
    say(f"case: attn_prompt V not finite dt={dt} bits={bits:x} H={H} hd={hd} T={T} pos={pos} at={at}")
    rng = np.random.default_rng(T + pos + at)
    ms, scale, d, kvh = pos + T + 3, float(np.float32(1 / np.sqrt(hd))), hd - 3, Hkv - 1
    q, k, v = (O.encode(rng.standard_normal(s).astype(np.float32), dt) for s in ((1, T, H, hd), (1, Hkv, ms, hd), (1, Hkv, ms, hd)))
    outs = []
    for x in (None, bits):
        vv = v.copy()
        if x is not None:
            vv[0, kvh, pos + at, d] = x
        out = hip.Buffer(T * H * hd * 2)
        hip.builtin("attn_prompt", [out, up(hip, q), up(hip, k), up(hip, vv), up(hip, np.array([pos + 1], np.int32))],
                    b=1, t=T, h=H, hkv=Hkv, hd=hd, maxseq=ms, dt=dt, scale=scale)
        outs.append(out.read(np.uint16).reshape(T, Hkv, H // Hkv, hd))
    hit = np.zeros(outs[0].shape, bool)
    hit[at:, kvh, :, d] = True
    assert np.array_equal(outs[0][~hit], outs[1][~hit])
    f = O.decode(outs[1][hit], dt)
    assert not np.isfinite(f).any()
    if bits in (0x7F80, 0x7C00, 0xFC00) and at // 16 == (T - 1) // 16:
        assert np.all(np.isinf(f) & (np.signbit(f) == (bits > 0x7FFF)))
