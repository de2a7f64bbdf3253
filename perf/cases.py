"""Performance cases: the decode work a program has this framework do, from a
GPT-2 small token to a whole Llama-8B-shape step, with the inputs, the outputs
and the 64-bit reference of each.

Three kinds of work, all through the public entry points:

  layers   one or a few transformer layers (or only their attention / FFN
           sublayers) of a decoder, captured once with ``Jit`` from the
           decoder's own op list and replayed: embedding -> layers -> residual
           stream and caches.  ``part`` is "all", "attn" or "ffn".
  decode   a whole model: ``set_state`` then ``replay(steps)`` -> logits.
  prompt   ``generate`` over a prompt (prompt ingestion to the first id).

A case is a dict of plain values: ``arch`` ("llama", "gpt2", "dsv2"), the
model's shape in the fields of ``thvm_amd.Decoder``, ``batch``, ``ctx`` (cache
rows before the step; the prompt length for "prompt") and the weight and
activation types.  Weights, caches and tokens are drawn from the seed alone,
tensor by tensor, so the reference makes the same model without a decoder."""
from __future__ import annotations

import math
import zlib

import torch

import thvm_amd as thvm

_DT = {"fp8": 9, "fp16": 11, "bf16": 12, "fp32": 13}
_TORCH = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
_SIZE = {"fp8": 1, "fp16": 2, "bf16": 2, "fp32": 4}
_ARCH = {"llama": 1, "gpt2": 2, "dsv2": 3}


# ---- the cases --------------------------------------------------------------

def _llama(name, **kw):
    c = dict(name=name, kind="layers", part="all", arch="llama", layers=1, dim=4096, heads=32, kv_heads=8,
             hd=128, ffn=14336, vocab=4096, batch=1, ctx=2048, wdt="fp8", adt="bf16")
    c.update(kw)
    return c


def _gpt2(name, **kw):
    c = dict(name=name, kind="layers", part="all", arch="gpt2", layers=12, dim=768, heads=12, kv_heads=12,
             hd=64, ffn=3072, vocab=50257, batch=1, ctx=128, wdt="fp32", adt="fp32")
    c.update(kw)
    return c


def _dsv2(name, **kw):
    c = dict(name=name, kind="layers", part="attn", arch="dsv2", layers=1, dim=2048, heads=16, kv_heads=16,
             hd=192, ffn=256, vocab=4096, batch=1, ctx=4096, wdt="fp8", adt="bf16", kv_lora=512, d_nope=128,
             d_rope=64, d_v=128, experts=64, shared=2, top_k=6, inter=1408)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest model a user runs: 16 greedy tokens of GPT-2 small in fp32, where launches dominate
        _gpt2("gpt2_small_decode", kind="decode", steps=16, ctx=16),
        # GPT-2 XL served to eight users: fp16 layers at a chat-sized context
        _gpt2("gpt2_xl_b8", layers=4, dim=1600, heads=25, kv_heads=25, ffn=6400, vocab=4096, batch=8,
              wdt="fp16", adt="fp16"),
        # the headline: one user's token of a Llama-8B-shape model with fp8 weights at context 2048, here eight of
        # its 32 layers and the whole head (two correct orders of the attention's sums leave logits of bf16
        # activations 1.4e-2 apart after 8 layers and 3.5e-2 after 32)
        _llama("llama_8b_decode", kind="decode", steps=1, layers=8, vocab=128256),
        # the same layer for three users at a ragged context, a serving batch, and a full batch at a short context
        _llama("llama_layer_b3", batch=3, ctx=1777),
        _llama("llama_layer_b16", batch=16),
        _llama("llama_layer_b60", batch=60, ctx=1000),
        # long documents: two rows at 40000 cache rows, 16-bit weights
        _llama("llama_long", batch=2, ctx=40000, wdt="bf16"),
        # DeepSeek-V2-Lite's latent attention, one user (eight layers' worth, so weights come from HBM) and a batch
        _dsv2("mla_b1", layers=8),
        _dsv2("mla_b32", batch=32, ctx=4001),
        # its mixture of experts, one user (three layers) and a batch
        _dsv2("moe_b1", part="ffn", layers=3, ctx=0),
        _dsv2("moe_b32", part="ffn", batch=32, ctx=0),
        # a prompt of 300 ids read in before the first new id
        _llama("llama_prompt", kind="prompt", layers=4, vocab=128256, ctx=300),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same kinds: any batch and context up to the listed
    ones', widths in multiples of 64, every type pairing the decoders take."""
    what = rng.choice(("llama", "llama", "llama", "gpt2", "gpt2", "mla", "mla", "moe", "moe", "decode", "prompt"))
    if what in ("mla", "moe"):
        batch = rng.choice((rng.randint(1, 4), 4 * _log(rng, 2, 12)))
        c = _dsv2("", batch=batch, part="attn" if what == "mla" else "ffn", dim=128 * rng.randint(8, 32),
                  wdt=rng.choice(("fp8", "fp8", "bf16")), layers=rng.randint(1, 3) if batch <= 4 else 1,
                  ctx=_log(rng, 16, 16384 if batch <= 4 else 4096) if what == "mla" else 0)
        if what == "mla":
            c["heads"] = c["kv_heads"] = rng.choice((8, 16, 16, 16, 32))
        else:
            c.update(experts=rng.randint(16, 64), top_k=rng.randint(2, 6), inter=64 * rng.randint(8, 24),
                     shared=rng.randint(1, 2))
    elif what == "gpt2" or (what == "decode" and rng.random() < 0.5):
        dt = rng.choice(("fp32", "fp16", "bf16"))
        heads = rng.randint(4, 25)
        c = _gpt2("", layers=rng.randint(1, 4), dim=64 * heads, heads=heads, kv_heads=heads, ffn=256 * heads,
                  vocab=4096, batch=rng.randint(1, 4) if dt == "fp32" else _log(rng, 1, 64), ctx=_log(rng, 1, 1000),
                  wdt=dt, adt=dt)
    else:
        hd, kv = rng.choice((64, 128)), rng.choice((1, 2, 4, 8))
        heads = kv * rng.choice([g for g in (1, 2, 4, 8) if 256 <= g * kv * hd <= 4096] or [4])
        batch = _log(rng, 1, 64)
        wdt, adt = rng.choice((("fp8", "bf16"), ("fp8", "bf16"), ("bf16", "bf16"), ("fp16", "fp16"), ("fp8", "fp16")))
        dim = 64 * _log(rng, 8, 64)
        c = _llama("", dim=dim, heads=heads, kv_heads=kv, hd=hd, ffn=64 * round(dim * rng.uniform(2, 4) / 64),
                   batch=batch, ctx=_log(rng, 1, min(32768, 131072 // batch)), wdt=wdt, adt=adt)
    if what == "decode":
        c.update(kind="decode", steps=1, layers=rng.randint(1, 4), vocab=rng.randint(2000, 65000),
                 ctx=min(c["ctx"], 4096))
    if what == "prompt":
        c.update(kind="prompt", layers=rng.randint(1, 4), vocab=rng.randint(2000, 65000), ctx=_log(rng, 4, 300),
                 batch=min(c["batch"], 8))
    del c["name"]
    return c


# ---- the model of a case, from the seed alone ----------------------------------

def _max_seq(c):
    return (c["ctx"] + c.get("steps", 1) + 8 + 63) // 64 * 64


def _shapes(c):
    """name -> (what, shape) of every tensor a case sets: "w" a weight matrix
    [out, in] (fp8: with per-row scales), "a" an activation-type tensor, "f"
    an fp32 matrix, "g" gains near 1, "b" fp32 biases, "c" cache rows."""
    D, V, B, ms, H = c["dim"], c["vocab"], c["batch"], _max_seq(c), c["heads"]
    t = {}
    head = c["kind"] != "layers"
    if c["arch"] == "gpt2":
        t.update({"wte": ("a", (V, D)), "wpe": ("a", (ms, D)), "lnf.g": ("g", (D,)), "lnf.b": ("b", (D,))})
    else:
        t.update({"emb": ("a", (V, D)), "norm_f": ("g", (D,))})
        if head:
            t["lm"] = ("w", (V, D))
    for layer in range(c["layers"]):
        p, F = "l%d." % layer, c["ffn"]
        if c["arch"] == "llama":
            hq, hk = H * c["hd"], c["kv_heads"] * c["hd"]
            t.update({p + "g_attn": ("g", (D,)), p + "g_ffn": ("g", (D,)), p + "wqkv": ("w", (hq + 2 * hk, D)),
                      p + "wo": ("w", (D, hq)), p + "wgu": ("w", (2 * F, D)), p + "wd": ("w", (D, F))})
        elif c["arch"] == "gpt2":
            t.update({p + "ln1.g": ("g", (D,)), p + "ln1.b": ("b", (D,)), p + "ln2.g": ("g", (D,)),
                      p + "ln2.b": ("b", (D,)), p + "c_attn": ("w", (3 * D, D)), p + "c_proj": ("w", (D, D)),
                      p + "c_fc": ("w", (F, D)), p + "mlp_proj": ("w", (D, F))})
            for n, m in (("c_attn", 3 * D), ("c_proj", D), ("c_fc", F), ("mlp_proj", D)):
                t[p + n + ".b"] = ("a", (m,))
        elif c["part"] == "attn":
            kv, dn, dr, dv = c["kv_lora"], c["d_nope"], c["d_rope"], c["d_v"]
            t.update({p + "win": ("g", (D,)), p + "wkvn": ("g", (kv,)), p + "wqkv": ("w", (H * (dn + dr) + kv + dr, D)),
                      p + "wuk": ("w", (H * kv, dn)), p + "wuv": ("w", (H * dv, kv)), p + "wo": ("w", (D, H * dv))})
        else:
            E, inter, S = c["experts"], c["inter"], c["shared"] * c["inter"]
            t.update({p + "wpost": ("g", (D,)), p + "gate": ("f", (E, D)), p + "wgu_e": ("w", (E * 2 * inter, D)),
                      p + "wd_e": ("w", (E * D, inter)), p + "wgu_s": ("w", (2 * S, D)), p + "wd_s": ("w", (D, S))})
        if c["arch"] != "dsv2":
            t[p + "kcache"] = t[p + "vcache"] = ("c", (B, c["kv_heads"], ms, c["hd"]))
        elif c["part"] == "attn":
            t.update({p + "ckv": ("c", (B, ms, c["kv_lora"])), p + "kpe": ("c", (B, ms, c["d_rope"]))})
    return t


def _rng(seed, name):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + zlib.crc32(name.encode())) % (1 << 62))


def _tensor(c, seed, name):
    """(values as stored, per-row scales or None) of one tensor."""
    what, shape = _shapes(c)[name]
    r = torch.randn(shape, generator=_rng(seed, name), device="cuda", dtype=torch.float32)
    if what == "g":
        return 1.0 + 0.1 * r, None
    if what == "b":
        return 0.02 * r, None
    if what == "f":
        return 0.02 * r, None
    if what == "c":   # rows [0, ctx) of a cache that a prompt has filled; nothing after them, or in an empty cache
        r = r.to(_TORCH[c["adt"]])
        r[..., (0 if c["kind"] == "prompt" else c["ctx"]):, :] = 0
        return r, None
    if what == "a":   # embeddings at the scale of a residual stream, except where they are the tied head too
        return (r * (1.0 if name == "emb" else 0.02)).to(_TORCH[c["adt"]]), None
    r *= 0.02
    if c["wdt"] != "fp8":
        return r.to(_TORCH[c["wdt"]]), None
    scale = r.abs().amax(1) / 448.0
    return (r / scale[:, None]).to(torch.float8_e4m3fn), scale


def _tokens(c, seed):
    n = c["ctx"] if c["kind"] == "prompt" else 1
    return torch.randint(0, c["vocab"], (c["batch"], n), generator=_rng(seed, "tokens"), device="cuda").cpu().numpy()


# ---- a program's side -------------------------------------------------------------

class _Model:
    """A decoder and the captured layers, released with the last view of them."""

    def __init__(self, c, seed):
        thvm.init()
        cfg = dict(arch=_ARCH[c["arch"]], n_layers=c["layers"], dim=c["dim"], n_heads=c["heads"],
                   n_kv_heads=c["kv_heads"], head_dim=c["hd"], ffn=c["ffn"], vocab=c["vocab"], max_seq=_max_seq(c),
                   batch=c["batch"], wdtype=_DT[c["wdt"]], adtype=_DT[c["adt"]], eps=1e-5, rope_theta=500000.0,
                   init_std=0.02)
        if c["arch"] == "dsv2":   # attention only: dense FFNs, so that no experts are made
            cfg.update(eps=1e-6, rope_theta=10000.0, kv_lora=c["kv_lora"], d_nope=c["d_nope"], d_rope=c["d_rope"],
                       d_v=c["d_v"], n_experts=c["experts"], n_shared=c["shared"], top_k=c["top_k"],
                       moe_inter=c["inter"], first_dense=c["layers"] if c["part"] == "attn" else 0)
        self.jit = None
        self.dec = thvm.Decoder(seed=int(seed) % (1 << 31), **cfg)

    def __del__(self):
        if self.jit is not None:
            self.jit.drop()
        if getattr(self, "dec", None) is not None:
            self.dec.close()


class _Span:
    """A device buffer for torch; keeps its model."""

    def __init__(self, model, name, kind):
        bid, _, nbytes = model.dec.tensor(name)
        self.model = model
        typ, size = {"fp8": ("|u1", 1), "bf16": ("<i2", 2), "fp16": ("<f2", 2), "fp32": ("<f4", 4),
                     "int32": ("<i4", 4)}[kind]
        self.__cuda_array_interface__ = dict(
            shape=(nbytes // size,), typestr=typ, version=2,
            data=(thvm.lib().thvm_hip_buf_device_ptr(bid), False))


def _view(model, name, kind, shape):
    t = torch.as_tensor(_Span(model, name, kind), device="cuda")
    return (t.view(torch.bfloat16) if kind == "bf16" else t).view(shape)


def prepare(case, seed):
    c = dict(case)
    m = _Model(c, seed)
    shapes = _shapes(c)
    for name, (what, shape) in shapes.items():
        v, scale = _tensor(c, seed, name)
        kind = {"w": c["wdt"], "a": c["adt"], "c": c["adt"]}.get(what, "fp32")
        _view(m, name, kind, shape).copy_(v.view(torch.uint8) if kind == "fp8" else v)
        if scale is not None:
            _view(m, name + ".scale", "fp32", scale.shape).copy_(scale)
        del v, scale
    torch.cuda.synchronize()
    m.dec.sync_weights()
    toks = _tokens(c, seed)
    start = 0 if c["kind"] == "prompt" else c["ctx"]
    m.dec.set_state(toks[:, 0], start)
    B, adt = c["batch"], c["adt"]
    if c["kind"] == "layers":
        # the embedding and the layers of the decoder's step, without its head
        want = {"all": (0, 1), "attn": (0,), "ffn": (1,)}[c["part"]]
        with thvm.Jit() as m.jit:
            for i, tag in enumerate(m.dec.op_tags().tolist()):
                if tag == -1 or (tag >= 0 and tag % 2 in want):
                    thvm.dispatch(*m.dec.op_info(i))
        m.jit.replay()
        out = {"x": _view(m, "x", adt, (B, c["dim"]))}
        out.update({n: _view(m, n, adt, s) for n, (w, s) in shapes.items() if w == "c"})
    else:
        m.dec.capture()                        # runs the step once
        m.dec.set_state(toks[:, 0], start)
        m.dec.replay()
        out = {"logits": _view(m, "logits", "fp32", (B, c["vocab"]))}
        for n in ("l0.kcache", "l0.vcache", "l%d.kcache" % (c["layers"] - 1), "l%d.vcache" % (c["layers"] - 1)):
            out[n] = _view(m, n, adt, shapes[n][1])
        if c["kind"] == "decode" and adt == "fp32":   # at 16 bits another rounding may pick another id
            out["ids"] = _view(m, "hist", "int32", (B, _max_seq(c) + 1))
    torch.cuda.synchronize()
    return {"case": c, "model": m, "tokens": toks, "out": out}


def run(state):
    c, m = state["case"], state["model"]
    if c["kind"] == "layers":
        m.jit.replay()
    elif c["kind"] == "decode":
        m.dec.set_state(state["tokens"][:, 0], c["ctx"])
        m.dec.replay(c["steps"])
    else:
        m.dec.generate(state["tokens"], 1)
    return state["out"]


def work(case):
    c = case
    steps, B, D = c.get("steps", 1), c["batch"], c["dim"]
    rows = B * (c["ctx"] if c["kind"] == "prompt" else 1)      # x rows each weight matrix meets
    wb = wn = cache = 0.0
    for name, (what, shape) in _shapes(c).items():
        n = math.prod(shape)
        if what == "w":
            live = 1.0
            if name.endswith("_e"):   # the experts that `rows` draws of top_k reach, on average
                live = 1.0 - (1.0 - c["top_k"] / c["experts"]) ** rows
            wb += live * (n * _SIZE[c["wdt"]] + (4 * shape[0] if c["wdt"] == "fp8" else 0))
            wn += n * (c["top_k"] / c["experts"] if name.endswith("_e") else 1.0) * \
                (B if name == "lm" else rows)
        elif what == "f":
            wb += 4 * n
            wn += n * rows
        elif name == "wte" and c["kind"] != "layers":
            wb += n * _SIZE[c["adt"]]
            wn += n * B
        elif what == "c":
            cache += B * math.prod(shape[1:]) / shape[-2] * (c["ctx"] + (steps + 1) / 2)
    attn = cache * (2.0 if c["arch"] == "dsv2" else c["heads"] / c["kv_heads"]) * \
        (2 * c["heads"] if c["arch"] == "dsv2" else 2)
    if c["kind"] == "prompt":
        attn *= c["ctx"] / 2
    io = rows * D * 2 * _SIZE[c["adt"]] + (4 * B * c["vocab"] if c["kind"] != "layers" else 0)
    return {"bytes": steps * (wb + cache * _SIZE[c["adt"]] + io), "flops": steps * (2 * wn + attn)}


def tolerance(case):
    """Four times what these outputs are from the 64-bit reference, or from
    themselves with the attention's sums in another order: 4.9e-3 for a bf16
    layer, 1e-3 for fp16, 4e-7 for fp32 (1e-6 taken); through a whole bf16
    model (1.4e-2) no more than 3e-2."""
    if case["adt"] == "fp32":
        return {"rel": 4e-6}
    if case["adt"] == "fp16":
        return {"rel": 0.004 if case["kind"] == "layers" else 0.008}
    return {"rel": 0.02 if case["kind"] == "layers" else 0.03}


# ---- the same in 64 bits -------------------------------------------------------------

class _Exact:
    """The case's model in float64: stored weights, caches and tokens, no rounding between."""

    def __init__(self, c, seed):
        self.c, self.seed = c, seed
        self.cache = {n: _tensor(c, seed, n)[0].double() for n, (w, _) in _shapes(c).items() if w == "c"}

    def w(self, name):
        v, scale = _tensor(self.c, self.seed, name)
        return v.double() if scale is None else v.double() * scale.double()[:, None]

    def embed(self, ids, pos):
        if self.c["arch"] == "gpt2":
            return self.w("wte")[ids] + self.w("wpe")[pos:pos + ids.shape[1]]
        return _tensor(self.c, self.seed, "emb")[0][ids].double()

    def norm(self, x, g, b=None):
        if b is not None:
            x = x - x.mean(-1, keepdim=True)
        eps = 1e-6 if self.c["arch"] == "dsv2" else 1e-5
        y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * self.w(g)
        return y if b is None else y + self.w(b)

    def rope(self, x, pos):
        """Rotates the pairs (2j, 2j+1) of x [B, T, h, d] at positions pos.. ."""
        d, dsv2 = x.shape[-1], self.c["arch"] == "dsv2"
        theta = 10000.0 if dsv2 else 500000.0
        j = torch.arange(d // 2, dtype=torch.float64, device=x.device)
        f = theta ** (-2 * j / d)
        if dsv2:   # YaRN, factor 40 over 4096 positions, beta 32 and 1
            lo, hi = (d * math.log(4096 / (b * 2 * math.pi)) / (2 * math.log(theta)) for b in (32.0, 1.0))
            lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), d - 1)
            ramp = ((j - lo) / max(hi - lo, 1e-3)).clamp(0, 1)
            f = f / 40 * ramp + f * (1 - ramp)
        a = (pos + torch.arange(x.shape[1], device=x.device, dtype=torch.float64))[:, None, None] * f
        e, o = x[..., 0::2], x[..., 1::2]
        e, o = e * a.cos() - o * a.sin(), o * a.cos() + e * a.sin()
        return torch.cat((e, o), -1) if dsv2 else torch.stack((e, o), -1).flatten(-2)

    def mask(self, s, pos):
        """Scores [.., T, rows]: position pos + t sees rows up to its own."""
        T, rows = s.shape[-2:]
        late = torch.arange(rows, device=s.device) > (pos + torch.arange(T, device=s.device))[:, None]
        return s.masked_fill(late, -math.inf).softmax(-1)

    def attention(self, x, p, pos):
        c, (B, T, _) = self.c, x.shape
        H, hk, hd = c["heads"], c["kv_heads"], c["hd"]
        if c["arch"] == "gpt2":
            y = self.norm(x, p + "ln1.g", p + "ln1.b") @ self.w(p + "c_attn").T + self.w(p + "c_attn.b")
        else:
            y = self.norm(x, p + "g_attn") @ self.w(p + "wqkv").T
        q, k, v = (t.unflatten(-1, (-1, hd)) for t in y.split((H * hd, hk * hd, hk * hd), -1))
        if c["arch"] == "llama":
            q, k = self.rope(q, pos), self.rope(k, pos)
        K, V = self.cache[p + "kcache"], self.cache[p + "vcache"]
        K[:, :, pos:pos + T], V[:, :, pos:pos + T] = k.transpose(1, 2), v.transpose(1, 2)
        K, V = K[:, :, :pos + T], V[:, :, :pos + T]
        q = q.transpose(1, 2).reshape(B, hk, H // hk * T, hd)          # a kv head's query heads, T positions each
        s = (q @ K.transpose(-1, -2).contiguous() / math.sqrt(hd)).unflatten(2, (H // hk, T))
        o = (self.mask(s, pos).flatten(2, 3) @ V).unflatten(2, (H // hk, T)).flatten(1, 2)
        o = o.transpose(1, 2).reshape(B, T, H * hd)
        if c["arch"] == "gpt2":
            return x + o @ self.w(p + "c_proj").T + self.w(p + "c_proj.b")
        return x + o @ self.w(p + "wo").T

    def latent(self, x, p, pos):
        c, (B, T, _) = self.c, x.shape
        H, kv, dn, dr, dv = (c[k] for k in ("heads", "kv_lora", "d_nope", "d_rope", "d_v"))
        y = self.norm(x, p + "win") @ self.w(p + "wqkv").T
        q, lat, kpe = y.split((H * (dn + dr), kv, dr), -1)
        q = q.unflatten(-1, (H, dn + dr))
        qpe = self.rope(q[..., dn:], pos)
        C, P = self.cache[p + "ckv"], self.cache[p + "kpe"]
        C[:, pos:pos + T], P[:, pos:pos + T] = self.norm(lat, p + "wkvn"), self.rope(kpe[:, :, None], pos)[:, :, 0]
        C, P = C[:, :pos + T], P[:, :pos + T]
        qlat = torch.einsum("bthd,hkd->bhtk", q[..., :dn], self.w(p + "wuk").view(H, kv, dn))
        ms = 0.1 * 0.707 * math.log(40.0) + 1.0
        s = (qlat.flatten(1, 2) @ C.transpose(1, 2).contiguous() +
             qpe.transpose(1, 2).flatten(1, 2) @ P.transpose(1, 2).contiguous()) * (dn + dr) ** -0.5 * ms * ms
        o = (self.mask(s.unflatten(1, (H, T)), pos).flatten(1, 2) @ C).unflatten(1, (H, T))
        o = torch.einsum("bhtk,hdk->bthd", o, self.w(p + "wuv").view(H, dv, kv))
        return x + o.flatten(2) @ self.w(p + "wo").T

    @staticmethod
    def swiglu(x, wgu, wd):
        y = x @ wgu.T
        return torch.nn.functional.silu(y[..., 0::2]) * y[..., 1::2] @ wd.T

    def ffn(self, x, p):
        c = self.c
        if c["arch"] == "gpt2":
            y = self.norm(x, p + "ln2.g", p + "ln2.b") @ self.w(p + "c_fc").T + self.w(p + "c_fc.b")
            y = torch.nn.functional.gelu(y, approximate="tanh")
            return x + y @ self.w(p + "mlp_proj").T + self.w(p + "mlp_proj.b")
        if c["arch"] == "llama":
            return x + self.swiglu(self.norm(x, p + "g_ffn"), self.w(p + "wgu"), self.w(p + "wd"))
        E, inter, D = c["experts"], c["inter"], c["dim"]
        h = self.norm(x, p + "wpost")
        prob, sel = (h @ self.w(p + "gate").T).softmax(-1).topk(c["top_k"], -1)
        y = self.swiglu(h, self.w(p + "wgu_s"), self.w(p + "wd_s"))
        wgu, wd = self.w(p + "wgu_e").view(E, 2 * inter, D), self.w(p + "wd_e").view(E, D, inter)
        for e in range(E):
            y = y + (prob * (sel == e)).sum(-1, keepdim=True) * self.swiglu(h, wgu[e], wd[e])
        return x + y

    def forward(self, ids, pos):
        """ids [B, T] at positions pos.. -> the residual stream [B, T, D]."""
        x, part = self.embed(ids, pos), self.c["part"]
        for layer in range(self.c["layers"]):
            p = "l%d." % layer
            if part != "ffn":
                x = (self.latent if self.c["arch"] == "dsv2" else self.attention)(x, p, pos)
            if part != "attn":
                x = self.ffn(x, p)
        return x

    def logits(self, x):
        if self.c["arch"] == "gpt2":
            return self.norm(x, "lnf.g", "lnf.b") @ self.w("wte").T
        return self.norm(x, "norm_f") @ self.w("lm").T


def exact(case, seed):
    c = dict(case)
    m = _Exact(c, seed)
    ids = torch.from_numpy(_tokens(c, seed)).cuda()
    pos = 0 if c["kind"] == "prompt" else c["ctx"]
    if c["kind"] == "layers":
        return {"x": m.forward(ids, pos)[:, -1], **m.cache}
    for s in range(c.get("steps", 1)):
        logits = m.logits(m.forward(ids, pos + s)[:, -1])
        ids = logits.argmax(-1, keepdim=True)
    last = "l%d." % (c["layers"] - 1)
    out = {"logits": logits, **{n: m.cache[n] for n in ("l0.kcache", "l0.vcache", last + "kcache", last + "vcache")}}
    if c["kind"] == "decode" and c["adt"] == "fp32":
        out["ids"] = None
    return out
