"""What the library is timed on: the calls of a decode engine's attention
layers and greedy head, at the sizes and layouts the benchmark, the tests and
the Node host use.

Five kinds of pass, each through the public entry points of ``nwd_attn``:

  step     one attention-layer step: append_decode (or, with "calls": 2,
           kv_append then decode) for `batch` sequences
  prefill  a prompt chunk through attention: kv_append, then prefill
  token    the attention layers of a token from the normalised hidden state:
           per layer qkv_append, decode, o_proj added to the residual
  chunk    a prompt chunk through one attention layer from the hidden state:
           q/k/v projections, kv_append, prefill, o_proj added to the residual
  head     lm_head with the greedy pick

`past` is the number of cached tokens per sequence; where `past_min` is
below it, every sequence draws its own from [past_min, past].
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "nemotron-webgpu-decode_amd"))
import nwd_attn as nw  # noqa: E402

HIDDEN = 3136  # the Nano-4B hidden size

# (query heads, KV heads, head size) of the model layouts the benchmark and
# the tests name.
LAYOUTS = [(32, 8, 128), (40, 8, 128), (28, 4, 128), (24, 8, 128), (12, 2, 128), (128, 8, 128),
           (32, 8, 64), (14, 2, 64), (15, 5, 64), (16, 8, 256), (32, 32, 96)]


def _case(kind, batch, layout, past, past_min=None, dtype="f16", **more):
    heads, kv, dim = layout
    return dict(kind=kind, batch=batch, heads=heads, kv=kv, dim=dim, past=past,
                past_min=past if past_min is None else past_min, dtype=dtype, **more)


def listed():
    base, nano = (32, 8, 128), (40, 8, 128)
    return [
        # The reference engine's own size (its cache holds 256 keys): one
        # token of a short chat, where the launch and its round trips count.
        dict(_case("step", 1, base, 152), name="step-153"),
        # A chat of some pages in the engine's own types (f32 q, k, v, out)
        # and head layout.
        dict(_case("step", 1, nano, 4096, dtype="f32"), name="step-4k-f32"),
        # A long document: the benchmark's headline, 1% of K/V at +-8.
        dict(_case("step", 1, base, 32768, outliers=True), name="step-32k"),
        # A server's batch of sequences of every length.
        dict(_case("step", 64, base, 16384, 512), name="step-ragged-64"),
        # A small model's layout (head size 64) at a long context.
        dict(_case("step", 1, (32, 8, 64), 16384), name="step-d64-16k"),
        # A prompt chunk onto a long context.
        dict(_case("prefill", 1, base, 8192, new=512), name="prefill-512"),
        # Short prompts of four chats at once, of odd length, onto what each
        # has, in the engine's types.
        dict(_case("prefill", 4, nano, 1500, 0, "f32", new=77), name="prefill-4x77-f32"),
        # One token through the model's four attention layers, as the Node
        # host drives them.
        dict(_case("token", 1, nano, 4096, dtype="f32", layers=4), name="token-4k"),
        # The same layer for a server's batch.
        dict(_case("token", 32, nano, 4096, 256, "f32", layers=1), name="token-32-ragged"),
        # A prompt chunk through an attention layer from the hidden state, as
        # the Node host's prefill drives it.
        dict(_case("chunk", 1, nano, 1024, dtype="f32", new=512), name="chunk-512"),
        # The end of a token: 131072 logits and the greedy pick.
        dict(kind="head", batch=1, hidden=HIDDEN, vocab=131072, name="head-1"),
        # The same for a server's batch.
        dict(kind="head", batch=16, hidden=HIDDEN, vocab=131072, name="head-16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "prefill", "token", "chunk", "head"])
    dtype = rng.choice(["f16", "f32"])
    if kind == "head":
        return dict(kind="head", batch=_log(rng, 1, 48), hidden=32 * _log(rng, 28, 160),
                    vocab=_log(rng, 30000, 131072))
    if kind == "step":
        heads, kv, dim = layout = rng.choice(LAYOUTS)
        batch = _log(rng, 1, 64)
        # at most the 64 x 16384 x 8 x 128 elements of the listed batch's cache
        top = min(32768, (64 * 16384 * 8 * 128) // (batch * kv * dim))
        past = _log(rng, 100, top)
        c = _case("step", batch, layout, past, rng.choice([past, past // 8]), dtype)
        return dict(c, calls=2) if rng.random() < 0.25 else c
    if kind == "prefill":
        heads, kv, dim = layout = rng.choice([x for x in LAYOUTS if x[0] < 128])
        new, batch = _log(rng, 16, 512), _log(rng, 1, 8)
        # at most the work of 512 tokens of 32 heads of 128 onto 8192
        top = min(16384, 512 * 8192 * 32 * 128 // (new * batch * heads * dim))
        past = _log(rng, 16, max(16, top))
        return _case("prefill", batch, layout, past, rng.choice([past, past // 8]), dtype, new=new)
    layout = rng.choice([(40, 8, 128), (32, 8, 128), (28, 4, 128), (14, 2, 64), (16, 8, 256)])
    hidden = 32 * _log(rng, 28, 128)
    if kind == "token":
        past = _log(rng, 100, 4096)
        return _case("token", _log(rng, 1, 64), layout, past, rng.choice([past, past // 8]),
                     rng.choice(["f16", "f32"]), layers=rng.choice([1, 2]), hidden=hidden)
    return _case("chunk", 1, layout, _log(rng, 1, 2048), dtype="f32", new=_log(rng, 16, 512),
                 hidden=hidden)


# ------------------------------------------------------------------- inputs

_T = {"f16": torch.float16, "f32": torch.float32}


def _pasts(c, seed):
    lo, hi = c["past_min"], c["past"]
    p = np.random.Generator(np.random.PCG64(seed)).integers(lo, hi + 1, size=c["batch"])
    if lo < hi:
        p[-1] = hi
    return [int(v) for v in p]


def _q4(g, n, k):
    """A 4-bit projection [k -> n] in the MatMulNBits format: every nibble,
    zero points around 8, outputs of N(0, 1) inputs near N(0, 1)."""
    nb = k // 32
    quant = torch.randint(0, 256, (n, nb, 16), generator=g, device="cuda", dtype=torch.uint8)
    scales = (torch.rand((n, nb), generator=g, device="cuda") + 0.5) * (0.21 / math.sqrt(k))
    z = torch.randint(6, 11, (2, (n * nb + 1) // 2), generator=g, device="cuda", dtype=torch.uint8)
    zp = z[0] | (z[1] << 4)
    return {"quant": quant, "scales": scales, "zp": zp, "w": nw.q4_weight(quant, scales, zp, n, nb)}


def _dense(w, c0=0, c1=None):
    """Columns c0:c1 of a projection as float64 [columns][k]."""
    n, nb = w["scales"].shape
    c1 = n if c1 is None else min(c1, n)
    i = torch.arange(c0 * nb, c1 * nb, device="cuda")
    z = torch.where(i % 2 == 0, w["zp"][i // 2] & 15, w["zp"][i // 2] >> 4).view(c1 - c0, nb, 1)
    q = w["quant"][c0:c1]
    nib = torch.stack([q & 15, q >> 4], dim=-1).view(c1 - c0, nb, 32)
    v = (nib.double() - z.double()) * w["scales"][c0:c1].double().unsqueeze(-1)
    return v.view(c1 - c0, nb * 32)


def _project(w, x):
    """x [rows][k] in float64 through a projection."""
    return torch.cat([x.double() @ _dense(w, c, c + 16384).t()
                      for c in range(0, w["scales"].shape[0], 16384)], dim=1)


def prepare(case, seed):
    c = dict(case)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def rnd(*shape, dtype="f32"):
        return torch.randn(shape, generator=g, device="cuda", dtype=_T[dtype])

    if c["kind"] == "head":
        s = {"c": c, "w": _q4(g, c["vocab"], c["hidden"]), "x": rnd(c["batch"], c["hidden"])}
        s["logits"] = torch.empty((c["batch"], c["vocab"]), device="cuda")
        s["token"] = torch.empty(c["batch"], dtype=torch.int32, device="cuda")
        s["ctx"] = nw.AttnContext(40, 8, 256, max_batch=c["batch"], q_dtype="f32", o_dtype="f32",
                                  kv_dtype="f32")
        return s
    B, H, KV, D, t = c["batch"], c["heads"], c["kv"], c["dim"], c["dtype"]
    new, layers, hidden = c.get("new", 1), c.get("layers", 1), c.get("hidden", HIDDEN)
    pasts = _pasts(c, seed)
    s = {"c": c, "max_len": max(pasts) + new}
    cap = -(-(s["max_len"] + 64) // 64) * 64
    s["pos"] = torch.tensor(pasts, dtype=torch.int32, device="cuda")
    s["ctx"] = nw.AttnContext(H, KV, cap, head_dim=D, max_batch=B, q_dtype=t, o_dtype=t, kv_dtype=t)

    def cache():
        k = rnd(B, KV, cap, D, dtype="f16")
        if c.get("outliers"):
            u = torch.rand(k.shape, generator=g, device="cuda", dtype=torch.float16)
            k = torch.where(u < 0.005, -8.0, torch.where(u > 0.995, 8.0, k)).half()
        return k

    s["k"], s["v"] = [cache() for _ in range(layers)], [cache() for _ in range(layers)]
    s["out"] = torch.empty((B, new, H, D), device="cuda", dtype=_T[t])
    if c["kind"] in ("step", "prefill"):
        s["q"] = rnd(B, new, H, D, dtype=t)
        s["k_new"], s["v_new"] = rnd(B, new, KV, D, dtype=t), rnd(B, new, KV, D, dtype=t)
        return s
    s["x"], s["h"] = rnd(B * new, hidden), rnd(B * new, hidden)
    s["weights"] = [{"q": _q4(g, H * D, hidden), "k": _q4(g, KV * D, hidden),
                     "v": _q4(g, KV * D, hidden), "o": _q4(g, hidden, H * D)}
                    for _ in range(layers)]
    s["q"] = torch.empty((B, new, H, D), device="cuda", dtype=_T[t])
    if c["kind"] == "chunk":
        s["k_new"] = torch.empty((new, KV, D), device="cuda")
        s["v_new"] = torch.empty((new, KV, D), device="cuda")
    else:
        # o_proj reads f32 rows: with f16 attention outputs the program
        # widens them
        s["wide"] = s["out"] if t == "f32" else torch.empty((B, new, H, D), device="cuda")
    return s


# --------------------------------------------------------------------- pass

def run(s):
    c, ctx = s["c"], s["ctx"]
    kind = c["kind"]
    if kind == "head":
        ctx.lm_head_argmax(s["x"], s["w"]["w"], s["token"], s["logits"], c["batch"])
        return {"logits": s["logits"], "token": s["token"]}
    B, pos, n = c["batch"], s["pos"], s["max_len"]
    k, v = s["k"][0], s["v"][0]
    if kind == "step":
        if c.get("calls", 1) == 2:
            ctx.kv_append(s["k_new"], s["v_new"], k, v, pos, B)
            ctx.decode(s["q"], k, v, pos, s["out"], B, n)
        else:
            ctx.append_decode(s["q"], s["k_new"], s["v_new"], k, v, pos, s["out"], B, n)
        return {"out": s["out"], "k": k, "v": v}
    if kind == "prefill":
        ctx.kv_append(s["k_new"], s["v_new"], k, v, pos, B, c["new"])
        ctx.prefill(s["q"], k, v, pos, s["out"], B, c["new"], n)
        return {"out": s["out"], "k": k, "v": v}
    if kind == "chunk":
        w, new = s["weights"][0], c["new"]
        ctx.q4_gemv(s["x"], w["q"]["w"], s["q"], new)
        ctx.q4_gemv(s["x"], w["k"]["w"], s["k_new"], new)
        ctx.q4_gemv(s["x"], w["v"]["w"], s["v_new"], new)
        ctx.kv_append(s["k_new"], s["v_new"], k, v, pos, 1, new)
        ctx.prefill(s["q"], k, v, pos, s["out"], 1, new, n)
        ctx.q4_gemv(s["out"], w["o"]["w"], s["h"], new, nw.NWD_Q4_ACCUMULATE)
        return {"h": s["h"], "q": s["q"], "out": s["out"], "k": k, "v": v}
    for w, k, v in zip(s["weights"], s["k"], s["v"]):
        ctx.qkv_append(s["x"], w["q"]["w"], w["k"]["w"], w["v"]["w"], s["q"], k, v, pos, B)
        ctx.decode(s["q"], k, v, pos, s["out"], B, n)
        if s["wide"] is not s["out"]:
            s["wide"].copy_(s["out"])
        ctx.q4_gemv(s["wide"], w["o"]["w"], s["h"], B, nw.NWD_Q4_ACCUMULATE)
    return {"h": s["h"], "q": s["q"], "out": s["out"], "k": s["k"], "v": s["v"]}


# ------------------------------------------------- what a pass cannot do without

def work(case):
    c = case

    def q4_bytes(n, k):
        return n * k // 32 * 20.5  # per 32 weights: quant 16, scale 4, zero point 1/2

    if c["kind"] == "head":
        n, k, b = c["vocab"], c["hidden"], c["batch"]
        return {"bytes": q4_bytes(n, k) + 4 * b * (n + k + 1), "flops": 2.0 * b * n * k}
    B, H, KV, D = c["batch"], c["heads"], c["kv"], c["dim"]
    e = 2 if c["dtype"] == "f16" else 4
    new, layers, hidden = c.get("new", 1), c.get("layers", 1), c.get("hidden", HIDDEN)
    # ragged lengths by their mean, which is what a seed's draw is near
    past = (c["past"] + c["past_min"]) / 2
    keys = B * (past + new)                          # K/V rows read
    pairs = B * new * (past + (new + 1) / 2)         # (query token, key) pairs
    attn = {"bytes": keys * KV * D * 4 + B * new * (H * D * 2 * e + KV * D * 2 * (e + 2)),
            "flops": 4.0 * pairs * H * D}
    if c["kind"] in ("step", "prefill"):
        return attn
    cols = (H + 2 * KV) * D
    per = {"bytes": q4_bytes(cols, hidden) + q4_bytes(hidden, H * D) + 12 * B * new * hidden,
           "flops": 2.0 * B * new * hidden * (cols + H * D)}
    return {k: layers * (attn[k] + per[k]) for k in ("bytes", "flops")}


def tolerance(case):
    # Four times what the path shows against 64 bits, and for "max" one fp16
    # unit (2^-10 of a value) that may fall either way wherever the outputs
    # or the new K/V rows are rounded to fp16, times four. The prefill also
    # rounds its softmax weights to fp16. Tokens are the same but for ties.
    kind, t = case["kind"], case.get("dtype", "f32")
    if kind == "head":
        return {"rel": 1.5e-6, "max": 1e-5}
    if kind == "step" and t == "f32":
        return {"rel": 3e-6, "max": 3e-5}
    if kind == "token" and t == "f32":
        return {"rel": 2e-5, "max": 4e-3}
    if kind in ("step", "token"):
        return {"rel": 1e-3, "max": 4e-3}
    return {"rel": 1.5e-3, "max": 1e-2}


# ------------------------------------------------------------- in 64 bits

def _attend(q, k, v, past):
    """softmax(q k^T / sqrt(D)) v in float64: q [new][H][D], k and v
    [KV][past + new][D], query i seeing the keys 0 .. past + i."""
    new, H, D = q.shape
    KV, L = k.shape[0], k.shape[1]
    out = torch.empty((new, H, D), dtype=torch.float64, device=q.device)
    hidden = torch.arange(L, device=q.device)[None] > past + torch.arange(new, device=q.device)[:, None]
    for h in range(H):
        kh, vh = k[h * KV // H].double(), v[h * KV // H].double()
        sc = (q[:, h].double() @ kh.t()) / math.sqrt(D)
        sc.masked_fill_(hidden, -math.inf)
        out[:, h] = torch.softmax(sc, dim=-1) @ vh
    return out


def _attend_all(c, pasts, q, k, v, k_new, v_new):
    """The caches with the new rows in, and the attention outputs."""
    B, new = c["batch"], c.get("new", 1)
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for b, p in enumerate(pasts):
        k[b, :, p:p + new] = k_new[b].transpose(0, 1).half()
        v[b, :, p:p + new] = v_new[b].transpose(0, 1).half()
        out[b] = _attend(q[b], k[b, :, :p + new], v[b, :, :p + new], p)
    return out


def exact(case, seed):
    s = prepare(case, seed)
    c = s["c"]
    if c["kind"] == "head":
        y = _project(s["w"], s["x"])
        return {"logits": y, "token": None}
    B, H, KV, D, new = c["batch"], c["heads"], c["kv"], c["dim"], c.get("new", 1)
    pasts, k, v = _pasts(c, seed), s["k"], s["v"]
    if c["kind"] in ("step", "prefill"):
        out = _attend_all(c, pasts, s["q"], k[0], v[0], s["k_new"], s["v_new"])
        return {"out": out, "k": k[0], "v": v[0]}
    h = s["h"].double()
    for i, w in enumerate(s["weights"]):
        q = _project(w["q"], s["x"]).view(B, new, H, D)
        k_new = _project(w["k"], s["x"]).view(B, new, KV, D)
        v_new = _project(w["v"], s["x"]).view(B, new, KV, D)
        out = _attend_all(c, pasts, q, k[i], v[i], k_new, v_new)
        h = h + _project(w["o"], out.view(B * new, H * D))
    r = {"h": h, "q": q, "out": out}
    return dict(r, k=k[0], v=v[0]) if c["kind"] == "chunk" else dict(r, k=k, v=v)
