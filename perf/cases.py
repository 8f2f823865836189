"""The work that programs have this library do, as cases that can be timed and checked.

A case is one block of a Gemma-4-E2B-shaped decoder (or the whole decoder
engine) called through the Python front end the way a program calls it: device
buffers from g4_alloc, the library's own queue, weights loaded once.  Sizes
are the E2B configuration's (hidden 1536, 8 heads, head dims 256 and 512, MLP
6144 and 12288, a 262144-entry vocabulary, a 512-key window) and the
benchmark's, or generic ones in between.

Kinds
  linear   one W4A16 projection, any row count, FP32 or BF16 in and out
  mlp      norm, gate/up, GELU product, down, norm, residual add
  qkv      norm, q/k/v projections, their norms and RoPE
  attn     attention of a few or many query rows over the KV cache
  head     final norm, tied BF16 head, softcap, greedy pick
  ple      per-layer inputs: table gather, projection, mix
  gather   rows of the W4 per-layer-embedding table, dequantized
  tokens   a token's projections layer after layer, recorded and replayed
  prompt   the engine's prefill of a prompt, with the first logits
  turn     the engine's chat turn: a short prompt, then greedy decoding
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("gemma4-js_amd"))
import g4hip  # noqa: E402

HEADS, PLE_DIM, LAYERS, EPS = 8, 256, 35, 1e-6
VOCAB = 262144
F32, BF16 = g4hip.F32, g4hip.BF16


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # the smallest: one token's MLP, op by op, as a driver without the engine runs it
        {"name": "mlp_token", "kind": "mlp", "rows": 1, "hidden": 1536, "inter": 6144},
        # a short chat message's rows through the wide MLP
        {"name": "mlp_short", "kind": "mlp", "rows": 23, "hidden": 1536, "inter": 12288},
        # the attention inputs of an ordinary prompt, continuing a cached one
        {"name": "qkv_prompt", "kind": "qkv", "rows": 389, "hidden": 1536, "hd": 256, "pos": 100,
         "full": False},
        # the benchmark's prefill projection
        {"name": "linear_2048", "kind": "linear", "rows": 2048, "k": 1536, "n": 6144, "x": "bf16",
         "y": "f32"},
        # one token against a long conversation in a global layer
        {"name": "attn_token", "kind": "attn", "rows": 1, "hd": 512, "keys": 3001, "full": True},
        # the benchmark prompt in a sliding layer
        {"name": "attn_prompt", "kind": "attn", "rows": 512, "hd": 256, "keys": 512, "full": False},
        # the second half of a long document in a global layer
        {"name": "attn_long", "kind": "attn", "rows": 2048, "hd": 512, "keys": 4096, "full": True},
        # what follows the last layer of every step
        {"name": "head", "kind": "head", "vocab": VOCAB, "hidden": 1536},
        # what precedes the first layer of a prompt
        {"name": "ple_prompt", "kind": "ple", "rows": 301, "hidden": 1536, "vocab": VOCAB},
        # a decode step's projections through 32 layers (640 MB of weights, none cached)
        {"name": "tokens_32", "kind": "tokens", "layers": 32, "hidden": 1536, "hd": 256,
         "inter": 6144},
        # the benchmark's prefill, all 35 layers
        {"name": "prompt_512", "kind": "prompt", "layers": 35, "vocab": VOCAB, "rows": 512},
        # a chat turn on the whole model
        {"name": "turn_35", "kind": "turn", "layers": 35, "vocab": VOCAB, "rows": 37, "steps": 48},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear"] * 4 + ["mlp"] * 3 + ["qkv"] * 2 + ["attn"] * 4 +
                      ["head", "ple", "gather", "tokens", "prompt", "turn"])
    if kind == "linear":
        k, n = rng.choice([(1536, 6144), (1536, 12288), (6144, 1536), (12288, 1536), (1536, 2048),
                           (2048, 1536), (1536, 4096), (4096, 1536), (1536, 256), (256, 1536),
                           (1536, 8960), (32 * rng.randint(3, 160), rng.randint(100, 5000))])
        return {"kind": kind, "rows": _log(rng, 1, 2048), "k": k, "n": n,
                "x": rng.choice(["f32", "f32", "bf16"]), "y": rng.choice(["f32", "f32", "bf16"])}
    if kind == "mlp":
        return {"kind": kind, "rows": _log(rng, 1, 1100), "hidden": 1536,
                "inter": rng.choice([6144, 12288])}
    if kind == "qkv":
        full = rng.random() < 0.3
        return {"kind": kind, "rows": _log(rng, 1, 1100), "hidden": 1536, "hd": 512 if full else 256,
                "pos": rng.randint(0, 900), "full": full}
    if kind == "attn":
        full = rng.random() < 0.5
        rows = rng.choice([1, _log(rng, 2, 1500)])
        keys = rows + rng.choice([0, _log(rng, 1, 2500)])
        return {"kind": kind, "rows": rows, "hd": 512 if full else 256, "keys": keys, "full": full}
    if kind == "head":
        return {"kind": kind, "vocab": _log(rng, 8000, VOCAB), "hidden": 1536}
    if kind == "ple":
        return {"kind": kind, "rows": _log(rng, 1, 1100), "hidden": 1536, "vocab": 32768}
    if kind == "gather":
        return {"kind": kind, "rows": _log(rng, 1, 4096), "vocab": 65536,
                "y": rng.choice(["f32", "bf16"])}
    if kind == "tokens":
        return {"kind": kind, "layers": rng.randint(8, 30), "hidden": 1536,
                "hd": rng.choice([256, 512]), "inter": rng.choice([6144, 12288])}
    if kind == "prompt":
        return {"kind": kind, "layers": rng.randint(16, 30), "vocab": 32768, "rows": _log(rng, 5, 600)}
    return {"kind": kind, "layers": rng.randint(16, 30), "vocab": 32768, "rows": _log(rng, 2, 200),
            "steps": rng.randint(8, 40)}


# ---- inputs ------------------------------------------------------------------

class _Seen:
    """A g4hip.Buffer as torch sees device memory; keeps the buffer alive."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr,
                                         "data": (buf.ptr, False), "version": 2}


def _view(buf, shape, dtype=torch.float32):
    """A torch tensor over the whole of a device buffer (no copy)."""
    code = {torch.float32: "<f4", torch.int32: "<i4", torch.bfloat16: "<i2"}[dtype]
    t = torch.as_tensor(_Seen(buf, shape, code), device="cuda")
    return t.view(torch.bfloat16) if dtype == torch.bfloat16 else t


def _buffer(t):
    """A device buffer holding tensor t."""
    t = t.contiguous()
    b = g4hip.Buffer(t.numel() * t.element_size())
    g4hip.sync()  # g4_alloc zero-fills on the library's queue
    _view(b, t.shape, t.dtype).copy_(t)
    torch.cuda.synchronize()
    return b


class _Out:
    """An output buffer and the tensor over it."""

    def __init__(self, *shape, dtype=torch.float32):
        n = int(np.prod(shape))
        self.buf = g4hip.Buffer(n * (2 if dtype == torch.bfloat16 else 4))
        self.t = _view(self.buf, shape, dtype)
        self.ptr = self.buf.ptr


def _gen(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _normal(g, *shape, sigma=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * sigma


def _weight(g, n, k):
    """Checkpoint bytes of a W4A16 weight: offset nibbles of q in [-7, 7] and
    BF16 |N(0,1)| * 0.02 scales, the benchmark's distributions."""
    p = torch.randint(0, 225, (n, k // 2), generator=g, device="cuda", dtype=torch.uint8)
    packed = (p % 15 + 1) | ((p // 15 + 1) << 4)
    scales = (torch.randn(n, k // 32, generator=g, device="cuda").abs() * 0.02).bfloat16()
    return packed, scales


def _load(pair):
    packed, scales = pair
    n, k = packed.shape[0], packed.shape[1] * 2
    torch.cuda.synchronize()
    h = g4hip._vp()
    g4hip.check(g4hip.lib().g4_w4_load_dev(packed.data_ptr(), scales.data_ptr(), n, k, 32,
                                           g4hip._c.byref(h)))
    return g4hip.W4Linear._from_handle(h.value, n, k)


def _norm_weight(g, n, at=1.0):
    return (torch.rand(n, generator=g, device="cuda") * 0.2 + 0.9) * at


def _ple_bytes(g, vocab, width):
    """(packed uint8 [vocab, width/2], scales bf16 [vocab, width/32]) of a
    per-layer-embedding table: two's-complement q in [-7, 7]."""
    p = torch.randint(0, 225, (vocab, width // 2), generator=g, device="cuda", dtype=torch.uint8)
    p = (((p % 15).to(torch.int8) - 7) & 15).to(torch.uint8) | \
        ((((p // 15).to(torch.int8) - 7) & 15) << 4).to(torch.uint8)
    s = (torch.randn(vocab, width // 32, generator=g, device="cuda").abs() * 0.05).bfloat16()
    return p, s


def _ple_table(packed, scales, width, per=4096):
    vocab = packed.shape[0]
    t = g4hip.PleTable(vocab, width, 32, per)
    for s in range(t.num_shards):
        a, b = s * per, min(vocab, (s + 1) * per)
        shard = torch.cat([packed[a:b].reshape(-1), scales[a:b].reshape(-1).view(torch.uint8)])
        torch.cuda.synchronize()
        g4hip.check(g4hip.lib().g4_ple_upload_shard_dev(t.h, s, shard.data_ptr(), shard.numel()))
        g4hip.sync()
    return t


def _ids(g, n, vocab):
    return torch.randint(0, vocab, (n,), generator=g, device="cuda", dtype=torch.int32)


def _rows_of(case, g):
    """The inputs of every kind but the engine's, as tensors, made from the seed alone."""
    kind = case["kind"]
    if kind == "linear":
        x = _normal(g, case["rows"], case["k"])
        return {"w": _weight(g, case["n"], case["k"]),
                "x": x.bfloat16() if case["x"] == "bf16" else x}
    h = case.get("hidden")
    if kind == "mlp":
        return {"gate": _weight(g, case["inter"], h), "up": _weight(g, case["inter"], h),
                "down": _weight(g, h, case["inter"]), "pre": _norm_weight(g, h),
                "post": _norm_weight(g, h), "x": _normal(g, case["rows"], h)}
    if kind == "qkv":
        hd = case["hd"]
        return {"q": _weight(g, HEADS * hd, h), "k": _weight(g, hd, h), "v": _weight(g, hd, h),
                "pre": _norm_weight(g, h), "qn": _norm_weight(g, hd), "kn": _norm_weight(g, hd),
                "x": _normal(g, case["rows"], h)}
    if kind == "attn":
        # normed rows: q.k of a few units, as trained q/k norm weights leave it
        hd = case["hd"]
        at = 1.5 / math.sqrt(math.sqrt(hd))
        return {"q": _normal(g, case["rows"], HEADS, hd, sigma=at),
                "k": _normal(g, case["keys"], hd, sigma=at), "v": _normal(g, case["keys"], hd)}
    if kind == "head":
        return {"E": _normal(g, case["vocab"], h, sigma=0.03).bfloat16(),
                "norm": _norm_weight(g, h), "x": _normal(g, 1, h)}
    if kind in ("ple", "gather"):
        packed, scales = _ple_bytes(g, case["vocab"], LAYERS * PLE_DIM)
        s = {"packed": packed, "scales": scales, "ids": _ids(g, case["rows"], case["vocab"])}
        if kind == "ple":
            s.update(E=_normal(g, case["vocab"], h, sigma=0.03).bfloat16(),
                     top=_weight(g, LAYERS * PLE_DIM, h), norm=_norm_weight(g, PLE_DIM))
        return s
    assert kind == "tokens"
    hd = case["hd"]
    s = {"x": _normal(g, 1, h), "ctx": _normal(g, 1, HEADS * hd), "act": _normal(g, 1, case["inter"])}
    for i in range(case["layers"]):
        for name, n, k in (("q", HEADS * hd, h), ("k", hd, h), ("v", hd, h), ("o", h, HEADS * hd),
                           ("gate", case["inter"], h), ("up", case["inter"], h),
                           ("down", h, case["inter"])):
            s["%s%d" % (name, i)] = _weight(g, n, k)
    return s


def _schedule(case):
    """The engine configuration: E2B's layers, the first `layers` of them (16 or
    more, so layers that reuse an earlier cache are among them)."""
    cfg = g4hip.e2b_config(1024)
    cfg.layers = case["layers"]
    cfg.vocab = case["vocab"]
    return cfg


def _engine_inputs(case, g):
    """Random weights of the E2B shapes.  q and k norm weights near 0.3 keep
    q.k within a few units (there is no 1/sqrt(head_dim)); the token rows
    differ in length, so the best logit stands clear of the others, as in a
    trained model."""
    cfg = _schedule(case)
    H, V, NL = cfg.hidden, cfg.vocab, cfg.layers
    E = _normal(g, V, H, sigma=0.03)
    E = (E * torch.exp(0.3 * torch.randn(V, 1, generator=g, device="cuda"))).bfloat16()
    packed, scales = _ple_bytes(g, V, NL * PLE_DIM)
    s = {"E": E, "ple": (packed, scales), "top": _weight(g, NL * PLE_DIM, H),
         "ple_norm": _norm_weight(g, PLE_DIM), "final": _norm_weight(g, H), "layers": []}
    for i in range(NL):
        hd, inter = cfg.head_dim[i], cfg.intermediate[i]
        own = cfg.kv_source[i] < 0
        shapes = [("q", HEADS * hd, H)] + ([("k", hd, H), ("v", hd, H)] if own else []) + [
            ("o", H, HEADS * hd), ("gate", inter, H), ("up", inter, H), ("down", H, inter),
            ("ple_gate", PLE_DIM, H), ("ple_proj", H, PLE_DIM)]
        norms = {n: _norm_weight(g, H)
                 for n in ("input", "post_attn", "pre_ffw", "post_ffw", "post_ple")}
        norms["q"] = _norm_weight(g, hd, 0.3)
        if own:
            norms["k"] = _norm_weight(g, hd, 0.3)
        s["layers"].append({"linear": {n: _weight(g, a, b) for n, a, b in shapes}, "norm": norms})
    s["ids"] = _ids(g, case["rows"], V)
    return cfg, s


def _engine(cfg, s):
    m = g4hip.Gemma(cfg)
    m.set_embedding(_buffer(s["E"]))
    m.set_ple(_ple_table(*s["ple"], cfg.layers * PLE_DIM))
    m.set_linear(-1, "top", _load(s["top"]))
    m.set_norm(-1, "ple_projection", s["ple_norm"].cpu().numpy())
    m.set_norm(-1, "final", s["final"].cpu().numpy())
    for i, layer in enumerate(s["layers"]):
        for n, w in layer["linear"].items():
            m.set_linear(i, n, _load(w))
        for n, v in layer["norm"].items():
            m.set_norm(i, n, v.cpu().numpy())
        m.set_layer_scalar(i, 1.0)
    return m


def prepare(case, seed):
    g4hip.init(0)
    g = _gen(case, seed)
    kind = case["kind"]
    if kind in ("prompt", "turn"):
        cfg, s = _engine_inputs(case, g)
        st = {"case": case, "m": _engine(cfg, s), "ids": s["ids"].cpu().numpy(),
              "logits": _Out(cfg.vocab), "last": _Out(cfg.hidden)}
        if kind == "turn":
            st["next"] = _Out(cfg.vocab)
        g4hip.sync()
        return st
    s = _rows_of(case, g)
    st = {"case": case}
    for n, v in s.items():
        if isinstance(v, tuple):
            st[n] = _load(v)
        elif n == "packed":
            st["table"] = _ple_table(v, s["scales"], LAYERS * PLE_DIM)
        elif n != "scales":
            st[n] = _buffer(v)
    if kind in ("ple", "gather"):  # the program has its ids on the host
        st["host_ids"] = s["ids"].cpu().numpy()
    r, h = case.get("rows", 1), case.get("hidden")
    if kind == "linear":
        st["y"] = _Out(r, case["n"], dtype=torch.bfloat16 if case["y"] == "bf16" else torch.float32)
    elif kind == "mlp":
        for n, w in (("pf", h), ("g", case["inter"]), ("u", case["inter"]), ("a", case["inter"]),
                     ("d", h), ("dn", h), ("y", h)):
            st[n] = _Out(r, w)
    elif kind == "qkv":
        hd = case["hd"]
        st["pf"] = _Out(r, h)
        for n, w in (("qr", HEADS * hd), ("kr", hd), ("vr", hd), ("qy", HEADS * hd), ("ky", hd),
                     ("vy", hd)):
            st[n] = _Out(r, w)
    elif kind == "attn":
        st["y"] = _Out(r, HEADS, case["hd"])
    elif kind == "head":
        st["hn"], st["logits"] = _Out(h), _Out(case["vocab"])
        st["token"] = _Out(1, dtype=torch.int32)
    elif kind == "ple":
        w = LAYERS * PLE_DIM
        st["hid"], st["tok"], st["proj"], st["projs"], st["y"] = (
            _Out(r, h), _Out(r, w), _Out(r, w), _Out(r, w), _Out(r, w))
    elif kind == "gather":
        st["y"] = _Out(r, LAYERS * PLE_DIM,
                       dtype=torch.bfloat16 if case["y"] == "bf16" else torch.float32)
    elif kind == "tokens":
        _prepare_tokens(st, case)
    g4hip.sync()
    return st


def _prepare_tokens(st, case):
    """The recording that a decode loop replays: four launches a layer."""
    hd, h, inter = case["hd"], case["hidden"], case["inter"]
    width = {"q": HEADS * hd, "k": hd, "v": hd, "o": h, "gate": inter, "up": inter, "down": h}
    st["y"] = {n: _Out(case["layers"], w) for n, w in width.items()}

    def layer(i):
        def out(n):
            return st["y"][n].ptr + 4 * i * width[n]

        def w(n):
            return st["%s%d" % (n, i)]

        g4hip.W4Linear.linear_multi([w("q"), w("k"), w("v")], st["x"].ptr, F32, 1,
                                    [out("q"), out("k"), out("v")])
        w("o").linear(st["ctx"].ptr, F32, 1, out("o"))
        g4hip.W4Linear.linear_multi([w("gate"), w("up")], st["x"].ptr, F32, 1,
                                    [out("gate"), out("up")])
        w("down").linear(st["act"].ptr, F32, 1, out("down"))

    with g4hip.Encoder() as enc:
        for i in range(case["layers"]):
            layer(i)
    st["record"] = enc.cmdbuf


# ---- one pass ------------------------------------------------------------------

def run(st):
    case = st["case"]
    kind, r, h = case["kind"], case.get("rows", 1), case.get("hidden")
    if kind == "linear":
        st["w"].linear(st["x"].ptr, BF16 if case["x"] == "bf16" else F32, r, st["y"].ptr,
                       BF16 if case["y"] == "bf16" else F32)
        return st["y"].t
    if kind == "mlp":
        n = r * case["inter"]
        g4hip.rms(st["x"], r, h, st["pre"], st["pf"], EPS)
        g4hip.W4Linear.linear_multi([st["gate"], st["up"]], st["pf"].ptr, F32, r,
                                    [st["g"].ptr, st["u"].ptr])
        g4hip.gelu_mul(st["g"], st["u"], n, st["a"])
        st["down"].linear(st["a"].ptr, F32, r, st["d"].ptr)
        g4hip.rms(st["d"], r, h, st["post"], st["dn"], EPS)
        g4hip.add_scale(st["x"], st["dn"], r * h, 1.0, st["y"])
        return {"act": st["a"].t, "y": st["y"].t}
    if kind == "qkv":
        hd, pos = case["hd"], case["pos"]
        base, angles = _rope_of(case)
        g4hip.rms(st["x"], r, h, st["pre"], st["pf"], EPS)
        g4hip.W4Linear.linear_multi([st["q"], st["k"], st["v"]], st["pf"].ptr, F32, r,
                                    [st["qr"].ptr, st["kr"].ptr, st["vr"].ptr])
        g4hip.norm_rope(st["qr"], r, HEADS, hd, pos, st["qn"], angles, base, st["qy"], EPS)
        g4hip.norm_rope(st["kr"], r, 1, hd, pos, st["kn"], angles, base, st["ky"], EPS)
        g4hip.rms(st["vr"], r, hd, None, st["vy"], EPS)
        return {"q": st["qy"].t, "k": st["ky"].t, "v": st["vy"].t}
    if kind == "attn":
        keys = case["keys"]
        g4hip.attention(st["q"], st["k"], st["v"], r, HEADS, case["hd"], keys, keys - r,
                        not case["full"], 512, st["y"])
        return st["y"].t
    if kind == "head":
        g4hip.rms(st["x"], 1, h, st["norm"], st["hn"], EPS)
        g4hip.bf16_head(st["hn"].ptr, st["E"].ptr, case["vocab"], h, st["logits"].ptr, 1.0, 30.0)
        g4hip.argmax(st["logits"], case["vocab"], st["token"])
        return {"logits": st["logits"].t, "token": st["token"].t}
    if kind == "ple":
        w = LAYERS * PLE_DIM
        g4hip.embed(st["E"], case["vocab"], h, st["ids"], r, math.sqrt(h), st["hid"])
        st["table"].gather(st["host_ids"], st["tok"].ptr)
        st["top"].linear(st["hid"].ptr, F32, r, st["proj"].ptr)
        g4hip.scale(st["proj"], r * w, 1.0 / math.sqrt(h), st["projs"])
        g4hip.ple_mix(st["projs"], st["norm"], st["tok"], r, PLE_DIM, LAYERS, st["y"])
        return {"hidden": st["hid"].t, "y": st["y"].t}
    if kind == "gather":
        st["table"].gather(st["host_ids"], st["y"].ptr, BF16 if case["y"] == "bf16" else F32)
        return st["y"].t
    if kind == "tokens":
        st["record"].submit()
        return {n: o.t for n, o in st["y"].items()}
    m = st["m"]
    m.reset()
    first = m.greedy(st["ids"], 0, st["logits"])
    if kind == "prompt":
        m.last_hidden(st["last"])
        return {"logits": st["logits"].t, "last": st["last"].t, "token": first}
    tokens = m.decode(case["steps"])
    m.last_hidden(st["last"])
    m.logits(st["last"], st["next"])
    return {"logits": st["logits"].t, "last": st["last"].t, "next": st["next"].t, "tokens": tokens}


def _rope_of(case):
    return (1e6, case["hd"] // 8) if case["full"] else (1e4, case["hd"] // 2)


# ---- the work that a pass cannot do without ------------------------------------

def _w4(n, k):
    return n * k // 2 + n * (k // 32) * 2


def _pairs(rows, keys, full):
    """Visible (query, key) pairs and the span of visible keys."""
    p = np.arange(keys - rows, keys, dtype=np.int64) + 1
    seen = p if full else np.minimum(p, 512)
    first = 0 if full else max(0, keys - rows + 1 - 512)
    return int(seen.sum()), keys - first


def work(case):
    kind, r, h = case["kind"], case.get("rows", 1), case.get("hidden")
    w = LAYERS * PLE_DIM
    if kind == "linear":
        size = {"f32": 4, "bf16": 2}
        n, k = case["n"], case["k"]
        return {"bytes": _w4(n, k) + r * (k * size[case["x"]] + n * size[case["y"]]),
                "flops": 2 * r * n * k}
    if kind == "mlp":
        i = case["inter"]
        return {"bytes": 3 * _w4(i, h) + 4 * (2 * r * h + r * i + 2 * h), "flops": 6 * r * h * i}
    if kind == "qkv":
        n = (HEADS + 2) * case["hd"]
        return {"bytes": _w4(n, h) + 4 * r * (h + n), "flops": 2 * r * n * h}
    if kind == "attn":
        pairs, span = _pairs(r, case["keys"], case["full"])
        return {"bytes": 4 * case["hd"] * (2 * r * HEADS + 2 * span),
                "flops": 4 * case["hd"] * HEADS * pairs}
    if kind == "head":
        return {"bytes": 2 * case["vocab"] * h + 4 * (case["vocab"] + h),
                "flops": 2 * case["vocab"] * h}
    if kind == "ple":
        return {"bytes": r * (w // 2 + w // 16) + _w4(w, h) + r * (2 * h + 4 * h + 4 * w),
                "flops": 2 * r * w * h}
    if kind == "gather":
        return {"bytes": r * (w // 2 + w // 16 + 4 + w * (2 if case["y"] == "bf16" else 4)),
                "flops": 0}
    if kind == "tokens":
        hd, i = case["hd"], case["inter"]
        n = (_w4((HEADS + 2) * hd, h) + _w4(h, HEADS * hd) + 3 * _w4(i, h))
        return {"bytes": case["layers"] * n, "flops": case["layers"] * n * 32 // 9}
    H, NL, V = 1536, case["layers"], case["vocab"]
    spec = [((512, True) if (i + 1) % 5 == 0 else (256, False)) + (6144 if i < 15 else 12288,)
            for i in range(NL)]
    elems = NL * PLE_DIM * H
    for i, (hd, full, inter) in enumerate(spec):
        elems += H * (2 * HEADS * hd + 3 * inter + 2 * PLE_DIM + (2 * hd if i < 15 else 0))

    def pass_of(rows, keys):
        b = elems * 9 // 16 + 2 * V * H + 4 * V
        f = 2 * rows * elems + 2 * V * H
        for hd, full, _ in spec:
            pairs, span = _pairs(rows, keys, full)
            b += 8 * span * hd
            f += 4 * hd * HEADS * pairs
        return b, f

    b, f = pass_of(r, r)
    for s in range(case.get("steps", 0)):
        db, df = pass_of(1, r + 1 + s)
        b, f = b + db, f + df
    return {"bytes": b, "flops": f}


# ---- how far another correct implementation may be off -------------------------

# About four times the largest error against 64 bits that was measured over the
# ranges.  One-row FP32 projections take x as two BF16 parts (4e-6 each, 7e-6 after
# a GELU product); the matrix-core ones take two FP16 parts (5e-7).

def tolerance(case):
    kind = case["kind"]
    if kind == "gather":
        return "exact"  # a table value times its scale, rounded once
    if kind == "linear" and case["y"] == "bf16":
        return {"rel": 6e-3}
    if kind in ("linear", "mlp", "ple"):
        return {"rel": 3e-5 if case["rows"] <= 4 else 2e-6}
    if kind in ("qkv", "tokens"):
        return {"rel": 3e-5}  # qkv: and 32-bit RoPE angles
    if kind == "attn":
        return {"rel": 3e-6}
    if kind == "head":
        return {"rel": 5e-7}
    return {"rel": 1e-4}  # 16 to 35 layers deep


# ---- the same in 64 bits ---------------------------------------------------------

def _dense(pair):
    packed, scales = pair
    n, kb = packed.shape
    q = torch.stack([packed & 15, packed >> 4], -1).reshape(n, kb * 2).double() - 8.0
    return (q.view(n, -1, 32) * scales.double()[:, :, None]).reshape(n, kb * 2)


def _rms(x, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _gelu(x):
    z = 0.7978845608028654 * (x + 0.044715 * x ** 3)
    return 0.5 * x * (1.0 + torch.tanh(z.clamp(-10.0, 10.0)))


def _rope(x, pos, base, angles):
    """Rotate-half RoPE of the first `angles` pairs; x [rows, heads, hd]."""
    rows, _, hd = x.shape
    half = hd // 2
    p = torch.arange(half, device=x.device, dtype=torch.float64)
    th = torch.arange(pos, pos + rows, device=x.device, dtype=torch.float64)[:, None] / \
        torch.pow(torch.tensor(base, dtype=torch.float64, device=x.device), 2 * p / hd)
    th[:, angles:] = 0.0
    c, s = torch.cos(th)[:, None, :], torch.sin(th)[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, k, v, pos, full):
    """q [rows, heads, hd] at positions pos.., k/v [keys, hd] from position 0."""
    rows, keys = q.shape[0], k.shape[0]
    at = torch.arange(pos, pos + rows, device=q.device)[:, None]
    key = torch.arange(keys, device=q.device)[None, :]
    hide = key > at
    if not full:
        hide = hide | (key + 512 <= at)
    out = []
    for i in range(q.shape[1]):
        s = (q[:, i, :] @ k.T).masked_fill(hide, -math.inf)
        out.append(torch.softmax(s, -1) @ v)
    return torch.stack(out, 1)


def _ple_rows(packed, scales, ids):
    p = packed[ids.long()]
    q = torch.stack([p & 15, p >> 4], -1).reshape(p.shape[0], -1).double()
    q = torch.where(q > 7, q - 16, q)
    return (q.view(p.shape[0], -1, 32) * scales[ids.long()].double()[:, :, None]).reshape(p.shape[0], -1)


def _ple_inputs(E, packed, scales, top, norm, ids, layers):
    """The scaled embedding rows and the per-layer inputs [rows, layers, PLE_DIM]."""
    h = E.shape[1]
    hid = E[ids.long()].double() * float(np.float32(math.sqrt(h)))
    proj = (hid @ top.T / math.sqrt(h)).view(len(ids), layers, PLE_DIM)
    tok = _ple_rows(packed, scales, ids).view(len(ids), layers, PLE_DIM)
    return hid, (_rms(proj, norm) + tok * 16.0) * 0.7071067811865476


def exact(case, seed):
    g = _gen(case, seed)
    kind = case["kind"]
    if kind in ("prompt", "turn"):
        return _exact_engine(case, g)
    s = _rows_of(case, g)
    if kind == "linear":
        return s["x"].double() @ _dense(s["w"]).T
    if kind == "mlp":
        x = s["x"].double()
        pf = _rms(x, s["pre"])
        act = _gelu(pf @ _dense(s["gate"]).T) * (pf @ _dense(s["up"]).T)
        return {"act": act, "y": x + _rms(act @ _dense(s["down"]).T, s["post"])}
    if kind == "qkv":
        r, hd = case["rows"], case["hd"]
        base, angles = _rope_of(case)
        pf = _rms(s["x"].double(), s["pre"])
        q = _rms((pf @ _dense(s["q"]).T).view(r, HEADS, hd), s["qn"])
        k = _rms((pf @ _dense(s["k"]).T).view(r, 1, hd), s["kn"])
        return {"q": _rope(q, case["pos"], base, angles).reshape(r, -1),
                "k": _rope(k, case["pos"], base, angles).reshape(r, -1),
                "v": _rms(pf @ _dense(s["v"]).T)}
    if kind == "attn":
        return _attend(s["q"].double(), s["k"].double(), s["v"].double(),
                       case["keys"] - case["rows"], case["full"])
    if kind == "head":
        x = _rms(s["x"].double(), s["norm"])[0]
        logits = 30.0 * torch.tanh(s["E"].double() @ x / 30.0)
        return {"logits": logits, "token": None}
    if kind == "ple":
        hid, y = _ple_inputs(s["E"], s["packed"], s["scales"], _dense(s["top"]), s["norm"],
                             s["ids"], LAYERS)
        return {"hidden": hid, "y": y.reshape(len(s["ids"]), -1)}
    if kind == "gather":
        return _ple_rows(s["packed"], s["scales"], s["ids"])
    src = {n: s["x"] for n in ("q", "k", "v", "gate", "up")}
    src.update(o=s["ctx"], down=s["act"])
    return {n: torch.stack([_dense(s["%s%d" % (n, i)]) @ x.double()[0]
                            for i in range(case["layers"])]) for n, x in src.items()}


def _exact_engine(case, g):
    cfg, s = _engine_inputs(case, g)
    H, NL = cfg.hidden, cfg.layers
    top = _dense(s["top"])
    dense = [{n: _dense(w) for n, w in layer["linear"].items()} for layer in s["layers"]]
    cache = {}

    def forward(ids, pos):
        hid, ple = _ple_inputs(s["E"], *s["ple"], top, s["ple_norm"], ids, NL)
        r = len(ids)
        for i in range(NL):
            w, n = dense[i], s["layers"][i]["norm"]
            hd, full, src = cfg.head_dim[i], bool(cfg.full[i]), cfg.kv_source[i]
            base, angles = (1e6, hd // 8) if full else (1e4, hd // 2)
            pre = _rms(hid, n["input"])
            q = _rope(_rms((pre @ w["q"].T).view(r, HEADS, hd), n["q"]), pos, base, angles)
            if src < 0:
                src = i
                k = _rope(_rms((pre @ w["k"].T).view(r, 1, hd), n["k"]), pos, base, angles)[:, 0]
                v = _rms(pre @ w["v"].T)
                old = cache.get(i)
                cache[i] = (k, v) if old is None else tuple(torch.cat(t) for t in zip(old, (k, v)))
            ctx = _attend(q, *cache[src], pos, full).reshape(r, -1)
            hid = hid + _rms(ctx @ w["o"].T, n["post_attn"])
            pf = _rms(hid, n["pre_ffw"])
            act = _gelu(pf @ w["gate"].T) * (pf @ w["up"].T)
            hid = hid + _rms(act @ w["down"].T, n["post_ffw"])
            pm = _gelu(hid @ w["ple_gate"].T) * ple[:, i]
            hid = hid + _rms(pm @ w["ple_proj"].T, n["post_ple"])
        return _rms(hid[-1], s["final"])

    E = s["E"].double()

    def logits_of(last):
        return 30.0 * torch.tanh(E @ last / 30.0)

    ids = s["ids"]
    last = forward(ids, 0)
    first = logits_of(last)
    if case["kind"] == "prompt":
        return {"logits": first, "last": last, "token": None}
    logits = first
    for step in range(case["steps"]):
        last = forward(logits.argmax().reshape(1), case["rows"] + step)
        logits = logits_of(last)
    return {"logits": first, "last": last, "next": logits, "tokens": None}
