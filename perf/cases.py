"""The work that programs have this library do, as measurable cases.

Every case goes through the public Python entry points (flock_amd.ops,
flock_amd.decoder, flock_amd.model) on device arrays, the way a serving loop
calls them: one attention layer of a decode step, a ragged batch, a prompt or
a chunk onto a long cache; one whole decoder layer over a chunk or a prompt;
the LM head; and a whole model's decode step replayed from a captured graph.
Shapes are the ones of the repository's benchmark and tests (Qwen3-0.6B: 16
query heads, 8 kv heads, head_dim 128, hidden 1024, ffn 3072, vocabulary
151936) and, for the sweeps, kv heads 1 to 8, groups 1 to 8, head_dim 64 and 128.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from flock_amd import ops
from flock_amd.decoder import DecoderConfig, DecoderLayer
from flock_amd.model import Model

EPS = 9.999999974752427e-7   # the layer configuration's default
ROPE_BASE = 1e6
VOCAB = 151936
QWEN = {"heads": 16, "kv_heads": 8, "head_dim": 128, "pairing": "neox"}
SMALL = {"heads": 32, "kv_heads": 8, "head_dim": 64, "pairing": "norm"}


def listed():
    return [
        # One attention layer of a decode step early in a chat: 513 keys, the
        # call a token makes 28 times, bound by launches and latency.
        {"name": "decode-513", "kind": "decode", **QWEN, "keys": 513},
        # The same step a few pages in, with head_dim 64, groups of four and
        # the adjacent-pair rotation.
        {"name": "decode-4097-d64", "kind": "decode", **SMALL, "keys": 4097},
        # ... and on a full 32k context, where the cache has to be streamed.
        {"name": "decode-32769", "kind": "decode", **QWEN, "keys": 32769},
        # A serving step: 64 sequences of 1025 to 16385 keys in one call.
        {"name": "ragged-64", "kind": "ragged", **QWEN, "seqs": 64, "low": 1025, "high": 16385,
         "lengths": 3},
        # An odd chunk in the middle of a document, head_dim 64.
        {"name": "chunk-777-at-1000-d64", "kind": "prefill", **SMALL, "tokens": 777, "pos0": 1000},
        # A prompt of ordinary length.
        {"name": "prefill-2048", "kind": "prefill", **QWEN, "tokens": 2048, "pos0": 0},
        # A 64-token replay chunk onto a full context.
        {"name": "chunk-64-at-32768", "kind": "prefill", **QWEN, "tokens": 64, "pos0": 32768},
        # A long prompt.
        {"name": "prefill-8192", "kind": "prefill", **QWEN, "tokens": 8192, "pos0": 0},
        # The head after the last layer: norm, 151936 x 1024 projection, argmax.
        {"name": "lm-head", "kind": "head", "rows": VOCAB, "hidden": 1024},
        # One whole layer over a 64-token replay chunk onto 448 keys.
        {"name": "layer-chunk-64", "kind": "layer", "tokens": 64, "pos0": 448},
        # One whole layer over a 2048-token prompt.
        {"name": "layer-prefill-2048", "kind": "layer", "tokens": 2048, "pos0": 0},
        # A token of the whole 28-layer model at 513 keys, from a captured graph.
        {"name": "model-token-513", "kind": "model", "layers": 28, "keys": 513, "vocab": VOCAB},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng):
    """Half the time the benchmark's heads, else any of the supported ones."""
    if rng.random() < 0.5:
        return dict(QWEN)
    kv = rng.choice((1, 2, 3, 4, 5, 8))
    return {"heads": kv * rng.randint(1, 8), "kv_heads": kv, "head_dim": rng.choice((64, 128)),
            "pairing": rng.choice(("neox", "norm"))}


def draw(rng):
    kind = rng.choice(("decode", "decode", "ragged", "prefill", "prefill", "prefill", "head",
                       "layer", "layer", "layer", "model"))
    if kind == "decode":
        return {"kind": kind, **_shape(rng), "keys": _log_int(rng, 60, 40000)}
    if kind == "ragged":
        seqs = _log_int(rng, 2, 300)
        high = max(200, min(16385, _log_int(rng, 1000, 600000) // seqs * 2))
        return {"kind": kind, **_shape(rng), "seqs": seqs, "low": rng.randint(1, high // 2),
                "high": high, "lengths": rng.randint(0, 1 << 30)}
    if kind == "prefill":
        while True:
            c = {"kind": kind, **_shape(rng), "tokens": _log_int(rng, 9, 8192),
                 "pos0": 0 if rng.random() < 0.4 else _log_int(rng, 1, 32768)}
            if work(c)["flops"] < 2.7e11:
                return c
    if kind == "head":
        return {"kind": kind, "rows": _log_int(rng, 2000, VOCAB),
                "hidden": 32 * _log_int(rng, 8, 96) if rng.random() < 0.5 else 1024}
    if kind == "layer":
        return {"kind": kind, "tokens": _log_int(rng, 2, 2048),
                "pos0": 0 if rng.random() < 0.5 else _log_int(rng, 1, 2048)}
    return {"kind": kind, "layers": rng.choice((2, 5, 12, 28)), "keys": _log_int(rng, 60, 8000),
            "vocab": rng.choice((512, 32000, VOCAB))}


# ------------------------------------------------------------------- inputs --
class _Device:
    """A library buffer, for torch's array-interface import (kept alive by it)."""

    def __init__(self, buf, shape):
        self.buf = buf
        self.__cuda_array_interface__ = {"data": (ops.ptr(buf), False), "shape": tuple(shape),
                                         "typestr": "<f4", "version": 3, "strides": None}


def _view(buf, shape):
    """A device tensor over a library buffer's memory."""
    return torch.as_tensor(_Device(buf, shape), device="cuda")


def _randn(gen, *shape):
    return torch.randn(*shape, device="cuda", generator=gen)


def _gains(gen, n):
    return 1 + 0.1 * _randn(gen, n)


def _lengths(case):
    r = np.random.default_rng(case["lengths"])
    return r.integers(case["low"], case["high"] + 1, case["seqs"])


def _q8(rng, rows, cols, scale=8e-4):
    """Random Q8_0 blocks: an f16 scale, then 32 signed quants."""
    n = rows * cols // 32
    blocks = np.frombuffer(rng.bytes(n * 34), np.uint8).reshape(n, 34).copy()
    blocks[:, :2] = (rng.random(n, np.float32) * scale + 1e-5).astype(np.float16).view(
        np.uint8).reshape(-1, 2)
    return blocks.ravel()


LAYER_GAINS = (("attn_norm.weight", "hidden"), ("ffn_norm.weight", "hidden"),
               ("attn_q_norm.weight", "headDim"), ("attn_k_norm.weight", "headDim"))


def _layer_weights(rng, cfg):
    w = {n: _q8(rng, r, c) for n, (r, c) in cfg.shapes().items()}
    for n, field in LAYER_GAINS:
        w[n] = rng.normal(1, 0.1, getattr(cfg, field)).astype(np.float32)
    return w


def _attention_inputs(case, seed):
    """Raw q, k, v of the new tokens, gains, and a filled K/V cache."""
    H, G, d = case["heads"], case["kv_heads"], case["head_dim"]
    if case["kind"] == "decode":
        n, rows = 1, case["keys"]
    elif case["kind"] == "ragged":
        n, rows = case["seqs"], int(_lengths(case).sum())
    else:
        n, rows = case["tokens"], case["pos0"] + case["tokens"]
    gen = torch.Generator("cuda").manual_seed(seed)
    return {"q": _randn(gen, n, H, d), "k": _randn(gen, n, G, d), "v": _randn(gen, n, G, d),
            "gq": _gains(gen, d), "gk": _gains(gen, d), "kc": _randn(gen, rows, G, d),
            "vc": _randn(gen, rows, G, d),
            "inv": torch.from_numpy(_inv_freq(d)).cuda()}


def _inv_freq(d):
    return np.array([1.0 / math.pow(ROPE_BASE, 2.0 * j / d) for j in range(d // 2)], np.float32)


def _layer_config(case):
    if case["kind"] == "layer":
        return DecoderConfig(maxKeys=case["pos0"] + case["tokens"], maxPrefill=case["tokens"])
    return DecoderConfig(maxKeys=case["keys"], maxPrefill=1)


def _fill_cache(layer, rows, gen):
    """Random keys and values in the first `rows` rows of a layer's caches."""
    c = layer.cfg
    kc, vc = (_view(layer.buf[n], (c.maxKeys, c.nKvHeads, c.headDim))
              for n in ("kcache", "vcache"))
    kc.zero_(), vc.zero_()
    if rows:
        kc[:rows] = _randn(gen, rows, c.nKvHeads, c.headDim)
        vc[:rows] = _randn(gen, rows, c.nKvHeads, c.headDim)
    return kc, vc


def _layer_hidden(case, gen):
    return _randn(gen, case["tokens"], DecoderConfig().hidden)


def _head_inputs(case, seed):
    rng = np.random.default_rng(seed)
    w = _q8(rng, case["rows"], case["hidden"])
    return (w, rng.standard_normal(case["hidden"]).astype(np.float32),
            rng.normal(1, 0.1, case["hidden"]).astype(np.float32))


def _model_inputs(case, seed):
    rng = np.random.default_rng(seed)
    cfg = _layer_config(case)
    layers = [_layer_weights(rng, cfg) for _ in range(case["layers"])]
    return (cfg, layers, _q8(rng, case["vocab"], cfg.hidden),
            rng.normal(1, 0.1, cfg.hidden).astype(np.float32),
            int(rng.integers(0, case["vocab"])))


class _State:
    """What a program holds between calls; library buffers go with it."""

    def __init__(self, case, **kw):
        self.case = case
        self.__dict__.update(kw)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "ragged", "prefill"):
        x = _attention_inputs(case, seed)
        H, G, d = case["heads"], case["kv_heads"], case["head_dim"]
        s = _State(case, qn=torch.empty_like(x["q"]), o=torch.empty_like(x["q"]), **x)
        if kind == "decode":
            s.ws = ops.Workspace(H, G, d, case["keys"])
            s.new = slice(case["keys"] - 1, case["keys"])
        elif kind == "ragged":
            keys = _lengths(case)
            offs = np.concatenate([[0], np.cumsum(keys)[:-1]])
            s.offs = torch.from_numpy(offs.astype(np.int64)).cuda()
            s.keys = torch.from_numpy(keys.astype(np.int32)).cuda()
            s.longest = int(keys.max())
            s.ws = ops.Workspace(H, G, d, s.longest, 0, case["seqs"])
        else:
            s.ws = ops.Workspace(H, G, d, case["pos0"] + case["tokens"], case["tokens"])
            s.new = slice(case["pos0"], case["pos0"] + case["tokens"])
        return s
    if kind == "head":
        w, x, gain = _head_inputs(case, seed)
        rows, hid = case["rows"], case["hidden"]
        return _State(case, w=ops.Q8Matrix.from_packed(w, rows, hid),
                      x=torch.from_numpy(x).cuda(), gain=torch.from_numpy(gain).cuda(),
                      normed=torch.empty(hid, device="cuda"),
                      logits=torch.empty(rows, device="cuda"),
                      val=torch.empty(1, device="cuda"),
                      idx=torch.empty(1, dtype=torch.int32, device="cuda"),
                      ws=ops.DeviceBuffer(ops.lm_head_ws_bytes(rows, hid)))
    gen = torch.Generator("cuda").manual_seed(seed)
    if kind == "layer":
        cfg = _layer_config(case)
        layer = DecoderLayer.create(cfg, _layer_weights(np.random.default_rng(seed), cfg))
        kc, vc = _fill_cache(layer, case["pos0"], gen)
        # The layer alternates between two output buffers.
        outs = {layer.buf[b].ptr: _view(layer.buf[b], (case["tokens"], cfg.hidden))
                for b in ("h", "out")}
        return _State(case, layer=layer, hidden=_layer_hidden(case, gen), outs=outs,
                      k_new=kc[case["pos0"]:], v_new=vc[case["pos0"]:])
    cfg, weights, embd, gain, token = _model_inputs(case, seed)
    m = Model(cfg, weights, embd, gain, case["vocab"], max_generate=8)
    caches = [_fill_cache(layer, case["keys"] - 1, gen) for layer in m.layers]
    m.state.upload(np.array([case["keys"], 0], np.uint32))
    m.tok_idx.upload(np.array([token], np.uint32))
    logits = torch.empty(case["vocab"], device="cuda")
    val = torch.empty(1, device="cuda")
    idx = torch.empty(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    # The step a sampling loop captures: embedding, layers (the position is in
    # device memory), head with its logits kept. It is launched on the default
    # stream, as everything else here.
    stream = ops.Stream()
    ops.set_stream(stream)
    with ops.Graph() as graph:
        ops.embed(m.embd, m.tok_idx, 1, m.x)
        src = m.x
        for layer in m.layers:
            layer.encode_dev(src, m.state)
            src = layer.outputBufferDev()
        ops.lm_head(src, m.g_out, cfg.eps, m.embd, m.normed, logits, val, idx, m.head_ws)
    ops.set_stream(None)
    return _State(case, model=m, graph=graph, logits=logits, val=val, idx=idx,
                  hidden=_view(src, (cfg.hidden,)), k_new=caches[-1][0][case["keys"] - 1:],
                  v_new=caches[-1][1][case["keys"] - 1:])


# ---------------------------------------------------------------------- runs --
def run(s):
    c = s.case
    kind = c["kind"]
    if kind == "decode":
        ops.decode_layer(s.q, s.k, s.v, s.gq, s.gk, s.inv, EPS, c["pairing"], s.qn, s.kc, s.vc,
                         s.o, c["keys"] - 1, c["heads"], c["kv_heads"], c["head_dim"], c["keys"],
                         s.ws)
        return {"o": s.o, "q": s.qn, "k": s.kc[s.new], "v": s.vc[s.new]}
    if kind == "ragged":
        ops.decode_layer_ragged(s.q, s.k, s.v, s.gq, s.gk, s.inv, EPS, c["pairing"], s.qn, s.kc,
                                s.vc, s.offs, s.keys, s.o, c["seqs"], s.longest, c["heads"],
                                c["kv_heads"], c["head_dim"], s.ws)
        return {"o": s.o, "q": s.qn, "k": s.kc, "v": s.vc}
    if kind == "prefill":
        n, pos0, rows = c["tokens"], c["pos0"], c["pos0"] + c["tokens"]
        ops.qk_prologue(s.q, s.k, s.v, s.gq, s.gk, s.inv, EPS, c["pairing"], s.qn, s.kc, s.vc, n,
                        pos0, c["heads"], c["kv_heads"], c["head_dim"], rows)
        ops.attn_prefill(s.qn, s.kc, s.vc, s.o, c["heads"], c["kv_heads"], c["head_dim"], n, pos0,
                         s.ws)
        return {"o": s.o, "q": s.qn, "k": s.kc[s.new], "v": s.vc[s.new]}
    if kind == "head":
        ops.lm_head(s.x, s.gain, EPS, s.w, s.normed, s.logits, s.val, s.idx, s.ws)
        return {"logits": s.logits, "normed": s.normed, "best": s.val, "token": s.idx}
    if kind == "layer":
        s.layer.nKeys = c["pos0"]  # the same positions again
        s.layer.encodePrefill(c["tokens"], src=s.hidden)
        return {"out": s.outs[s.layer.outputBuffer().ptr], "k": s.k_new, "v": s.v_new}
    s.graph.launch()
    return {"logits": s.logits, "best": s.val, "token": s.idx, "hidden": s.hidden,
            "k": s.k_new, "v": s.v_new}


# ---------------------------------------------------------------------- work --
def _pairs(n, pos0):
    return n * pos0 + n * (n + 1) // 2


def _layer_params():
    return sum(r * c for r, c in DecoderConfig().shapes().values())


def work(case):
    kind = case["kind"]
    if kind in ("decode", "ragged", "prefill"):
        H, G, d = case["heads"], case["kv_heads"], case["head_dim"]
        if kind == "decode":
            n, rows = 1, case["keys"]
            pairs = rows
        elif kind == "ragged":
            n, rows = case["seqs"], int(_lengths(case).sum())
            pairs = rows
        else:
            n, rows = case["tokens"], case["pos0"] + case["tokens"]
            pairs = _pairs(n, case["pos0"])
        # Raw q, k, v in; q, o and the new rows out; the cached rows in once.
        new = 4 * n * d * (H + 2 * G + 2 * H + 2 * G)
        return {"bytes": new + 8 * (rows - n) * G * d, "flops": 4.0 * H * d * pairs}
    if kind == "head":
        rows, hid = case["rows"], case["hidden"]
        return {"bytes": rows * hid * 34 // 32 + 4 * (3 * hid + rows), "flops": 2.0 * rows * hid}
    cfg = DecoderConfig()
    H, G, d = cfg.nHeads, cfg.nKvHeads, cfg.headDim
    if kind == "layer":
        n, pos0 = case["tokens"], case["pos0"]
        return {"bytes": _layer_params() * 34 // 32 + 8 * pos0 * G * d
                + 4 * n * (2 * cfg.hidden + 2 * G * d),
                "flops": 2.0 * n * _layer_params() + 4.0 * H * d * _pairs(n, pos0)}
    n_layers, keys, vocab = case["layers"], case["keys"], case["vocab"]
    return {"bytes": n_layers * (_layer_params() * 34 // 32 + 8 * keys * G * d)
            + vocab * cfg.hidden * 34 // 32 + 4 * vocab,
            "flops": n_layers * (2.0 * _layer_params() + 4.0 * H * d * keys)
            + 2.0 * vocab * cfg.hidden}


def tolerance(case):
    """f32 sums in another order, at about four times the distance from 64
    bits that was measured over the listed and drawn cases: attention outputs
    2e-7 to 8e-7, a layer's 2e-7, a 28-layer model's logits 1.7e-6. The
    projections' order of sums is part of their contract, so the head's
    numbers stay the same; attention's is not."""
    kind = case["kind"]
    if kind == "head":
        return "exact"
    if kind == "model":
        return {"rel": 8e-6, "max": 1e-4, "differ": 0.0}
    if kind == "layer":
        return {"rel": 1e-6, "max": 2e-5}
    return {"rel": 4e-6, "max": 1e-4}


# --------------------------------------------------------- 64-bit references --
def _norm64(x, gain):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gain.double()


def _rope64(x, inv, pos, pairing):
    """x [n][heads][d]; the angle is position * inv_freq rounded to 32 bits,
    as the entry points define it."""
    theta = (pos.double()[:, None] * inv.double()).float().double()
    c, s = torch.cos(theta)[:, None], torch.sin(theta)[:, None]
    if pairing == "neox":
        a, b = x.chunk(2, -1)
        return torch.cat([a * c - b * s, b * c + a * s], -1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)


def _attend64(q, kc, vc, pos0):
    """Causal attention of q [n][H][d] at positions pos0.. over rows 0..pos0+n-1."""
    n, H, d = q.shape
    group = H // kc.shape[1]
    rows = pos0 + n
    o = torch.empty_like(q)
    for kv in range(kc.shape[1]):
        k, v = kc[:rows, kv].double().contiguous(), vc[:rows, kv].double().contiguous()
        kt = k.t().contiguous()
        for a in range(0, n, 1024):
            b = min(n, a + 1024)
            hidden = torch.arange(rows, device="cuda") > torch.arange(
                pos0 + a, pos0 + b, device="cuda")[:, None]
            for h in range(kv * group, (kv + 1) * group):
                p = (q[a:b, h].contiguous() @ kt) / math.sqrt(d)
                p = torch.softmax(p.masked_fill_(hidden, -math.inf), -1)
                o[a:b, h] = p @ v
    return o


def _dequant64(packed, rows, cols):
    t = torch.from_numpy(packed).cuda().view(rows * cols // 32, 34)
    scale = t[:, :2].contiguous().view(torch.float16).double()
    return (t[:, 2:].contiguous().view(torch.int8).double() * scale).view(rows, cols)


def _layer64(x, w, cfg, kc, vc, pos0):
    """One decoder layer in 64 bits; kc, vc: the cache's first pos0 rows."""
    n = x.shape[0]
    H, G, d = cfg.nHeads, cfg.nKvHeads, cfg.headDim
    m = {name: _dequant64(w[name], r, c) for name, (r, c) in cfg.shapes().items()}
    g = {name: torch.from_numpy(w[name]).cuda() for name, _ in LAYER_GAINS}
    inv = torch.from_numpy(_inv_freq(d)).cuda()
    pos = torch.arange(pos0, pos0 + n, device="cuda")

    def proj(name, v):
        return v @ m[name].t().contiguous()

    y = _norm64(x, g["attn_norm.weight"])
    q = _rope64(_norm64(proj("attn_q.weight", y).view(n, H, d), g["attn_q_norm.weight"]), inv,
                pos, cfg.ropePairing)
    k = _rope64(_norm64(proj("attn_k.weight", y).view(n, G, d), g["attn_k_norm.weight"]), inv,
                pos, cfg.ropePairing)
    v = proj("attn_v.weight", y).view(n, G, d)
    o = _attend64(q, torch.cat([kc.double(), k]), torch.cat([vc.double(), v]), pos0)
    x = x.double() + proj("attn_output.weight", o.reshape(n, H * d))
    y = _norm64(x, g["ffn_norm.weight"])
    act = torch.nn.functional.silu(proj("ffn_gate.weight", y)) * proj("ffn_up.weight", y)
    return x + proj("ffn_down.weight", act), k, v


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "ragged", "prefill"):
        x = _attention_inputs(case, seed)
        pairing = case["pairing"]
        if kind == "ragged":
            keys = torch.from_numpy(_lengths(case)).cuda()
            pos, ends = keys - 1, torch.cumsum(keys, 0).tolist()
        else:
            pos0 = case["keys"] - 1 if kind == "decode" else case["pos0"]
            pos = torch.arange(pos0, pos0 + x["q"].shape[0], device="cuda")
        q = _rope64(_norm64(x["q"], x["gq"]), x["inv"], pos, pairing)
        k = _rope64(_norm64(x["k"], x["gk"]), x["inv"], pos, pairing)
        v = x["v"].double()
        if kind == "ragged":
            o = torch.empty_like(q)
            kc, vc = x["kc"].double(), x["vc"].double()
            for b, (end, n) in enumerate(zip(ends, keys.tolist())):
                kc[end - 1], vc[end - 1] = k[b], v[b]
                o[b] = _attend64(q[b:b + 1], kc[end - n:end], vc[end - n:end], n - 1)[0]
            return {"o": o, "q": q, "k": kc, "v": vc}
        o = _attend64(q, torch.cat([x["kc"][:pos0].double(), k]),
                      torch.cat([x["vc"][:pos0].double(), v]), pos0)
        return {"o": o, "q": q, "k": k, "v": v}
    if kind == "head":
        w, x, gain = _head_inputs(case, seed)
        normed = _norm64(torch.from_numpy(x).cuda(), torch.from_numpy(gain).cuda())
        logits = _dequant64(w, case["rows"], case["hidden"]) @ normed
        return {"logits": logits, "normed": normed, "best": logits.max()[None],
                "token": logits.argmax()[None].int()}
    gen = torch.Generator("cuda").manual_seed(seed)
    if kind == "layer":
        cfg, n, pos0 = _layer_config(case), case["tokens"], case["pos0"]
        w = _layer_weights(np.random.default_rng(seed), cfg)
        kv = [_randn(gen, pos0, cfg.nKvHeads, cfg.headDim) if pos0 else
              torch.empty(0, cfg.nKvHeads, cfg.headDim, device="cuda") for _ in range(2)]
        out, k, v = _layer64(_layer_hidden(case, gen), w, cfg, kv[0], kv[1], pos0)
        return {"out": out, "k": k, "v": v}
    cfg, weights, embd, gain, token = _model_inputs(case, seed)
    table = _dequant64(embd, case["vocab"], cfg.hidden)
    x, pos0 = table[token:token + 1].clone(), case["keys"] - 1
    for w in weights:
        kv = [_randn(gen, pos0, cfg.nKvHeads, cfg.headDim) for _ in range(2)]
        x, k, v = _layer64(x, w, cfg, kv[0], kv[1], pos0)
    logits = table @ _norm64(x[0], torch.from_numpy(gain).cuda())
    return {"logits": logits, "best": logits.max()[None], "token": logits.argmax()[None].int(),
            "hidden": x[0], "k": k, "v": v}
