"""The engine's measured workloads: what a program that serves Qwen3-MoE models at batch 1 calls,
through the package's public entry points, with the inputs such a program has in hand.

Each case names its `path`:
  prefill  a prompt through the batched prefill from an empty cache, the last token's logits
  score    a prompt, then given continuation tokens one step each with their logits (scoring an
           answer; each step is what a chat turn runs per generated token)
  decode   greedy generation by the exact token step: prompt tokens, then new ones
  sample   one draw of the device sampler from logits, with the padding-vocabulary mask
  attend   attention of one query token over device-resident keys and values
  matvec   the matrix-vector products of one decoder layer, one backend call each, as a host-driven
           model issues them

Models are random-init with the repository's own 30B-A3B layer shapes, a few layers deep (the
layers are alike; more of them only repeat the same work).  The embedding rows are scaled up so
that, as in a trained model, the residual stream is large against one layer's update: otherwise a
random model's routing sits on ties and its logits follow every rounding.
"""
import importlib
import math
import os
import struct

import numpy as np
import torch  # before the engine's library, so that both use one HIP runtime

engine = importlib.import_module("qwen-30brust_amd")
synth = importlib.import_module("qwen-30brust_amd.synth")

VOCAB = 151936
EMBED_SCALE = 64.0
# bytes and weights of one block
BLOCK = {0: (4, 1), 2: (18, 32), 8: (34, 32), 12: (144, 256), 13: (176, 256), 14: (210, 256)}
MAIN = {"q4_k_m": 12, "q5_k_m": 13, "q6_k": 14, "q8_0": 8, "q4_0": 2, "small": 12}


def spec_of(weights):
    """The synthetic model of a weight mix.  q4_k_m: four 30B-A3B layers, the full vocabulary and a
    4,096-token context; the other mixes two layers and a small vocabulary; small: another
    geometry, which the persistent token step and the batched prefill do not cover."""
    main = MAIN[weights]
    kinds = synth._k_types(attn=main, down=main, out=14 if main >= 12 else main, embd=12)
    more = 14 if weights in ("q4_k_m", "q5_k_m") else synth.NONE
    if weights == "small":
        return synth.Spec(1024, 4, 16, 4, 64, 32, 4, 512, 32768, 512, types=dict(kinds, ffn_down_exps=14), seed=5)
    if weights == "q4_k_m":
        return synth.Spec(2048, 4, 32, 4, 128, 128, 8, 768, VOCAB, 4096, types=kinds, more_bits_type=more, seed=11)
    return synth.Spec(2048, 2, 32, 4, 128, 128, 8, 768, 4096, 4096, types=kinds, more_bits_type=more, seed=13)


def listed():
    return [
        # a short chat message
        {"name": "prefill-24", "path": "prefill", "weights": "q4_k_m", "tokens": 24},
        # a chat prompt with some context, ragged against every tile
        {"name": "prefill-331", "path": "prefill", "weights": "q4_k_m", "tokens": 331},
        # the benchmark's prompt
        {"name": "prefill-2048", "path": "prefill", "weights": "q4_k_m", "tokens": 2048},
        # a long document: a second chunk that attends to the first
        {"name": "prefill-3159", "path": "prefill", "weights": "q4_k_m", "tokens": 3159},
        # the same path on a file quantised to 8 bits
        {"name": "prefill-517-q8_0", "path": "prefill", "weights": "q8_0", "tokens": 517},
        # scoring an answer after a prompt
        {"name": "score-640", "path": "score", "weights": "q4_k_m", "tokens": 640, "more": 12},
        # generation through the exact step
        {"name": "decode-48", "path": "decode", "weights": "q4_k_m", "tokens": 32, "more": 16},
        # the same on a model of other shapes (per-phase kernels)
        {"name": "decode-40-small", "path": "decode", "weights": "small", "tokens": 24, "more": 16},
        # the chat front end's default sampling
        {"name": "sample-chat", "path": "sample", "vocab": VOCAB, "temperature": 0.2, "top_k": 20, "top_p": 0.8},
        # sampling from the whole distribution
        {"name": "sample-full", "path": "sample", "vocab": VOCAB, "temperature": 1.0, "top_k": 0, "top_p": 0.95},
        # decode attention late in the context
        {"name": "attend-3581", "path": "attend", "keys": 3581, "heads": 32, "kvheads": 4, "dim": 128},
        # one layer's products through Backend.matvec
        {"name": "matvec-layer", "path": "matvec", "weights": "q4_k_m", "layer": 0, "experts": 8},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    path = rng.choice(["prefill", "prefill", "prefill", "prefill", "score", "decode", "sample", "sample", "attend",
                       "matvec"])
    if path == "prefill":
        return {"path": path, "weights": rng.choice(["q4_k_m"] * 4 + ["q5_k_m", "q6_k", "q8_0", "q4_0"]),
                "tokens": _log_int(rng, 8, 3159)}
    if path == "score":
        return {"path": path, "weights": "q4_k_m", "tokens": _log_int(rng, 16, 1800), "more": rng.randint(2, 12)}
    if path == "decode":
        return {"path": path, "weights": rng.choice(["q4_k_m", "q8_0", "q5_k_m", "small"]),
                "tokens": _log_int(rng, 2, 32), "more": rng.randint(2, 16)}
    if path == "sample":
        return {"path": path, "vocab": rng.choice([_log_int(rng, 2000, VOCAB), VOCAB]),
                "temperature": round(rng.uniform(0.2, 1.3), 2), "top_k": rng.choice([0, 0, 1, 20, 50, _log_int(rng, 2, 1500)]),
                "top_p": rng.choice([0.8, 0.9, 0.95, 1.0])}
    if path == "attend":
        dim = rng.choice([64, 128, 128, 128])
        kvheads = rng.choice([2, 4, 8])
        return {"path": path, "keys": _log_int(rng, 16, 4096), "heads": kvheads * rng.choice([1, 4, 5, 8]),
                "kvheads": kvheads, "dim": dim}
    weights = rng.choice(["q4_k_m", "q5_k_m", "q6_k", "q8_0"])
    return {"path": path, "weights": weights, "layer": rng.randrange(spec_of(weights).layers), "experts": rng.randint(1, 8)}


# --------------------------------------------------------------- models --
_models = {}
_device = None


def _tensors(img):
    """name -> (kind, dims, byte offset) of a GGUF image."""
    def text(o):
        n, = struct.unpack_from("<Q", img, o)
        return bytes(img[o + 8:o + 8 + n]).decode(), o + 8 + n

    def skip(kind, o):
        if kind == 8:
            return text(o)[1]
        if kind == 9:
            k, n = struct.unpack_from("<IQ", img, o)
            o += 12
            for _ in range(n):
                o = skip(k, o)
            return o
        return o + {0: 1, 1: 1, 2: 2, 3: 2, 4: 4, 5: 4, 6: 4, 7: 1, 10: 8, 11: 8, 12: 8}[kind]

    _, _, count, keys = struct.unpack_from("<IIQQ", img, 0)
    o, align = 24, 32
    for _ in range(keys):
        key, o = text(o)
        kind, = struct.unpack_from("<I", img, o)
        if key == "general.alignment":
            align, = struct.unpack_from("<I", img, o + 4)
        o = skip(kind, o + 4)
    found = {}
    for _ in range(count):
        name, o = text(o)
        rank, = struct.unpack_from("<I", img, o)
        dims = struct.unpack_from("<%dQ" % rank, img, o + 4)
        kind, at = struct.unpack_from("<IQ", img, o + 4 + 8 * rank)
        found[name] = [kind, dims, at]
        o += 16 + 8 * rank
    base = -(-o // align) * align
    return {n: (k, d, base + a) for n, (k, d, a) in found.items()}


def _model(weights):
    """(model, image, tensor table) of a weight mix: loaded once, as a serving program does."""
    if weights not in _models:
        spec = spec_of(weights)
        img = synth.build_image(spec, threads=min(16, os.cpu_count() or 1))
        tensors = _tensors(img)
        kind, dims, at = tensors["token_embd.weight"]
        blocks = img[at:at + dims[0] * dims[1] // 256 * 144].reshape(-1, 144)
        assert kind == 12
        scales = np.ascontiguousarray(blocks[:, :4]).view(np.float16) * np.float16(EMBED_SCALE)
        blocks[:, :4] = scales.view(np.uint8)
        _models[weights] = engine.Model(img, spec.context, device=engine.Device(0)), img, tensors
    return _models[weights]


def _shared_device():
    global _device
    if _device is None:
        _device = engine.Device(0)
    return _device


def _matvec_names(spec, layer, experts):
    p = "blk.%d." % layer
    H, qd, ff = spec.hidden, spec.heads * spec.head_dim, spec.ff
    named = [(p + "attn_q.weight", None, H), (p + "attn_k.weight", None, H), (p + "attn_v.weight", None, H),
             (p + "attn_output.weight", None, qd), (p + "ffn_gate_inp.weight", None, H)]
    for e in experts:
        named += [(p + "ffn_gate_exps.weight", e, H), (p + "ffn_up_exps.weight", e, H), (p + "ffn_down_exps.weight", e, ff)]
    return named


# -------------------------------------------------------------- measured --
def prepare(case, seed):
    rng = np.random.default_rng(seed)
    path = case["path"]
    if path in ("prefill", "score", "decode"):
        model = _model(case["weights"])[0]
        n = case["tokens"] + (case["more"] if path == "score" else 0)
        return {"path": path, "model": model, "tokens": rng.integers(0, model.config["vocab"], n).astype(np.uint32),
                "n": case["tokens"], "more": case.get("more", 0)}
    if path == "sample":
        # logits spread as a language model's: a broad bulk and a few likely ids
        n = case["vocab"]
        logits = rng.normal(0.0, 2.5, n).astype(np.float32)
        logits[rng.integers(0, n, 64)] += rng.uniform(4.0, 12.0, 64).astype(np.float32)
        valid = np.ones(n, np.uint8)
        valid[n - n // 512:] = 0
        sampler = engine.Sampler(seed % 2 ** 32, case["temperature"], case["top_k"], case["top_p"])
        return {"path": path, "dev": _shared_device(), "sampler": sampler, "logits": logits, "valid": valid}
    if path == "attend":
        gen = torch.Generator(device="cuda").manual_seed(seed)
        d, kv, h, t = case["dim"], case["kvheads"], case["heads"], case["keys"]
        q, k, v = (torch.randn(n, generator=gen, device="cuda") for n in (h * d, t * kv * d, t * kv * d))
        q *= 2.0  # normed and weighted queries: a few keys stand out
        torch.cuda.synchronize()
        return {"path": path, "dev": _shared_device(), "q": q, "k": k, "v": v, "heads": h, "kvheads": kv, "dim": d,
                "out": torch.empty_like(q), "stream": torch.cuda.Stream()}
    spec = spec_of(case["weights"])
    named = _matvec_names(spec, case["layer"], rng.permutation(spec.experts)[:case["experts"]].tolist())
    return {"path": path, "backend": engine.HipBackend(_model(case["weights"])[0]),
            "calls": [(name, e, rng.standard_normal(cols).astype(np.float32)) for name, e, cols in named]}


def run(state):
    path = state["path"]
    if path in ("prefill", "score", "decode"):
        model, tokens, n = state["model"], state["tokens"], state["n"]
        model.reset()
        if path == "decode":
            ids, logits = model.generate(tokens, state["more"], want_logits=True)
            return {"ids": ids, "logits": logits}
        last = model.prefill(tokens[:n])[1]
        if path == "prefill":
            return {"logits": last}
        return {"logits": [last] + [model.forward(int(t)) for t in tokens[n:]]}
    if path == "sample":
        return {"id": int(state["sampler"].sample(state["dev"], state["logits"], state["valid"]))}
    if path == "attend":
        s, dev = state, state["dev"]
        dev._check(engine.lib().qh_attention_noalloc(dev.h, s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                                                     s["k"].numel(), s["heads"], s["kvheads"], s["dim"],
                                                     s["out"].data_ptr(), s["stream"].cuda_stream))
        return {"out": s["out"]}
    return {"y": [state["backend"].matvec(name, e, x) for name, e, x in state["calls"]]}


# ----------------------------------------------------------------- bounds --
def _bytes(kind, weights):
    size, per = BLOCK[kind]
    return weights * size / per


def _layer(spec, i):
    """(bytes, weights) of a layer's attention and router, and of one expert."""
    n = spec.layers
    more = spec.more_bits_type != synth.NONE and (i < n // 8 or i >= 7 * n // 8 or (i - n // 8) % 3 == 2)
    t = {k: (14 if more and k in ("attn_v", "ffn_down_exps") else v) for k, v in spec.types.items()}
    H, qd, kvd = spec.hidden, spec.heads * spec.head_dim, spec.kvheads * spec.head_dim
    dense = (_bytes(t["attn_q"], qd * H) + _bytes(t["attn_k"], kvd * H) + _bytes(t["attn_v"], kvd * H)
             + _bytes(t["attn_output"], qd * H) + 4 * spec.experts * H)
    expert = 2 * _bytes(t["ffn_gate_exps"], spec.ff * H) + _bytes(t["ffn_down_exps"], spec.ff * H)
    return dense, 2 * (qd + kvd) * H + spec.experts * H, expert, 3 * spec.ff * H


def _tokens_work(spec, n, past=0):
    """n tokens at positions past.. in one pass over the weights, one vocabulary projection."""
    kvd, H = spec.kvheads * spec.head_dim, spec.hidden
    used = spec.experts * (1 - (1 - spec.top / spec.experts) ** n)
    head = _bytes(spec.types["output"], spec.vocab * H)
    total, flops = head + 4 * spec.vocab + n * _bytes(spec.types["token_embd"], H), 2 * spec.vocab * H
    for i in range(spec.layers):
        dense, dense_w, expert, expert_w = _layer(spec, i)
        total += dense + used * expert + 8 * kvd * (past + n)
        pairs = n * past + n * (n + 1) / 2
        flops += 2 * n * (dense_w + spec.top * expert_w) + 4 * spec.heads * spec.head_dim * pairs
    return total, flops


def work(case):
    path = case["path"]
    if path == "sample":
        n = case["vocab"]
        return {"bytes": 5 * n, "flops": 2 * n}
    if path == "attend":
        d, t = case["dim"], case["keys"]
        return {"bytes": 8 * case["kvheads"] * t * d + 8 * case["heads"] * d, "flops": 4 * case["heads"] * t * d}
    spec = spec_of(case["weights"])
    if path == "matvec":
        dense, dense_w, expert, expert_w = _layer(spec, case["layer"])
        n = case["experts"]
        floats = sum(cols for _, _, cols in _matvec_names(spec, 0, range(n)))
        floats += (spec.heads + 2 * spec.kvheads) * spec.head_dim + spec.hidden + spec.experts
        floats += n * (2 * spec.ff + spec.hidden)
        return {"bytes": dense + n * expert + 4 * floats, "flops": 2 * (dense_w + n * expert_w)}
    n = case["tokens"]
    steps = [(n, 0)] if path != "decode" else [(1, p) for p in range(n)]
    if path == "score":
        steps += [(1, n + i) for i in range(case["more"])]
    elif path == "decode":
        steps += [(1, n + i) for i in range(max(0, case["more"] - 1))]
    both = [_tokens_work(spec, m, p) for m, p in steps]
    return {"bytes": sum(b for b, _ in both), "flops": sum(f for _, f in both)}


def tolerance(case):
    path = case["path"]
    if path == "sample":
        return "exact"
    if path in ("prefill", "score"):
        small = case["weights"] == "small"
        return {"rel": 1e-5, "max": 1e-4} if small else {"rel": 6e-3, "max": 3e-2}  # fp16 operands
    if path == "decode":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 4e-6, "max": 4e-5}  # 32-bit sums


# ------------------------------------------------------- the same in f64 --
def _decode(raw, kind):
    """Values (f64) of packed GGML blocks; raw is (rows, row bytes) uint8 on the GPU."""
    if kind == 0:
        return raw.contiguous().view(torch.float32).double()
    b = raw.reshape(raw.shape[0], -1, BLOCK[kind][0])

    def half(at):
        return b[..., at:at + 2].contiguous().view(torch.float16).double()

    if kind == 8:
        v = b[..., 2:].contiguous().view(torch.int8).double() * half(0)
    elif kind == 2:
        q = b[..., 2:]
        v = (torch.cat([q & 15, q >> 4], -1).double() - 8) * half(0)
    elif kind == 14:
        ql, qh = b[..., :128].reshape(*b.shape[:2], 2, 2, 32), b[..., 128:192].reshape(*b.shape[:2], 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], -2)  # (.., half, 4 runs of 32, 32)
        high = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], -2)
        q = (low | (high << 4)).double() - 32
        sc = b[..., 192:208].contiguous().view(torch.int8).double().reshape(*b.shape[:2], 2, 4, 2, 1)
        v = q.reshape(*b.shape[:2], 2, 4, 2, 16) * sc * half(208).reshape(*b.shape[:2], 1, 1, 1, 1)
    else:
        s = b[..., 4:16].int()
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], -1).double()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
        qs = b[..., -128:].reshape(*b.shape[:2], 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], -2).reshape(*b.shape[:2], 8, 32)
        if kind == 13:
            qh = b[..., 16:48].reshape(*b.shape[:2], 1, 32)
            q = q | torch.cat([((qh >> i) & 1) << 4 for i in range(8)], -2)
        v = q.double() * (half(0) * sc)[..., None] - (half(2) * mn)[..., None]
    return v.reshape(raw.shape[0], -1)


class _Exact:
    """The model's forward pass in 64 bits."""

    def __init__(self, weights):
        self.spec = spec_of(weights)
        _, self.img, self.tensors = _model(weights)

    def rows(self, name, ids=None):
        kind, dims, at = self.tensors[name]
        size, per = BLOCK[kind]
        count = math.prod(dims[1:])
        raw = self.img[at:at + count * dims[0] // per * size].reshape(count, -1)
        raw = raw if ids is None else raw[ids]
        return _decode(torch.from_numpy(np.ascontiguousarray(raw)).cuda(), kind)

    def vector(self, name):
        return self.rows(name)[0]

    def expert(self, name, e):
        n = self.tensors[name][1][1]
        return self.rows(name, slice(e * n, (e + 1) * n))

    def norm(self, x, w):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + self.spec.eps) * w

    def logits(self, tokens, last):
        """Logits after each of the `last` last tokens."""
        s = self.spec
        n, d, half = len(tokens), s.head_dim, s.head_dim // 2
        x = self.rows("token_embd.weight", np.asarray(tokens, np.int64))
        freq = np.float32(s.theta) ** (np.float32(-2) * np.arange(half, dtype=np.float32) / np.float32(d))
        # the table's angles are 32-bit by definition
        angle = torch.from_numpy(np.arange(n, dtype=np.float32)[:, None] * freq[None, :]).cuda().double()
        cos, sin = angle.cos()[:, None], angle.sin()[:, None]

        def rope(v):
            a, b = v[..., :half], v[..., half:]
            return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

        mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
        for i in range(s.layers):
            p = "blk.%d." % i
            h = self.norm(x, self.vector(p + "attn_norm.weight"))
            q, k, v = ((h @ self.rows(p + "attn_%s.weight" % m).T).reshape(n, -1, d) for m in "qkv")
            q = rope(self.norm(q, self.vector(p + "attn_q_norm.weight")))
            k = rope(self.norm(k, self.vector(p + "attn_k_norm.weight")))
            out = torch.empty_like(q)
            for j in range(s.heads):
                g = j * s.kvheads // s.heads
                a = (q[:, j] @ k[:, g].T / math.sqrt(d)).masked_fill_(mask, -math.inf)
                out[:, j] = torch.softmax(a, -1) @ v[:, g]
            x = x + out.reshape(n, -1) @ self.rows(p + "attn_output.weight").T
            h = self.norm(x, self.vector(p + "ffn_norm.weight"))
            top, ids = (h @ self.rows(p + "ffn_gate_inp.weight").T).topk(s.top, -1)
            w = torch.softmax(top, -1)
            for e in ids.unique().tolist():
                t, r = (ids == e).nonzero(as_tuple=True)
                gate = h[t] @ self.expert(p + "ffn_gate_exps.weight", e).T
                up = h[t] @ self.expert(p + "ffn_up_exps.weight", e).T
                y = (gate * torch.sigmoid(gate) * up) @ self.expert(p + "ffn_down_exps.weight", e).T
                x.index_add_(0, t, y * w[t, r][:, None])
        return self.norm(x[n - last:], self.vector("output_norm.weight")) @ self.rows("output.weight").T


def exact(case, seed):
    path = case["path"]
    if path == "sample":
        return None  # an id
    state = prepare(case, seed)
    if path == "attend":
        h, kv, d = state["heads"], state["kvheads"], state["dim"]
        q, k, v = (state[m].double().reshape(-1, c, d) for m, c in (("q", h), ("k", kv), ("v", kv)))
        k, v = (m.repeat_interleave(h // kv, 1).transpose(0, 1) for m in (k, v))
        a = torch.softmax((k @ q[0][:, :, None])[..., 0] / math.sqrt(d), -1)
        return {"out": (a[:, None, :] @ v).reshape(-1)}
    m = _Exact(case["weights"])
    if path == "matvec":
        y = []
        for name, e, x in state["calls"]:
            w = m.rows(name) if e is None else m.expert(name, e)
            y.append(w @ torch.from_numpy(x).cuda().double())
        return {"y": y}
    tokens = state["tokens"].tolist()
    if path == "prefill":
        return {"logits": m.logits(tokens, 1)[0]}
    if path == "score":
        return {"logits": list(m.logits(tokens, state["more"] + 1))}
    for _ in range(state["more"]):
        logits = m.logits(tokens, 1)[0]
        tokens.append(int(logits.argmax()))
    return {"ids": None, "logits": logits}
