"""Timed workloads of the Gemma 3 Q8_0 token loop: single layers through the standalone Q8_0 entry
points, and whole calls of the executor (teacher-forced decode, prompt prefill, a chat turn on a
long context, batched decode of independent sequences), at the Gemma-3-270M shape and around it.

Weights, activations and token ids are made on the GPU from a seed: N(0, 0.02) matrices quantised
to Q8_0 along their rows, norm weights 1 + N(0, 0.1), N(0, 1) activations, uniform token ids.
"""
import ctypes
import os
import sys
import weakref

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vortex-rt_amd"))
import synth  # noqa: E402
import vrt  # noqa: E402

SHAPE = synth.GEMMA3_270M
CONTEXT = 8704          # positions of the executor: the 8192-token prompt and room to decode
D, HEADS, HD = SHAPE["d_model"], SHAPE["n_heads"], SHAPE["head_dim"]
FFN, VOCAB, WINDOW = SHAPE["ffn"], SHAPE["vocab"], SHAPE["window"]
EPS = SHAPE["eps"]
QW = HEADS * HD


def listed():
    return [
        # the fused q|k|v projection of one decoder layer for one token: the smallest call
        {"name": "qkv_layer", "kind": "multi", "k": D, "rows0": QW, "rows1": HD, "rows2": HD},
        # the feed-forward of one decoder layer for one token
        {"name": "ffn_layer", "kind": "ffn", "k": D, "ffn": FFN, "out": D},
        # one projection of a size that fits no power of two: 35 blocks a row, an odd row count
        {"name": "matvec_ragged", "kind": "matvec", "k": 1120, "rows": 5003},
        # the tied LM head as its own call, and the greedy token from its logits
        {"name": "head_argmax", "kind": "head", "k": D, "rows": VOCAB},
        # quantising a loaded fp32 matrix to Q8_0 and expanding it back
        {"name": "codec", "kind": "codec", "rows": 65536, "k": D, "variant": 0},
        # the headline loop: one sequence decoding from a short prompt, 136 positions
        {"name": "decode_136", "kind": "decode", "blocks": 18, "steps": 136, "kv": "f32"},
        # a chat turn: a long prompt in one prefill, then token by token with a half-precision cache
        {"name": "chat_4096", "kind": "chat", "blocks": 18, "prompt": 4096, "steps": 32, "kv": "f16"},
        # a short question's prompt, of an odd length
        {"name": "prefill_37", "kind": "prefill", "blocks": 18, "tokens": 37, "kv": "f32"},
        # the benchmark's prompt
        {"name": "prefill_512", "kind": "prefill", "blocks": 18, "tokens": 512, "kv": "f32"},
        # a document: more positions than one pass of the prefill holds
        {"name": "prefill_8192", "kind": "prefill", "blocks": 18, "tokens": 8192, "kv": "f32"},
        # a small service: a few sequences together, from their first token on
        {"name": "batch_8", "kind": "batch", "blocks": 18, "seqs": 8, "steps": 48},
        # a full batch, over short histories and ones that have outgrown the short path
        {"name": "batch_64", "kind": "batch", "blocks": 18, "seqs": 64, "steps": 48},
    ]


def _log(rng, lo, hi):
    """An integer between lo and hi, even over its logarithm."""
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    kind = rng.choice(["multi", "ffn", "matvec", "head", "codec", "decode", "chat", "prefill", "prefill", "batch", "batch"])
    if kind == "multi":   # projections of one layer, of any width the matvec takes
        return {"kind": kind, "k": 32 * _log(rng, 4, 64), "rows0": _log(rng, 64, 4096), "rows1": _log(rng, 32, 1024),
                "rows2": _log(rng, 32, 1024)}
    if kind == "ffn":
        return {"kind": kind, "k": 32 * _log(rng, 4, 64), "ffn": 32 * _log(rng, 8, 256), "out": _log(rng, 64, 2048)}
    if kind == "matvec":
        return {"kind": kind, "k": 32 * _log(rng, 2, 256), "rows": _log(rng, 16, 16384)}
    if kind == "head":
        return {"kind": kind, "k": 32 * _log(rng, 4, 20), "rows": _log(rng, 4096, VOCAB)}
    if kind == "codec":
        return {"kind": kind, "rows": _log(rng, 64, 65536), "k": 32 * _log(rng, 4, 20), "variant": rng.randrange(2)}
    blocks = rng.choice([6, 12, 18])
    kv = rng.choice(["f32", "f16", "bf16"])
    if kind == "decode":
        return {"kind": kind, "blocks": blocks, "steps": _log(rng, 8, 136), "kv": kv}
    if kind == "chat":
        return {"kind": kind, "blocks": blocks, "prompt": _log(rng, 128, 4096), "steps": _log(rng, 4, 32), "kv": kv}
    if kind == "prefill":
        return {"kind": kind, "blocks": blocks, "tokens": _log(rng, 8, 8192), "kv": kv}
    return {"kind": kind, "blocks": blocks, "seqs": _log(rng, 1, 64), "steps": _log(rng, 6, 48)}


# ---- inputs ---------------------------------------------------------------------------------

class Span:
    """Device memory of a torch tensor, as the binding's functions take a buffer."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()
        self.nbytes = tensor.numel() * tensor.element_size()


_ctx = None


def _context():
    """The program's device context: one, as long as it runs."""
    global _ctx
    if _ctx is None:
        _ctx = vrt.Context("0")
    return _ctx


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _blocks(gen, rows, k, out=None, std=0.02):
    """A [rows x k] N(0, std^2) matrix as Q8_0 blocks, uint8 [rows * k / 32, 34]."""
    n = rows * k // 32
    w = torch.randn(n, 32, generator=gen, device="cuda").mul_(std)
    scale = w.abs().amax(dim=1).div_(127.0)
    if out is None:
        out = torch.empty(n, 34, dtype=torch.uint8, device="cuda")
    out[:, :2] = scale.half().view(torch.uint8).view(n, 2)
    out[:, 2:] = w.div_(scale[:, None]).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
    return out


def _dense(blocks, rows, k):
    """The matrix that Q8_0 blocks stand for, in 64 bits."""
    s = blocks[:, :2].contiguous().view(torch.float16).double()
    return (s * blocks[:, 2:].contiguous().view(torch.int8).double()).view(rows, k)


def _matrices(gen, shapes):
    """Q8_0 matrices one after another in one buffer, as a file's tensor section holds them: the
    buffer, the byte offset of each, and their blocks."""
    offs, at = [], 0
    for rows, k in shapes:
        offs.append(at)
        at += (rows * k // 32 * 34 + 31) // 32 * 32
    arena = torch.zeros(at + 256, dtype=torch.uint8, device="cuda")
    views = []
    for (rows, k), o in zip(shapes, offs):
        n = rows * k // 32
        v = arena[o:o + n * 34].view(n, 34)
        _blocks(gen, rows, k, v)
        views.append(v)
    return arena, offs, views


_LAYER = (("attn_q", QW, D), ("attn_k", HD, D), ("attn_v", HD, D), ("attn_output", D, QW), ("ffn_gate", FFN, D),
          ("ffn_up", FFN, D), ("ffn_down", D, FFN))
_NORMS = (("attn_norm", D), ("attn_q_norm", HD), ("attn_k_norm", HD), ("post_attention_norm", D), ("ffn_norm", D),
          ("post_ffw_norm", D))


def _weights(seed, blocks):
    """A random-init model of `blocks` decoder blocks: its tensor section on the device and its norms."""
    shapes = [(VOCAB, D)] + [(r, k) for _ in range(blocks) for _, r, k in _LAYER]
    arena, offs, views = _matrices(_generator(seed), shapes)
    rng = np.random.default_rng(seed)
    norms = [{n: (1.0 + 0.1 * rng.standard_normal(size)).astype(np.float32) for n, size in _NORMS} for _ in range(blocks)]
    out_norm = (1.0 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    return arena, offs, views, norms, out_norm


class Model(vrt.Gemma3):
    """The executor over a tensor section that is on the device already (vrt_g3_create)."""

    def __init__(self, ctx, seed, blocks):
        self.h = None
        self.ctx, self.arena = ctx, None
        self.blob, offs, _, norms, out_norm = _weights(seed, blocks)
        torch.cuda.synchronize()
        c = vrt.G3Config(CONTEXT, D, blocks, FFN, HEADS, 1, HD, HD, VOCAB, WINDOW, EPS, SHAPE["rope_global"], 1.0e4)
        layers = (vrt.G3Layer * blocks)()
        for l in range(blocks):
            for i, (name, _, _) in enumerate(_LAYER):
                setattr(layers[l], name, offs[1 + l * len(_LAYER) + i])
            for name, _ in _NORMS:
                setattr(layers[l], name, vrt.ptr(norms[l][name]))
        desc = vrt.G3Desc(c, self.blob.data_ptr(), self.blob.numel(), offs[0], vrt.ptr(out_norm), layers, 1)
        h = ctypes.c_void_p()
        vrt.check(vrt.lib().vrt_g3_create(ctx.h, ctypes.byref(desc), ctypes.byref(h)))
        self.h, self.config, self.kv_f16 = h.value, c, False
        self._batches = weakref.WeakSet()
        ctx._children.add(self)


def _ids(seed, *shape):
    return np.random.default_rng(seed + 7).integers(2, VOCAB, size=shape).astype(np.uint32)


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    s = {"ctx": ctx, "case": case}
    if kind in ("multi", "ffn", "matvec", "head"):
        gen, k = _generator(seed), case["k"]
        if kind == "multi":
            shapes = [(case[f"rows{i}"], k) for i in range(3)]
        elif kind == "ffn":
            shapes = [(case["ffn"], k), (case["ffn"], k), (case["out"], case["ffn"])]
        else:
            shapes = [(case["rows"], k)]
        arena, s["offs"], _ = _matrices(gen, shapes)
        s["dims"] = [r for r, _ in shapes]
        s["w"] = Span(arena)
        s["x"] = Span(torch.randn(k, generator=gen, device="cuda"))
        s["y"] = Span(torch.zeros(case["out"] if kind == "ffn" else sum(s["dims"]), device="cuda"))
        if kind == "ffn":
            s["ws"] = Span(torch.zeros(2 * case["ffn"], device="cuda"))
        if kind == "head":
            s["best"] = Span(torch.zeros(2, dtype=torch.int32, device="cuda"))
    elif kind == "codec":
        n = case["rows"] * case["k"]
        s["x"] = Span(torch.randn(n, generator=_generator(seed), device="cuda").mul_(0.02))
        s["q"] = Span(torch.zeros(n // 32 * 34, dtype=torch.uint8, device="cuda"))
        s["y"] = Span(torch.zeros(n, device="cuda"))
    else:
        s["model"] = Model(ctx, seed, case["blocks"])
        if case.get("kv", "f32") != "f32":
            s["model"].set_kv_format(case["kv"])
        if kind == "batch":
            s["batch"] = vrt.Gemma3Batch(s["model"], case["seqs"], 64)
            s["seqs"] = np.arange(case["seqs"], dtype=np.uint32)
            s["ids"] = _ids(seed, case["steps"], case["seqs"])
        else:
            s["ids"] = _ids(seed, case.get("prompt", 0) + case.get("steps", 0) + case.get("tokens", 0))
    torch.cuda.synchronize()
    return s


# ---- one pass -------------------------------------------------------------------------------

def run(s):
    ctx, case = s["ctx"], s["case"]
    kind = case["kind"]
    if kind == "multi":
        vrt.q8_matvec_multi(ctx, s["w"], s["offs"], s["dims"], case["k"], s["x"], s["y"])
        return s["y"].tensor
    if kind == "ffn":
        vrt.q8_ffn(ctx, s["w"], *s["offs"], case["k"], case["ffn"], case["out"], s["x"], s["ws"], s["y"])
        return {"y": s["y"].tensor, "workspace": s["ws"].tensor}
    if kind == "matvec":
        vrt.q8_matvec(ctx, s["w"], 0, s["x"], s["y"], case["k"], case["rows"])
        return s["y"].tensor
    if kind == "head":
        vrt.q8_matvec(ctx, s["w"], 0, s["x"], s["y"], case["k"], case["rows"])
        vrt.argmax(ctx, s["y"], case["rows"], s["best"])
        best = s["best"].tensor
        return {"logits": s["y"].tensor, "index": best[:1], "value": best[1:].view(torch.float32)}
    if kind == "codec":
        n = case["rows"] * case["k"]
        vrt.q8_quantize(ctx, s["x"], n, case["variant"], s["q"])
        vrt.q8_dequantize(ctx, s["q"], n // 32, s["y"])
        return {"blocks": s["q"].tensor, "values": s["y"].tensor}
    m, ids = s.get("model"), s["ids"]
    if kind == "decode":
        # the generate loop's steps with the tokens given, so that a near tie cannot fork two runs;
        # the last position leaves its logits
        n = case["steps"] - 1
        r = m.forced(ids[:n], 0)
        (index, value), hidden = m.decode(int(ids[n]), n, top_k=2, hidden=True)
        return {"index": np.append(r["index"], index).astype(np.int64), "value": np.append(r["value"], np.float32(value)),
                "hidden": hidden, "logits": m.logits()}
    if kind == "prefill":
        (index, value), hidden = m.prefill(ids, top_k=2, hidden=True)
        return {"value": np.float32(value), "hidden": hidden, "logits": m.logits()}
    if kind == "chat":
        n, values = case["prompt"], []
        (_, v), _ = m.prefill(ids[:n], top_k=1)
        values.append(v)
        for i in range(case["steps"] - 1):
            (_, v), _ = m.decode(int(ids[n + i]), n + i, top_k=1)
            values.append(v)
        (_, v), hidden = m.decode(int(ids[-1]), len(ids) - 1, top_k=2, hidden=True)
        values.append(v)
        return {"value": np.asarray(values, dtype=np.float32), "hidden": hidden, "logits": m.logits()}
    b, index, value = s["batch"], [], []
    b.reset()
    for t in range(case["steps"]):
        i, v = b.step(s["seqs"], ids[t])
        index.append(i)
        value.append(v)
    return {"index": np.stack(index).astype(np.int64), "value": np.stack(value), "logits": b.logits(case["seqs"] - 1)}


# ---- what a pass cannot do without -------------------------------------------------------------

def _q8(rows, k):
    return rows * k // 32 * 34


def _span(l, p):
    """Positions that block l's attention sees at position p."""
    return p + 1 if (l + 1) % 6 == 0 else min(p + 1, WINDOW)


def work(case):
    kind = case["kind"]
    if kind in ("multi", "matvec", "head"):
        rows = case["rows0"] + case["rows1"] + case["rows2"] if kind == "multi" else case["rows"]
        return {"bytes": _q8(rows, case["k"]) + 4 * (case["k"] + rows), "flops": 2 * rows * case["k"]}
    if kind == "ffn":
        k, f, o = case["k"], case["ffn"], case["out"]
        return {"bytes": 2 * _q8(f, k) + _q8(o, f) + 4 * (k + o + 2 * f), "flops": 4 * f * k + 2 * o * f}
    if kind == "codec":
        n = case["rows"] * case["k"]
        return {"bytes": 2 * (4 * n + n // 32 * 34), "flops": 4 * n}
    blocks = case["blocks"]
    kv = 4 if case.get("kv", "f32") == "f32" else 2
    per_block = sum(r * k for _, r, k in _LAYER)
    layers = blocks * (per_block // 32 * 34 + 4 * sum(n for _, n in _NORMS))
    head = _q8(VOCAB, D)

    def step(p):   # one decode step at position p
        seen = sum(_span(l, p) for l in range(blocks))
        return layers + head + 2 * seen * HD * kv, 2 * blocks * per_block + 2 * VOCAB * D + 4 * QW * seen

    def prefill(n):   # weights once, every position's keys and values once
        loc = sum(min(p + 1, WINDOW) for p in range(n))
        glo = n * (n + 1) // 2
        ng = blocks // 6
        seen = (blocks - ng) * loc + ng * glo
        return layers + head + 2 * blocks * n * HD * kv, 2 * n * blocks * per_block + 2 * VOCAB * D + 4 * QW * seen

    if kind == "decode":
        parts = [step(p) for p in range(case["steps"])]
    elif kind == "prefill":
        parts = [prefill(case["tokens"])]
    elif kind == "chat":
        parts = [prefill(case["prompt"])] + [step(case["prompt"] + i) for i in range(case["steps"])]
    else:
        parts, n = [], case["seqs"]
        for p in range(case["steps"]):
            by, fl = step(p)
            parts.append((by + (n - 1) * (by - layers - head), n * fl))
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    kind = case["kind"]
    if kind == "codec":
        return "exact"
    # about four times the distance from 64 bits that the paths show: 32-bit sums of up to 8192
    # products 2.4e-7, 32-bit arithmetic through 18 blocks 5e-6; with a 16-bit cache now and then a
    # key or value rounds the other way, 2.4e-5 (fp16) and 1.4e-4 (bf16) after a long prompt and
    # more after a short one
    if kind in ("multi", "matvec", "head", "ffn"):
        return {"rel": 1e-6, "max": 1e-5}
    if case.get("kv", "f32") == "bf16":
        return {"rel": 2e-3, "max": 2e-2, "differ": 0.01}
    if case.get("kv", "f32") == "f16":
        return {"rel": 4e-4, "max": 4e-3, "differ": 0.01}
    return {"rel": 4e-5, "max": 4e-4, "differ": 0.01}


# ---- the same in 64 bits ----------------------------------------------------------------------

def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + EPS) * w


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _rope_table(n, base):
    """cos and sin [n][HD / 2] as the model defines them: 32-bit frequencies, angles and entries."""
    e = (2.0 * np.arange(HD // 2, dtype=np.float32)) / np.float32(HD)
    inv = np.float32(1.0) / np.power(np.float64(base), e.astype(np.float64)).astype(np.float32)
    a = (np.arange(n, dtype=np.float32)[:, None] * inv[None, :]).astype(np.float64)
    return [torch.from_numpy(f(a).astype(np.float32)).cuda().double() for f in (np.cos, np.sin)]


def _rope(x, cs):
    c, s = cs
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _round_kv(x, kv):
    return x if kv == "f32" else x.float().to(torch.float16 if kv == "f16" else torch.bfloat16).double()


def _forward(seed, blocks, ids, kv):
    """Hidden states [B, T, D] after the output norm of the sequences ids [B, T], and the LM head."""
    _, _, views, norms, out_norm = _weights(seed, blocks)
    t64 = lambda a: torch.from_numpy(a).cuda().double()  # noqa: E731
    B, T = ids.shape
    emb = _dense(views[0], VOCAB, D)
    h = emb[torch.from_numpy(ids.astype(np.int64)).cuda()] * float(np.sqrt(np.float32(D)))
    tables = [_rope_table(T, 1.0e4), _rope_table(T, SHAPE["rope_global"])]
    pos = torch.arange(T, device="cuda")
    scale = 1.0 / float(np.sqrt(np.float32(HD)))
    for l in range(blocks):
        W = [_dense(views[1 + l * len(_LAYER) + i], r, k) for i, (_, r, k) in enumerate(_LAYER)]
        N = {n: t64(a) for n, a in norms[l].items()}
        glob = (l + 1) % 6 == 0
        x = _rms(h, N["attn_norm"])
        q = _rms((x @ W[0].t()).view(B, T, HEADS, HD), N["attn_q_norm"])
        k = _rms(x @ W[1].t(), N["attn_k_norm"])
        v = _round_kv(x @ W[2].t(), kv)
        k = _round_kv(_rope(k, tables[glob]), kv)
        att = torch.empty(B, T, QW, dtype=torch.float64, device="cuda")
        for i in range(HEADS):
            qi = _rope(q[:, :, i], tables[glob])
            for t0 in range(0, T, 2048):   # queries in runs: the score rows of a long prompt are large
                t1 = min(T, t0 + 2048)
                sc = torch.matmul(qi[:, t0:t1], k[:, :t1].transpose(1, 2).contiguous()) * scale
                see = pos[None, :t1] <= pos[t0:t1, None]
                if not glob:
                    see &= pos[None, :t1] + WINDOW > pos[t0:t1, None]
                sc.masked_fill_(~see, float("-inf"))
                att[:, t0:t1, i * HD:(i + 1) * HD] = torch.matmul(torch.softmax(sc, dim=-1), v[:, :t1])
        h = h + _rms(att @ W[3].t(), N["post_attention_norm"])
        x = _rms(h, N["ffn_norm"])
        h = h + _rms((_gelu(x @ W[4].t()) * (x @ W[5].t())) @ W[6].t(), N["post_ffw_norm"])
    return _rms(h, t64(out_norm)), emb


def _best(hidden, emb):
    """The largest logit of each row of hidden [n, D]."""
    return torch.cat([(hidden[i:i + 256] @ emb.t()).amax(dim=1) for i in range(0, hidden.shape[0], 256)])


def exact(case, seed):
    kind = case["kind"]
    if kind == "codec":
        return None
    if kind in ("multi", "ffn", "matvec", "head"):
        s = prepare(case, seed)
        x = s["x"].tensor.double()
        blk = lambda o, r, k: s["w"].tensor[o:o + _q8(r, k)].view(-1, 34)  # noqa: E731
        if kind == "ffn":
            k, f, o = case["k"], case["ffn"], case["out"]
            up = _dense(blk(s["offs"][1], f, k), f, k) @ x
            h = _gelu(_dense(blk(s["offs"][0], f, k), f, k) @ x) * up
            return {"y": _dense(blk(s["offs"][2], o, f), o, f) @ h, "workspace": torch.cat([h, up])}
        y = torch.cat([_dense(blk(o, r, case["k"]), r, case["k"]) @ x for o, r in zip(s["offs"], s["dims"])])
        return {"logits": y, "index": None, "value": y.amax().view(1)} if kind == "head" else y
    if kind == "batch":
        ids = np.ascontiguousarray(_ids(seed, case["steps"], case["seqs"]).T)
        h, emb = _forward(seed, case["blocks"], ids, "f32")
        best = _best(h.transpose(0, 1).reshape(-1, D), emb).view(case["steps"], case["seqs"])
        return {"index": None, "value": best, "logits": emb @ h[-1, -1]}
    ids = _ids(seed, case.get("prompt", 0) + case.get("steps", 0) + case.get("tokens", 0))
    h, emb = _forward(seed, case["blocks"], ids[None], case["kv"])
    last = h[0, -1]
    out = {"hidden": last, "logits": emb @ last}
    if kind == "decode":
        return {"index": None, "value": _best(h[0], emb), **out}
    if kind == "chat":
        return {"value": _best(h[0, case["prompt"] - 1:], emb), **out}
    return {"value": out["logits"].amax(), **out}
