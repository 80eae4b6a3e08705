"""Performance cases of the packed-ternary BitNet b1.58 path on one MI355X.

Each case is one piece of work that a program using this framework has it do,
through the C ABI of `include/lbt.h` (the `lbt_hip` binding): the fused ternary
linears of a decode step, of a batched step and of a prefill, the tied bf16
and the int8 LM head, the device sampler, prefill layers, and whole requests
(prompt, then greedy decode), alone and batched.  Widths are those of the
BitNet b1.58 2B4T shape (hidden 2560, FFN 6912, 20 / 5 heads, vocab 128256, 30
layers) and generic odd ones.

listed() holds fixed cases, draw(rng) makes more of the same ranges,
prepare / run / work / tolerance / exact serve any of them.
"""
from __future__ import annotations

import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "lemonade-burn_amd"))
import lbt_hip  # noqa: E402

HIDDEN, FFN, KV, VOCAB, LAYERS, HEADS, KV_HEADS, MAX_POS = 2560, 6912, 640, 128256, 30, 20, 5, 4096
EPS, THETA = 1e-5, 500000.0
DEV = "cuda"


# ---- the cases -----------------------------------------------------------------


def linear(m, cols, *rows, name=None):
    """n fused ternary linears on one f32 input of m rows (quantized inside)."""
    c = {"kind": "linear", "m": m, "cols": cols, "n": len(rows)}
    c.update({"rows%d" % i: r for i, r in enumerate(rows)})
    return dict(c, name=name) if name else c


def listed():
    return [
        # the FFN products of one decoded token, gate / up and then down: the smallest calls, latency
        {"kind": "ffn", "m": 1, "name": "decode_ffn_1"},
        # q / k / v of a batched step of 13 sequences: a ragged few-token product
        linear(13, HIDDEN, HIDDEN, KV, KV, name="batch_qkv_13"),
        # two layers of another model on a 301-token prompt: columns that need padding, odd rows and tokens
        linear(301, 1000, 1503, 203, name="odd_301x1000"),
        # the down projection of a 2048-token prompt, the largest product of a long prefill
        linear(2048, FFN, HIDDEN, name="prefill_down_2048"),
        # logits of one token: the tied bf16 head, 657 MB
        {"kind": "head", "m": 1, "cols": HIDDEN, "rows": VOCAB, "name": "head_1"},
        # logits of the 24 sequences of a batched step
        {"kind": "head", "m": 24, "cols": HIDDEN, "rows": VOCAB, "name": "head_24"},
        # the opt-in int8 head for a small batch
        {"kind": "q8head", "m": 6, "cols": HIDDEN, "rows": VOCAB, "name": "q8head_6"},
        # one token each for four sampled requests, temperature and nucleus cut
        {"kind": "sample", "rows": 4, "vocab": VOCAB, "temperature": 0.8, "top_p": 0.95, "top_k": 0,
         "name": "sample_4"},
        # decoder layers over a long prompt (embedding, two layers, head of the last token)
        {"kind": "prefill", "layers": 2, "tokens": 2048, "vocab": 32000, "name": "prefill_layers_2048"},
        # one whole request: a 64-token prompt, 32 greedy tokens, then the next token's logits
        {"kind": "request", "tokens": 64, "steps": 32, "name": "request_64_32"},
        # a long-context request: a 3000-token prompt and a short answer
        {"kind": "request", "tokens": 3000, "steps": 8, "name": "request_3000_8"},
        # sixteen requests decoded together, prompts of 100 to 300 tokens, 24 greedy tokens each
        {"kind": "batch", "nseq": 16, "tokens": 300, "steps": 24, "name": "batch_16_24"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "head", "q8head", "sample", "prefill", "request", "batch"])
    if kind == "linear":
        if rng.random() < 0.2:
            return {"kind": "ffn", "m": _log(rng, 2, 512)}
        cols = rng.choice([HIDDEN, FFN, _log(rng, 100, 7000)])
        return linear(_log(rng, 1, 2048), cols, *[_log(rng, 64, 7000) for _ in range(rng.randint(1, 3))])
    if kind in ("head", "q8head"):
        return {"kind": kind, "m": _log(rng, 1, 64), "cols": rng.choice([HIDDEN, 8 * _log(rng, 16, 320)]),
                "rows": _log(rng, 4000, VOCAB)}
    if kind == "sample":
        return {"kind": "sample", "rows": _log(rng, 1, 16), "vocab": _log(rng, 4000, VOCAB),
                "temperature": rng.choice([0.0, 0.6, 0.8, 1.0]), "top_p": rng.choice([0.9, 0.95, 1.0]),
                "top_k": rng.choice([0, 0, 40])}
    if kind == "prefill":
        return {"kind": "prefill", "layers": rng.randint(1, 3), "tokens": _log(rng, 9, 2500),
                "vocab": _log(rng, 4000, 32000)}
    if kind == "batch":
        return {"kind": "batch", "nseq": rng.randint(2, 20), "tokens": _log(rng, 9, 250), "steps": rng.randint(4, 20)}
    return {"kind": "request", "tokens": _log(rng, 8, 1500), "steps": rng.randint(4, 24)}


# ---- preparation ---------------------------------------------------------------

_CTX = None


def _ctx():
    """The program's one device context."""
    global _CTX
    if _CTX is None:
        _CTX = lbt_hip.Ctx(0)
    return _CTX


def _gen(seed, tag):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + tag) & 0x7FFFFFFF)


def _activations(seed, m, cols):
    """Rows as a normed residual stream has them: normal values, a few channels far larger."""
    g = _gen(seed, 1)
    x = torch.randn(m, cols, generator=g, device=DEV)
    big = torch.randint(cols, (max(1, cols // 256),), generator=g, device=DEV)
    x[:, big] *= 12.0
    return x.contiguous()


def _ternary(seed, i, rows, cols):
    """Weights -1 / 0 / 1 with probabilities 0.3 / 0.4 / 0.3."""
    u = torch.rand(rows, cols, generator=_gen(seed, 10 + i), device=DEV)
    return (u > 0.7).to(torch.int8) - (u < 0.3).to(torch.int8)


def _pack(w):
    """The packed layout of include/lbt.h: 128-weight blocks of 32 bytes, bits 2k.. of byte j = w[32 k + j] + 1."""
    rows, cols = w.shape
    kp = lbt_hip.padded_cols(cols)
    code = torch.ones(rows, kp, dtype=torch.uint8, device=DEV)
    code[:, :cols] = (w + 1).to(torch.uint8)
    code = code.view(rows, kp // 128, 4, 32)
    p = code[:, :, 0] | (code[:, :, 1] << 2) | (code[:, :, 2] << 4) | (code[:, :, 3] << 6)
    return p.reshape(rows, kp // 4).contiguous()


def _calls(case):
    """(columns, rows of each matrix) of the case's linears, in their order."""
    if case["kind"] == "ffn":
        return [(HIDDEN, [FFN, FFN]), (FFN, [HIDDEN])]
    return [(case["cols"], [case["rows%d" % i] for i in range(case["n"])])]


def _wscale(cols):
    return float(np.float32(math.sqrt(0.6 * cols)))


def _bf16_matrix(seed, rows, cols):
    w = torch.rand(rows, cols, generator=_gen(seed, 30), device=DEV, dtype=torch.float32).mul_(2).sub_(1)
    return w.to(torch.bfloat16)


def _logits(seed, rows, vocab):
    """Logit rows as a language model gives them: a wide normal bulk and a few likely tokens."""
    g = _gen(seed, 40)
    x = torch.randn(rows, vocab, generator=g, device=DEV) * 2.5
    top = torch.randint(vocab, (rows, 24), generator=g, device=DEV)
    x.scatter_add_(1, top, 6.0 + 3.0 * torch.rand(rows, 24, generator=g, device=DEV))
    return x.contiguous()


def _p(t):
    return C.c_void_p(t.data_ptr())


class _Handle:
    """Frees what a state holds beside tensors and arrays."""

    def __init__(self, free):
        self._free = free

    def __del__(self):
        try:
            self._free()
        except Exception:
            pass


def _config(c):
    full = c["kind"] in ("request", "batch")
    return lbt_hip.make_config(layers=LAYERS if full else c["layers"], vocab=VOCAB if full else c["vocab"])


def prepare(case, seed):
    ctx, kind = _ctx(), case["kind"]
    lib = ctx.lib
    s = {"case": case, "ctx": ctx}
    if kind in ("linear", "ffn"):
        s["calls"], s["keep"], s["out"] = [], [], []
        at = 0
        for j, (cols, rows) in enumerate(_calls(case)):
            m, n = case["m"], len(rows)
            x = _activations(seed + j, m, cols)
            ws, outs = [], []
            for r in rows:
                packed = _pack(_ternary(seed, at, r, cols))
                torch.cuda.synchronize()  # the context's stream reads it
                h = C.c_void_p()
                ctx.check(lib.lbt_weight_upload_dev(ctx.h, _p(packed), r, cols, C.c_float(_wscale(cols)), C.byref(h)))
                ws.append(lbt_hip.Weight(ctx, h, r, cols, _wscale(cols)))
                outs.append(torch.empty(m, r, device=DEV))
                at += 1
            s["calls"].append(((C.c_void_p * n)(*[w.h for w in ws]), n, _p(x), m, cols,
                               (C.c_void_p * n)(*[o.data_ptr() for o in outs])))
            s["keep"].append((x, ws))
            s["out"] += outs
    elif kind in ("head", "q8head"):
        m, cols, rows = case["m"], case["cols"], case["rows"]
        s["x"] = torch.randn(m, cols, generator=_gen(seed, 1), device=DEV)
        s["out"] = torch.empty(m, rows, device=DEV)
        w = _bf16_matrix(seed, rows, cols).view(torch.int16).cpu().numpy().view(np.uint16)
        s["w"] = ctx.bf16_upload(w)
        if kind == "q8head":
            s["w"] = ctx.q8head_from_bf16(s["w"])
    elif kind == "sample":
        rows = case["rows"]
        s["logits"] = _logits(seed, rows, case["vocab"])
        s["seeds"] = torch.randint(1, 1 << 62, (rows,), generator=_gen(seed, 41), device=DEV)
        s["states"] = torch.empty_like(s["seeds"])
        s["out"] = torch.empty(rows, dtype=torch.int32, device=DEV)
        s["params"] = lbt_hip.LbtSampleParams(case["temperature"], case["top_p"], case["top_k"])
    else:
        s["model"] = lbt_hip.Model.synthetic(ctx, _config(case), int(seed) & 0xFFFFFFFF)
        s["owner"] = _Handle(s["model"].free)
        if kind == "batch":
            s["prompts"] = _prompts(case, seed)
            s["batch"] = s["model"].new_batch(case["nseq"], 1024)
            batch, model = s["batch"], s["model"]

            def free():
                batch.free()
                model.free()

            s["owner"]._free = free
        else:
            s["prompt"] = _prompt(case, seed)
    torch.cuda.synchronize()
    return s


def _prompt(case, seed):
    vocab = VOCAB if case["kind"] == "request" else case["vocab"]
    return np.random.default_rng(int(seed)).integers(0, vocab, case["tokens"]).astype(np.uint32)


def _prompts(case, seed):
    """One prompt per sequence, from a third of the case's tokens to all of them."""
    rng = np.random.default_rng(int(seed))
    lens = rng.integers(case["tokens"] // 3, case["tokens"] + 1, case["nseq"])
    return [rng.integers(0, VOCAB, n).astype(np.uint32) for n in lens]


# ---- one pass ------------------------------------------------------------------


def run(s):
    case, ctx = s["case"], s["ctx"]
    lib, kind = ctx.lib, case["kind"]
    if kind in ("linear", "ffn"):
        for call in s["calls"]:
            ctx.check(lib.lbt_ternary_linear_dev(ctx.h, *call))
        return s["out"]
    if kind == "head":
        ctx.check(lib.lbt_bf16_linear_dev(ctx.h, s["w"].h, _p(s["x"]), case["m"], _p(s["out"])))
        return s["out"]
    if kind == "q8head":
        ctx.check(lib.lbt_q8head_linear_dev(ctx.h, s["w"].h, _p(s["x"]), case["m"], _p(s["out"])))
        return s["out"]
    if kind == "sample":  # every request starts from its own seed
        rows = case["rows"]
        ctx.check(lib.lbt_memcpy_d2d(ctx.h, _p(s["states"]), _p(s["seeds"]), rows * 8))
        ctx.check(lib.lbt_sample_dev(ctx.h, _p(s["logits"]), rows, case["vocab"], C.byref(s["params"]),
                                     _p(s["states"]), _p(s["out"])))
        return {"ids": s["out"], "states": s["states"]}
    if kind == "batch":
        batch = s["batch"]
        first = np.empty(case["nseq"], np.uint32)
        for i, prompt in enumerate(s["prompts"]):  # a new request takes the slot
            ctx.check(lib.lbt_batch_reset(batch.h, i))
            first[i] = batch.prefill(i, prompt)
        tokens, _ = batch.decode_greedy(first, case["steps"])
        logits, _ = batch.forward(tokens[-1])
        return {"first": first.astype(np.int64), "tokens": tokens.astype(np.int64), "logits": logits}
    model = s["model"]
    cache = model.new_cache()
    try:
        logits = model.forward(s["prompt"], cache)
        if kind == "prefill":
            return logits
        tokens, _ = model.decode_greedy(cache, int(logits[0].argmax()), case["steps"])
        last = model.forward(tokens[-1:], cache)
        return {"prompt_logits": logits, "tokens": tokens.astype(np.int64), "logits": last}
    finally:
        cache.free()


# ---- what a pass cannot do without ----------------------------------------------


def _layer_bytes():
    return (2 * HIDDEN + 2 * KV) * HIDDEN // 4 + 3 * FFN * HIDDEN // 4


def _layer_ops(m, vis):
    """Operations of m tokens in one layer, `vis` visible keys summed over the tokens."""
    return 2.0 * m * 4 * _layer_bytes() + 4.0 * HIDDEN * vis


def work(case):
    kind = case["kind"]
    if kind in ("linear", "ffn"):
        m, calls = case["m"], [(cols, sum(rows)) for cols, rows in _calls(case)]
        return {"bytes": sum(r * lbt_hip.padded_cols(c) / 4 + 4.0 * m * (c + r) for c, r in calls),
                "flops": sum(2.0 * m * c * r for c, r in calls)}
    if kind in ("head", "q8head"):
        m, cols, rows = case["m"], case["cols"], case["rows"]
        w = 2.0 * rows * cols if kind == "head" else rows * (cols + 4.0)
        return {"bytes": w + 4.0 * m * (cols + rows), "flops": 2.0 * m * cols * rows}
    if kind == "sample":
        return {"bytes": case["rows"] * (4.0 * case["vocab"] + 20), "flops": 4.0 * case["rows"] * case["vocab"]}
    cfg = _config(case)
    n, layers, vocab = case["tokens"], cfg.num_hidden_layers, cfg.vocab_size
    kv_row = 2.0 * 2 * KV  # bytes of K and V of one position in one layer

    def forward(m, pos0, seqs=1):
        """m tokens after pos0 positions, or one token in each of `seqs` sequences."""
        vis = seqs * (m * pos0 + m * (m + 1) / 2)
        b = layers * (_layer_bytes() + seqs * kv_row * (pos0 + m)) + 2.0 * vocab * HIDDEN
        b += seqs * (2.0 * m * HIDDEN + 4.0 * vocab)
        return b, layers * _layer_ops(m * seqs, vis) + 2.0 * vocab * HIDDEN * seqs

    if kind == "batch":
        n, seqs = n * 2 // 3, case["nseq"]  # the mean prompt
        passes = [forward(n, 0)] * seqs + [forward(1, n + i, seqs) for i in range(case["steps"] + 1)]
    else:
        passes = [forward(n, 0)]
    if kind == "request":
        passes += [forward(1, n + i) for i in range(case["steps"] + 1)]
    return {"bytes": sum(p[0] for p in passes), "flops": sum(p[1] for p in passes)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear", "ffn"):
        # exact integers and one f32 product per output (6e-8 off 64 bits); an activation within
        # rounding of two codes takes either (6e-5 off at 2048 x 6912)
        return {"rel": 3e-4, "max": 0.05}
    if kind in ("head", "q8head"):  # f32 sums: 1.3e-7 off 64 bits
        return {"rel": 6e-7, "max": 1e-5}
    if kind == "sample":
        return "exact"
    # Activations quantized to 8 bits and K / V rounded to 16 in every layer: a last bit of one sum
    # moves a code or a 16-bit value by one step, and with these random weights a step of one of
    # the few large FFN values moves the logits by 1e-2 and more (two layers 0.024 off 64 bits,
    # thirty layers 0.06 .. 0.07).
    return {"rel": 0.03, "max": 0.4, "differ": 0.01}


# ---- the same in 64 bits ----------------------------------------------------------

_M1, _M2, _GOLD = -0x40A7B892E31B1A47, -0x6B2FB644ECCEEE15, -0x61C8864680B583EB


def _shr(z, k):
    return (z >> k) & ((1 << (64 - k)) - 1)


def _splitmix(z):
    z = z + _GOLD
    z = (z ^ _shr(z, 30)) * _M1
    z = (z ^ _shr(z, 27)) * _M2
    return z ^ _shr(z, 31)


def _draws(seed, tensor, n, at=0):
    """Draws at..at+n-1 of the synthetic model's tensor (one 64-bit word per element)."""
    base = _splitmix(torch.tensor((int(seed) & 0xFFFFFFFF) ^ (tensor << 40), device=DEV))
    return _splitmix(base + torch.arange(at, at + n, device=DEV))


def _synth_ternary(seed, tensor, rows, cols):
    b = _shr(_shr(_draws(seed, tensor, rows * cols), 32) * 10, 32)
    return ((b >= 7).to(torch.float64) - (b < 3).to(torch.float64)).view(rows, cols)


def _synth_unit(seed, tensor, n, at=0):
    return _shr(_draws(seed, tensor, n, at), 40).to(torch.float32) * 2.0**-24


def _quant(x):
    """ActQuant per row: the 8-bit codes, and the f32 scale they were made with."""
    x = x.to(torch.float32)
    s = 127.0 / x.abs().amax(-1, keepdim=True).clamp_min(1e-5)
    return (x * s).round().clamp(-128, 127).double(), s.double()


def _rms(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w


def _exact_prefill(case, seed):
    cfg = _config(case)
    tok = torch.from_numpy(_prompt(case, seed).astype(np.int64)).to(DEV)
    m, hd, g = len(tok), HIDDEN // HEADS, HEADS // KV_HEADS
    emb_at = torch.stack([_synth_unit(seed, 1, HIDDEN, int(t) * HIDDEN) for t in tok.tolist()])
    x = (emb_at * 2.0 - 1.0).to(torch.bfloat16).double()
    inv = torch.from_numpy((1.0 / THETA ** (np.arange(hd // 2) * 2 / hd)).astype(np.float32)).to(DEV)
    ang = (torch.arange(m, device=DEV, dtype=torch.float32)[:, None] * inv[None]).double()
    cos, sin = (torch.cat([f(ang)] * 2, -1).to(torch.float32).double() for f in (torch.cos, torch.sin))
    mask = torch.full((m, m), -math.inf, device=DEV, dtype=torch.float64).triu(1)

    def rope(v):  # [heads, m, hd]
        return v * cos + torch.cat([-v[..., hd // 2:], v[..., : hd // 2]], -1) * sin

    for l in range(cfg.num_hidden_layers):
        def lin(v, which, rows, cols):
            q, s = _quant(v)
            return q @ _synth_ternary(seed, 16 + 16 * l + which, rows, cols).T / (s * _wscale(cols))

        nw = [(0.5 + _synth_unit(seed, 16 + 16 * l + 7 + k, FFN if k == 3 else HIDDEN)).double() for k in range(4)]
        n1 = _rms(x, nw[0])
        q = rope(lin(n1, 0, HIDDEN, HIDDEN).view(m, HEADS, hd).transpose(0, 1))
        k = rope(lin(n1, 1, KV, HIDDEN).view(m, KV_HEADS, hd).transpose(0, 1)).to(torch.bfloat16).double()
        v = lin(n1, 2, KV, HIDDEN).view(m, KV_HEADS, hd).transpose(0, 1).to(torch.bfloat16).double()
        att = torch.empty(m, HEADS, hd, device=DEV, dtype=torch.float64)
        for h in range(HEADS):
            p = torch.softmax(q[h] @ k[h // g].T * hd**-0.5 + mask, -1)
            att[:, h] = p @ v[h // g]
        x = x + lin(_rms(att.reshape(m, HIDDEN), nw[2]), 3, HIDDEN, HIDDEN)
        n2 = _rms(x, nw[1])
        h = lin(n2, 4, FFN, HIDDEN).clamp_min(0).square() * lin(n2, 5, FFN, HIDDEN)
        x = x + lin(_rms(h, nw[3]), 6, HIDDEN, FFN)
    final = (0.5 + _synth_unit(seed, 2, HIDDEN)).double()
    y = _rms(x[-1:], final)
    out = []
    for r0 in range(0, cfg.vocab_size, 16384):
        rows = min(16384, cfg.vocab_size - r0)
        e = (_synth_unit(seed, 1, rows * HIDDEN, r0 * HIDDEN) * 2.0 - 1.0).to(torch.bfloat16)
        out.append(y @ e.double().view(rows, HIDDEN).T)
    return torch.cat(out, 1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear", "ffn"):
        out = []
        for j, (cols, rows) in enumerate(_calls(case)):
            q, s = _quant(_activations(seed + j, case["m"], cols))
            out += [q @ _ternary(seed, len(out) + i, r, cols).double().T / (s * _wscale(cols))
                    for i, r in enumerate(rows)]
        return out
    if kind in ("head", "q8head"):
        x = torch.randn(case["m"], case["cols"], generator=_gen(seed, 1), device=DEV).double()
        w = _bf16_matrix(seed, case["rows"], case["cols"])
        out = []
        for b in w.split(16384):
            b = b.float()
            if kind == "q8head":  # scale = amax / 127, codes to the nearest even
                sc = b.abs().amax(1, keepdim=True) / 127.0
                out.append((x @ (b / sc).round().clamp(-127, 127).double().T) * sc.double().T)
            else:
                out.append(x @ b.double().T)
        return torch.cat(out, 1)
    if kind == "prefill":
        return _exact_prefill(case, seed)
    if kind == "request":  # the tokens, and so the last logits, are the program's own choice
        return {"prompt_logits": _exact_prefill(case, seed), "tokens": None, "logits": None}
    return None  # whole numbers; and a batch's logits follow its own tokens
