"""Performance cases of the decode framework: the calls that its users make, at the sizes they make them.

A case is a dict of plain values with a ``kind``:

* ``matvec``   one weight-only matvec (``int8_gemv`` / ``fp8_gemv`` / ``int4_gemv``), weights resident;
* ``quantize`` one weight matrix quantized at load time (``quantize_per_channel`` / ``quantize_fp8`` /
  ``quantize_int4``);
* ``decode``   a whole 28-layer model from an empty cache: an 8-token prompt and greedy tokens after it,
  one ``decode_step`` call per token (the reference's loop) or one ``generate`` launch;
* ``longctx``  the INT8 model fed token by token behind a cache filled to a depth;
* ``prefill``  a prompt through the INT8 model's prompt-batched ``prefill``;
* ``batch``    up to 16 independent sequences of the 1.7B shape, one token each per step.

The framework has no entry point that returns logits: a decode step returns its token, and its
continuous results are the K and V rows it writes into every layer's cache (each layer's rows
depend on all the layers before it), so the model cases return those rows beside the tokens.
"""
from __future__ import annotations

import importlib
import math

import torch

mq = importlib.import_module("megaqwen-a10_amd")

DEV = "cuda"
V, D, NQ, NKV, EPS = 151936, 128, 16, 8, 1e-6
SHAPES = {"0.6b": (1024, 3072), "1.7b": (2048, 6144)}          # hidden, intermediate
LAYERS = 28
PROMPT = 8
# projection matrices [out, in] of the two model shapes; the fused ones as the matvec benchmark has them
MATRICES = [(4096, 1024), (1024, 2048), (6144, 1024), (1024, 3072),
            (4096, 2048), (2048, 2048), (12288, 2048), (2048, 6144)]


def listed():
    return [
        # the smallest call: the attention output projection of one layer, a few MB of weights
        {"name": "matvec_int8_o", "kind": "matvec", "format": "int8", "m": 1024, "k": 2048},
        # the largest matvec of a step: the LM head
        {"name": "matvec_int8_lm_head", "kind": "matvec", "format": "int8", "m": V, "k": 1024},
        # the fused gate and up projections in the format with the fewest bytes
        {"name": "matvec_int4_gate_up", "kind": "matvec", "format": "int4", "m": 6144, "k": 1024},
        # loading a checkpoint: its largest matrix through the quantizer
        {"name": "quantize_int8_lm_head", "kind": "quantize", "format": "int8", "m": V, "k": 1024},
        # the headline: greedy INT8 decoding, one call per token
        {"name": "decode_int8_steps", "kind": "decode", "format": "int8", "tokens": 32, "loop": "steps"},
        # the reference's unquantized path, a whole reply in one launch
        {"name": "generate_bf16", "kind": "decode", "format": "bf16", "tokens": 32, "loop": "launch"},
        # FP8 weights, a whole reply in one launch
        {"name": "generate_fp8", "kind": "decode", "format": "fp8", "tokens": 24, "loop": "launch"},
        # a long conversation goes on: attention over 8192 cached positions in every step
        {"name": "longctx_int8_8192", "kind": "longctx", "depth": 8192, "steps": 64},
        # a few users at once, an odd number of them
        {"name": "batch_3", "kind": "batch", "batch": 3, "steps": 32},
        # the batched decoder full
        {"name": "batch_16", "kind": "batch", "batch": 16, "steps": 32},
        # a chat message: a short ragged prompt
        {"name": "prefill_77", "kind": "prefill", "prompt": 77},
        # a page of text: one full prefill chunk
        {"name": "prefill_512", "kind": "prefill", "prompt": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "quantize", "decode", "longctx", "prefill", "prefill", "batch"])
    if kind in ("matvec", "quantize"):
        fmt = rng.choice(["int8", "int8", "fp8", "int4"])
        if rng.random() < 0.5:
            m, k = rng.choice(MATRICES)
            m -= rng.choice([0, 0, 1, 3, 17])                   # a shard, a pruned or an odd matrix
        else:
            m, k = _log_int(rng, 256, V), 128 * rng.randint(4, 8)
        return {"kind": kind, "format": fmt, "m": m, "k": k}
    if kind == "decode":
        return {"kind": kind, "format": rng.choice(["int8", "int8", "bf16", "fp8", "int4"]),
                "tokens": rng.randint(8, 48), "loop": rng.choice(["steps", "launch"])}
    if kind == "longctx":
        return {"kind": kind, "depth": _log_int(rng, 256, 8000), "steps": rng.randint(8, 48)}
    if kind == "prefill":
        return {"kind": kind, "prompt": _log_int(rng, 17, 1100)}
    return {"kind": kind, "batch": rng.randint(1, 16), "steps": rng.randint(8, 32)}


# ---- inputs ----------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _weight(g, shape):
    """Random-init weights of the benchmarks: N(0, 0.02) rounded to bf16."""
    return (torch.randn(shape, generator=g, device=DEV) * 0.02).to(torch.bfloat16)


def _gain(g, n):
    return (1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)).to(torch.bfloat16)


def _model_inputs(case, seed):
    """bf16 weights of the case's model in the packing order, and its token ids."""
    shape = "1.7b" if case["kind"] == "batch" else "0.6b"
    H, I = SHAPES[shape]
    g = _gen(seed)
    embed = _weight(g, (V, H))
    layers = []
    for _ in range(LAYERS):
        layers.append([_gain(g, H), _weight(g, (NQ * D, H)), _weight(g, (NKV * D, H)), _weight(g, (NKV * D, H)),
                       _gain(g, D), _gain(g, D), _weight(g, (H, NQ * D)), _gain(g, H),
                       _weight(g, (I, H)), _weight(g, (I, H)), _weight(g, (H, I))])
    final = _gain(g, H)
    n = {"decode": (PROMPT,), "longctx": (case.get("steps"),), "prefill": (case.get("prompt"),),
         "batch": (case.get("steps"), case.get("batch"))}[case["kind"]]
    tokens = torch.randint(0, V, n, generator=g, device=DEV).tolist()
    return H, I, embed, layers, final, tokens


def _seq_len(case):
    """Cache positions: the decoder's default of 2048, more where the case reaches past it."""
    if case["kind"] == "batch":
        return 256
    return max(2048, case.get("depth", 0) + case.get("steps", 0), case.get("prompt", 0) + 64)


def _projections():
    return (1, 2, 3, 6, 8, 9, 10)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("matvec", "quantize"):
        g = _gen(seed)
        w = _weight(g, (case["m"], case["k"]))
        if kind == "quantize":
            return {"case": case, "w": w}
        quant = {"int8": mq.quantize_per_channel, "fp8": mq.quantize_fp8, "int4": mq.quantize_int4}[case["format"]]
        q, s = quant(w)
        return {"case": case, "x": torch.randn(case["k"], generator=g, device=DEV), "q": q, "s": s}

    H, I, embed, layers, final, tokens = _model_inputs(case, seed)
    S = _seq_len(case)
    cos, sin = mq.precompute_rope_freqs(D, S, 1e6, device=DEV)
    fmt = case.get("format", "int8")
    if fmt == "bf16":
        dec = mq.A10MegakernelDecoder(embed, [t for l in layers for t in l], final, embed, cos, sin, LAYERS, S)
        return {"case": case, "dec": dec, "tokens": tokens}
    quant = {"int8": mq.quantize_per_channel, "fp8": mq.quantize_fp8, "int4": mq.quantize_int4}[fmt]
    flat, scales = [], []
    for l in layers:
        for i, t in enumerate(l):
            if i in _projections():
                t, s = quant(t)
                scales.append(s)
            flat.append(t)
    lm, lm_s = (mq.quantize_fp8 if fmt == "fp8" else mq.quantize_per_channel)(embed)
    cls = {"int8": mq.A10Int8MegakernelDecoder, "fp8": mq.A10Fp8MegakernelDecoder,
           "int4": mq.A10Int4MegakernelDecoder}[fmt]
    args = (embed, flat, scales, lm, lm_s, final, cos, sin, LAYERS, S)
    dec = mq.A10Int8BatchDecoder(*args, case["batch"]) if kind == "batch" else cls(*args)
    return {"case": case, "dec": dec, "tokens": tokens, "seed": seed}


# ---- one pass ----------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "matvec":
        f = {"int8": mq.int8_gemv, "fp8": mq.fp8_gemv, "int4": mq.int4_gemv}[case["format"]]
        return f(state["x"], state["q"], state["s"])
    if kind == "quantize":
        f = {"int8": mq.quantize_per_channel, "fp8": mq.quantize_fp8, "int4": mq.quantize_int4}[case["format"]]
        return f(state["w"])

    dec, tokens = state["dec"], state["tokens"]
    if kind == "decode":
        dec.reset()
        n = case["tokens"]
        if case["loop"] == "launch":
            out = dec.generate(tokens, n)
        else:
            for t in tokens:
                tok = dec.decode_step(t)
            out = [tok]
            while len(out) < n:
                tok = dec.decode_step(tok)
                out.append(tok)
        rows = slice(0, PROMPT + n - 1)
    elif kind == "longctx":
        dec.prefill_random_kv(case["depth"], seed=state["seed"])
        out = [dec.decode_step(t) for t in tokens]
        rows = slice(case["depth"], case["depth"] + case["steps"])
    elif kind == "prefill":
        dec.reset()
        dec.prefill(tokens)
        return {"k": dec.k_cache[:, :, :case["prompt"]], "v": dec.v_cache[:, :, :case["prompt"]]}
    else:
        dec.reset()
        out = [dec.decode_step(t) for t in tokens]
        return {"tokens": torch.tensor(out), "k": dec.k_cache[:, :, :, :case["steps"]],
                "v": dec.v_cache[:, :, :, :case["steps"]]}
    return {"tokens": torch.tensor(out), "k": dec.k_cache[:, :, rows], "v": dec.v_cache[:, :, rows]}


# ---- what a pass cannot do without ---------------------------------------------------------------
def _matrix_bytes(fmt, m, k):
    return {"int8": m * k + 4 * m, "fp8": m * k + 4 * m, "int4": m * k // 2 + m * k // 32, "bf16": 2 * m * k}[fmt]


def work(case):
    kind, fmt = case["kind"], case.get("format", "int8")
    if kind == "matvec":
        m, k = case["m"], case["k"]
        return {"bytes": _matrix_bytes(fmt, m, k) + 4 * (k + m), "flops": 2 * m * k}
    if kind == "quantize":
        m, k = case["m"], case["k"]
        return {"bytes": 2 * m * k + _matrix_bytes(fmt, m, k), "flops": 2 * m * k}
    H, I = SHAPES["1.7b" if kind == "batch" else "0.6b"]
    mats = [((NQ + 2 * NKV) * D, H), (H, NQ * D), (2 * I, H), (H, I)]
    layer = sum(_matrix_bytes(fmt, m, k) for m, k in mats) + 2 * (2 * H + 2 * D)
    layer_flops = 2 * sum(m * k for m, k in mats)
    head = _matrix_bytes("int8" if fmt == "int4" else fmt, V, H) + 2 * H
    row = LAYERS * 2 * NKV * D * 2                      # K and V of one position, all layers
    pair = LAYERS * 4 * NQ * D                          # operations of one query position against one cached one
    if kind == "prefill":
        P = case["prompt"]
        return {"bytes": LAYERS * layer + P * (2 * H + row), "flops": P * LAYERS * layer_flops + pair * P * (P + 1) // 2}
    first = case.get("depth", 0)
    steps = case["steps"] if "steps" in case else PROMPT + case["tokens"] - 1
    seqs = case.get("batch", 1)
    cached = sum(first + i + 1 for i in range(steps)) * seqs
    return {"bytes": steps * (LAYERS * layer + head + seqs * (2 * H + row)) + row * cached,
            "flops": seqs * steps * (LAYERS * layer_flops + 2 * V * H) + pair * cached}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    if case["kind"] == "matvec":
        return {"rel": 5e-7, "max": 5e-6}               # 32-bit sums: 1.2e-7 against 64 bits
    # one flipped bf16 rounding travels through all the layers and positions after it: against 64 bits the
    # batched steps and the 8192-position attention measure 8e-3, the other paths 0 (no rounding differs)
    return {"rel": 0.03 if case["kind"] in ("batch", "longctx") else 0.01, "max": 0.3, "differ": 0.01}


# ---- the same in 64 bits ---------------------------------------------------------------------------
def _quantized(w, fmt):
    """(codes, scales, dequantized float64 weight) of a bf16 matrix."""
    M, K = w.shape
    f = w.float()

    def over(a, n):                 # IEEE division (torch multiplies by the reciprocal of a scalar divisor)
        return a / torch.full_like(a, n)

    if fmt == "int8":
        s = over(f.abs().amax(1), 127.0).to(torch.bfloat16).float().clamp(min=1e-12)
        q = (f / s[:, None]).round().clamp(-128, 127)
        return q.to(torch.int8), s, q.double() * s.double()[:, None]
    if fmt == "fp8":
        s = over(f.abs().amax(1), 448.0).clamp(min=1e-12)
        q = (f / s[:, None]).to(torch.float8_e4m3fn)
        return q.view(torch.uint8), s, q.double() * s.double()[:, None]
    f = f.view(M, K // 128, 128)
    s = over(f.abs().amax(2), 7.0).to(torch.bfloat16).float().clamp(min=1e-12)
    q = (f / s[:, :, None]).round().clamp(-8, 7)
    d = (q.double() * s.double()[:, :, None]).view(M, K)
    q = q.view(M, K).to(torch.int32) & 15
    return (q[:, 0::2] | (q[:, 1::2] << 4)).to(torch.uint8), s, d


def _f32(x):
    return x.float().double()


def _bf16(x):
    return x.float().to(torch.bfloat16).double()


def _norm(x, gain):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gain


class _Model:
    """The decode step in float64, rounded where the reference stores a 32- or 16-bit value."""

    def __init__(self, case, seed):
        self.H, self.I, self.embed, layers, final, self.tokens = _model_inputs(case, seed)
        fmt = case.get("format", "int8")
        take = (lambda w: w.double()) if fmt == "bf16" else (lambda w: _quantized(w, fmt)[2])
        self.layers = [[take(t) if i in _projections() else t.double() for i, t in enumerate(l)] for l in layers]
        self.final = final.double()
        head = self.embed if fmt == "bf16" else None
        self.head = head.double() if head is not None else _quantized(self.embed, "fp8" if fmt == "fp8" else "int8")[2]
        S = _seq_len(case)
        inv = 1.0 / (1e6 ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
        freq = torch.arange(S, dtype=torch.float32)[:, None] * inv
        self.cos = freq.cos().to(torch.bfloat16).double().to(DEV)
        self.sin = freq.sin().to(torch.bfloat16).double().to(DEV)
        self.scale = float(torch.tensor(1.0 / math.sqrt(D), dtype=torch.float32))

    def cache(self, seqs, rows):
        shape = (seqs, LAYERS, NKV, rows, D)
        return torch.zeros(shape, dtype=torch.float64, device=DEV), torch.zeros(shape, dtype=torch.float64, device=DEV)

    def _rope(self, x, c, s):
        lo, hi = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([lo * c - hi * s, lo * s + hi * c], -1)

    def rows(self, tokens, pos, kc, vc):
        """Tokens of one sequence at positions pos, pos + 1, ...: fills their cache rows and gives the last hidden state."""
        P, T = len(tokens), pos + len(tokens)
        c, s = self.cos[pos:T, None], self.sin[pos:T, None]
        later = torch.arange(T, device=DEV)[None] > torch.arange(pos, T, device=DEV)[:, None]
        h = self.embed[torch.tensor(tokens, device=DEV)].double()
        for l, (in_ln, wq, wk, wv, qn, kn, wo, post, wg, wu, wd) in enumerate(self.layers):
            n = _f32(_norm(h, in_ln))
            q = _f32(n @ wq.T).view(P, NQ, D)
            k = _f32(n @ wk.T).view(P, NKV, D)
            v = _f32(n @ wv.T).view(P, NKV, D)
            q = _f32(self._rope(_norm(q, qn), c, s))
            kc[l, :, pos:T] = _bf16(_f32(self._rope(_norm(k, kn), c, s))).transpose(0, 1)
            vc[l, :, pos:T] = _bf16(v).transpose(0, 1)
            heads = []
            for j in range(NKV):                        # the two query heads of a KV head
                qj = q[:, 2 * j:2 * j + 2].transpose(0, 1).reshape(2 * P, D)
                a = (qj @ kc[l, j, :T].T.contiguous() * self.scale).view(2, P, T).masked_fill(later, -math.inf)
                heads += list((torch.softmax(a, -1).view(2 * P, T) @ vc[l, j, :T]).view(2, P, D))
            attn = _f32(torch.cat(heads, -1))
            x = _f32(attn @ wo.T + h)
            n2 = _f32(_norm(x, post))
            g = n2 @ wg.T
            m = _f32(g / (1.0 + torch.exp(-g)) * (n2 @ wu.T))
            h = _bf16(m @ wd.T + x)
        return h[-1]

    def token(self, h):
        return int(torch.argmax(self.head @ _f32(_norm(h, self.final))))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("matvec", "quantize"):
        g = _gen(seed)
        w = _weight(g, (case["m"], case["k"]))
        q, s, d = _quantized(w, case["format"])
        if kind == "quantize":
            return q, s
        return d @ torch.randn(case["k"], generator=g, device=DEV).double()

    model = _Model(case, seed)
    tokens = model.tokens
    if kind == "decode":
        n = case["tokens"]
        kc, vc = (t[0] for t in model.cache(1, PROMPT + n - 1))
        h, out = model.rows(tokens, 0, kc, vc), []
        while True:
            out.append(model.token(h))
            if len(out) == n:
                return {"tokens": torch.tensor(out), "k": kc, "v": vc}
            h = model.rows(out[-1:], PROMPT + len(out) - 1, kc, vc)
    if kind == "longctx":
        depth, T = case["depth"], case["depth"] + case["steps"]
        kc, vc = (t[0] for t in model.cache(1, T))
        g = _gen(seed)
        for cache in (kc, vc):
            for l in range(LAYERS):
                cache[l, :, :depth] = _bf16(torch.randn((NKV, depth, D), generator=g, device=DEV))
        out = [model.token(model.rows([t], depth + i, kc, vc)) for i, t in enumerate(tokens)]
        return {"tokens": torch.tensor(out), "k": kc[:, :, depth:], "v": vc[:, :, depth:]}
    if kind == "prefill":
        kc, vc = (t[0] for t in model.cache(1, case["prompt"]))
        model.rows(tokens, 0, kc, vc)
        return {"k": kc, "v": vc}
    kc, vc = model.cache(case["batch"], case["steps"])
    for b in range(case["batch"]):
        model.rows([step[b] for step in tokens], 0, kc[b], vc[b])
    return {"tokens": None, "k": kc, "v": vc}
