"""What is timed when this package is made faster: calls that a program makes
through its public entry points, over the ranges that such a program uses.

Three kinds of case:

  op       one operator on device pointers (c2h_quantize_q8k_dev,
           c2h_gemv_dev, c2h_gemv_f32_dev) and the wait for it: what a
           program that runs single layers of its own pays per call
  decode   a forward of the last prompt token, greedy steps from there, and
           the logits after them: the generate loop at a context length
  prefill  a prompt (or a later turn of a session, pos > 0) taken in, and
           the logits after it: what stands before the first token

over the four layer shapes the package knows (Qwen2.5-0.5B with K-quant
projections and in the published file's formats, Qwen2.5-1.5B, Qwen3-1.7B).
Whole models run with all their layers and the full vocabulary where the
whole call is the point; the others run four layers of the real shape and a
vocabulary of 4,096, so that the layers are what is timed.

Every result of this package is a function of its inputs bit for bit (the
reference's arithmetic in the reference's order), so the tolerance is
"exact" throughout.  exact() is the same model in 64 bits, with the one
rounding that is part of the model itself: a K-quant matrix multiplies the
Q8_K quantisation of its input.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from c2slm_amd import _lib as H
from c2slm_amd import gguf as G

PENALTY = 1.15
MODELS = {
    "0.5b": G.QWEN05B,                        # K-quants throughout: Q8_K x int8 projections
    "0.5b-published": G.QWEN05B_REAL_FORMATS,  # Q5_0 / Q8_0 projections on f32 rows, Q6_K ffn_down
    "1.5b": G.QWEN25_1_5B,                    # head_dim 128, biases
    "1.7b-qwen3": G.QWEN3_1_7B,               # head_dim 128, QK-norm, 8 KV heads
}
TYPES = {"Q4_K": G.Q4_K, "Q6_K": G.Q6_K, "Q8_0": G.Q8_0, "Q5_0": G.Q5_0}
SMALL_VOCAB = 4096
MAX_CTX = 16384  # the package's default session length


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # The smallest call: the k projection of one decode step, input
        # quantised first; launch and wait are most of it.
        dict(name="op-k-proj-q4k", kind="op", op="gemv", type="Q4_K", rows=128, cols=896),
        # A full output projection without a worker pool on a f32 row: the
        # largest operator, a stream through memory.
        dict(name="op-vocab-f32-q8_0", kind="op", op="gemv_f32", type="Q8_0", rows=151936, cols=896),
        # A chat turn's reply, short context: the package's headline workload.
        dict(name="decode-0.5b-40", kind="decode", model="0.5b", layers=24, vocab=151936, pos=40, steps=16),
        # The same on the published file's formats, a few hundred tokens in.
        dict(name="decode-0.5b-published-300", kind="decode", model="0.5b-published", layers=24, vocab=151936,
             pos=300, steps=12),
        # A reply late in a long session.
        dict(name="decode-0.5b-4096", kind="decode", model="0.5b", layers=24, vocab=151936, pos=4096, steps=8),
        # Layers of the larger models: ordinary context, then a longer one.
        dict(name="decode-1.7b-qwen3-100", kind="decode", model="1.7b-qwen3", layers=4, vocab=SMALL_VOCAB, pos=100,
             steps=12),
        dict(name="decode-1.5b-1500", kind="decode", model="1.5b", layers=4, vocab=SMALL_VOCAB, pos=1500, steps=8),
        # A one-line question.
        dict(name="prefill-0.5b-37", kind="prefill", model="0.5b", layers=24, vocab=SMALL_VOCAB, pos=0, n=37),
        # A page of text.
        dict(name="prefill-0.5b-512", kind="prefill", model="0.5b", layers=24, vocab=SMALL_VOCAB, pos=0, n=512),
        # A paragraph, on the published file's formats.
        dict(name="prefill-0.5b-published-300", kind="prefill", model="0.5b-published", layers=24,
             vocab=SMALL_VOCAB, pos=0, n=300),
        # A document: several passes of the batch, long attention.
        dict(name="prefill-0.5b-3000", kind="prefill", model="0.5b", layers=4, vocab=SMALL_VOCAB, pos=0, n=3000),
        # A system prompt on a head_dim-128 model.
        dict(name="prefill-1.7b-qwen3-400", kind="prefill", model="1.7b-qwen3", layers=4, vocab=SMALL_VOCAB, pos=0,
             n=400),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case: operators over rows, columns and formats; decode over
    context lengths; prompts over lengths, some of them a later turn."""
    kind = rng.choice(["op", "decode", "prefill", "prefill"])
    if kind == "op":
        op = rng.choice(["gemv", "gemv_f32"])
        ty = rng.choice(sorted(TYPES))
        # Q8_0 and Q5_0 rows of c2h_gemv_dev go up to 1,024 columns; ragged
        # widths keep whole blocks only, as the operators define
        hi = 1024 if (op == "gemv" and ty in ("Q8_0", "Q5_0")) else 11008
        return dict(kind="op", op=op, type=ty, rows=_log(rng, 1, 12000), cols=_log(rng, 256, hi))
    model = rng.choice(sorted(MODELS))
    wide = MODELS[model].head_dim == 128
    layers = rng.randint(2, 4)
    if kind == "decode":
        pos = _log(rng, 2, 2000 if wide else 6000)
        return dict(kind="decode", model=model, layers=layers, vocab=SMALL_VOCAB, pos=pos, steps=rng.randint(3, 8))
    n = _log(rng, 1, 350 if wide else 2000)
    pos = rng.choice([0, 0, _log(rng, 1, 600 if wide else 2500)])
    return dict(kind="prefill", model=model, layers=layers, vocab=SMALL_VOCAB, pos=pos, n=n)


# ------------------------------------------------------------- models, inputs

# Offset of the fp16 scale in a block, and the standard deviation of the
# unscaled weights that SYNTH draws.
SCALE = {G.Q4_K: (0, 167.0), G.Q6_K: (208, 674.0), G.Q8_0: (0, 73.3), G.Q5_0: (0, 9.23)}


def _matrix(rng, tt, rows, cols):
    """Blocks of a matrix as trained weights have them: centred, of standard
    deviation about 1/sqrt(cols), so that activations stay of order one and
    attention spreads over the context."""
    qk, bs = G.BLOCK[tt]
    raw = G.SYNTH[tt](rng, rows * (cols // qk))
    b = raw.reshape(-1, bs)
    at, std = SCALE[tt]
    d = rng.uniform(0.5, 1.5, len(b)) / (std * math.sqrt(cols))
    b[:, at:at + 2] = d.astype(np.float16).reshape(-1, 1).view(np.uint8)
    if tt == G.Q4_K:  # the mins are the scales and dmin 7.5 d: quants 0..15 about their middle
        b[:, 2:4] = (7.5 * d).astype(np.float16).reshape(-1, 1).view(np.uint8)
        b[:, 8:12] = b[:, 4:8]
        b[:, 12:16] = (b[:, 12:16] & 15) * 17
    return raw


@functools.lru_cache(maxsize=2)
def _weights(model, layers, vocab):
    """(layer, role, ggml type, rows, cols, host bytes) of every tensor: the
    model file, the same for every seed of the inputs."""
    s = MODELS[model]
    rng = np.random.default_rng([20261201, sorted(MODELS).index(model), layers, vocab])
    E, F, KV = s.n_embd, s.n_ff, s.n_kv_heads * s.head_dim
    out = []

    def quant(layer, role, tt, rows, cols):
        out.append((layer, role, tt, rows, cols, _matrix(rng, tt, rows, cols)))

    def f32(layer, role, v):
        out.append((layer, role, G.F32, 1, len(v), np.asarray(v, np.float32)))

    quant(0, "TOKEN_EMBD", s.t_embd, vocab, E)
    f32(0, "OUTPUT_NORM", rng.uniform(0.5, 1.5, E))
    for i in range(layers):
        f32(i, "ATTN_NORM", rng.uniform(0.5, 1.5, E))
        quant(i, "ATTN_Q", s.t_q, E, E)
        quant(i, "ATTN_K", s.t_k, KV, E)
        quant(i, "ATTN_V", s.t_v, KV, E)
        if s.arch == "qwen3":
            f32(i, "ATTN_Q_NORM", rng.uniform(0.5, 1.5, s.head_dim))
            f32(i, "ATTN_K_NORM", rng.uniform(0.5, 1.5, s.head_dim))
        else:
            for role, n in (("ATTN_Q_BIAS", E), ("ATTN_K_BIAS", KV), ("ATTN_V_BIAS", KV)):
                f32(i, role, rng.normal(0.0, 0.02, n))
        quant(i, "ATTN_OUT", s.t_o, E, E)
        f32(i, "FFN_NORM", rng.uniform(0.5, 1.5, E))
        quant(i, "FFN_GATE", s.t_gate, F, E)
        quant(i, "FFN_UP", s.t_up, F, E)
        quant(i, "FFN_DOWN", s.t_down, E, F)
    return out


def _special(vocab):
    """(im_end, eos)"""
    return (151645, 151643) if vocab > 151645 else (vocab - 1, vocab - 3)


def _tokens(case, seed):
    """Token ids of positions 0 .. (all that the case reads)."""
    n = case["pos"] + case.get("n", 0)
    return np.random.default_rng([seed, 1]).integers(0, case["vocab"], n).astype(np.int32)


FILLED = 512  # contexts beyond this start from a restored cache of N(0,1) keys and values


def _cached(case):
    """Positions in hand before the call (a decode runs its last prompt token again)."""
    return case["pos"] - 1 if case["kind"] == "decode" else case["pos"]


def _restored_kv(case, seed):
    """[2][layers][kv heads][positions][head_dim] of a restored session, on the GPU."""
    s = MODELS[case["model"]]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 13)
    return torch.randn((2, case["layers"], s.n_kv_heads, _cached(case), s.head_dim), generator=g, device="cuda")


def _op_input(case, seed):
    rng = np.random.default_rng([seed, 2])
    tt = TYPES[case["type"]]
    w = _matrix(rng, tt, case["rows"], case["cols"])
    return tt, w, rng.normal(0.0, 1.0, case["cols"]).astype(np.float32)


# ------------------------------------------------------------ prepare and run

def prepare(case, seed):
    if case["kind"] == "op":
        tt, w, x = _op_input(case, seed)
        rows, cols = case["rows"], case["cols"]
        packed = torch.from_numpy(H.pack_weights(tt, rows, cols, w)).cuda()
        kq = case["op"] == "gemv" and tt in (G.Q4_K, G.Q6_K)
        st = dict(case=case, tt=tt, ctx=H.Ctx(), w=packed, x=torch.from_numpy(x).cuda(),
                  y=torch.zeros(rows, device="cuda"),
                  q=torch.zeros(cols // 256 * 292, dtype=torch.uint8, device="cuda") if kq else None)
        torch.cuda.synchronize()
        return st
    s = MODELS[case["model"]]
    d = H.ModelDesc()
    d.n_layers, d.n_vocab, d.max_ctx = case["layers"], case["vocab"], MAX_CTX
    d.n_embd, d.n_heads, d.n_kv_heads, d.head_dim, d.n_ff = s.n_embd, s.n_heads, s.n_kv_heads, s.head_dim, s.n_ff
    d.rms_eps, d.rope_theta = s.rms_eps, s.rope_theta
    ctx = H.Ctx(d)
    for layer, role, tt, rows, cols, data in _weights(case["model"], case["layers"], case["vocab"]):
        ctx.upload(layer, role, tt, rows, cols, data)
    toks = _tokens(case, seed)
    n = _cached(case)
    if n > FILLED:
        kv = _restored_kv(case, seed).cpu().numpy()
        for which in range(2):
            for layer in range(case["layers"]):
                for h in range(s.n_kv_heads):
                    ctx.set_kv(which, layer, h, 0, kv[which, layer, h])
        ctx.set_token_ids(0, toks[:n])
        ctx.set_seq(n)
    elif n > 0:
        ctx.prefill(toks[:n], 0)
    return dict(case=case, ctx=ctx, tokens=toks)


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "op":
        lib = H.lib()
        ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        rows, cols, tt = case["rows"], case["cols"], state["tt"]
        if case["op"] == "gemv_f32":
            rc = lib.c2h_gemv_f32_dev(ctx.h, tt, ptr(state["w"]), ptr(state["x"]), rows, cols, ptr(state["y"]))
        else:
            rc, x = 0, state["x"]
            if state["q"] is not None:
                rc, x = lib.c2h_quantize_q8k_dev(ctx.h, ptr(x), cols, ptr(state["q"])), state["q"]
            rc = rc or lib.c2h_gemv_dev(ctx.h, tt, ptr(state["w"]), ptr(x), rows, cols, ptr(state["y"]), None)
        rc = rc or lib.c2h_sync(ctx.h)  # y is read on another stream than the context's
        if rc:
            raise H.C2hError(rc, case["op"])
        return dict(y=state["y"]) if state["q"] is None else dict(y=state["y"], q8k=state["q"])
    toks, pos = state["tokens"], case["pos"]
    if case["kind"] == "prefill":
        normx = ctx.prefill(toks[pos:], pos)
        return dict(normx=normx, logits=ctx.logits())
    im_end, eos = _special(case["vocab"])
    first = ctx.forward(int(toks[pos - 1]), pos - 1)
    out = [ctx.step(pos + i, PENALTY, im_end, eos) for i in range(case["steps"])]
    return dict(first=first, tokens=np.array(out, np.int32), normx=ctx.normx(), logits=ctx.logits())


# --------------------------------------------------------- work and tolerance

def _row_bytes(tt, cols):
    qk, bs = G.BLOCK[tt]
    return cols // qk * bs


def _used(tt, cols):
    qk = G.BLOCK[tt][0]
    return cols // qk * qk


def _layer(s):
    """(weight bytes, multiply-adds per token) of one layer's projections."""
    E, F, KV = s.n_embd, s.n_ff, s.n_kv_heads * s.head_dim
    mats = [(s.t_q, E, E), (s.t_k, KV, E), (s.t_v, KV, E), (s.t_o, E, E), (s.t_gate, F, E), (s.t_up, F, E),
            (s.t_down, E, F)]
    return sum(r * _row_bytes(t, c) for t, r, c in mats), sum(r * _used(t, c) for t, r, c in mats)


def work(case):
    if case["kind"] == "op":
        tt, rows, cols = TYPES[case["type"]], case["rows"], case["cols"]
        return dict(bytes=rows * _row_bytes(tt, cols) + 4 * cols + 4 * rows, flops=2 * rows * _used(tt, cols))
    s, pos = MODELS[case["model"]], case["pos"]
    wb, macs = _layer(s)
    vb, vmacs = case["vocab"] * _row_bytes(s.t_embd, s.n_embd), case["vocab"] * s.n_embd
    kvb = 2 * s.n_kv_heads * s.head_dim * 4  # bytes of K and V per position and layer
    if case["kind"] == "prefill":
        # the weights once, the cache read and written once, one row of logits
        n = case["n"]
        pairs = n * pos + n * (n + 1) // 2
        b = case["layers"] * (wb + (pos + n) * kvb) + vb + 4 * case["vocab"]
        f = case["layers"] * (2 * macs * n + 4 * pairs * s.n_embd) + 2 * vmacs
        return dict(bytes=b, flops=f)
    # every step is a pass of its own over weights and cache
    b = f = 0
    for i in range(case["steps"] + 1):
        T = pos + i
        b += case["layers"] * (wb + T * kvb) + vb
        f += case["layers"] * (2 * macs + 4 * T * s.n_embd) + 2 * vmacs
    return dict(bytes=b + 4 * case["vocab"], flops=f)


def tolerance(case):
    return "exact"


# -------------------------------------------------------------- in 64 bits

def _dequant(tt, raw, rows, cols):
    """[rows, whole blocks] in 64 bits, on the GPU."""
    qk, bs = G.BLOCK[tt]
    b = torch.from_numpy(np.ascontiguousarray(raw)).cuda().view(rows * (cols // qk), bs)

    def half(o):
        return b[:, o:o + 2].contiguous().view(torch.float16).double()

    if tt == G.Q8_0:
        w = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif tt == G.Q5_0:
        sh = torch.arange(8, device="cuda", dtype=torch.uint8)
        hi = ((b[:, 2:6].unsqueeze(2) >> sh) & 1).reshape(-1, 32)
        lo = torch.cat([b[:, 6:] & 15, b[:, 6:] >> 4], 1)
        w = half(0) * ((lo | (hi << 4)).double() - 16)
    elif tt == G.Q4_K:
        p = b[:, 4:16]
        sc = torch.cat([p[:, 0:4] & 63, (p[:, 8:12] & 15) | ((p[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([p[:, 4:8] & 63, (p[:, 8:12] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        w = (half(0) * sc).unsqueeze(2) * q - (half(2) * mn).unsqueeze(2)
    else:  # Q6_K
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        hi = torch.cat([(qh >> (2 * k)) & 3 for k in range(4)], 2)
        q = (lo | (hi << 4)).reshape(-1, 16, 16).double() - 32
        w = (half(208) * b[:, 192:208].contiguous().view(torch.int8).double()).unsqueeze(2) * q
    return w.reshape(rows, -1)


def _q8k(x):
    """The Q8_K rounding of rows of 256-element blocks."""
    v = x[..., :x.shape[-1] // 256 * 256].float().reshape(*x.shape[:-1], -1, 256)
    amax = v.abs().amax(-1, keepdim=True)
    t = v * torch.where(amax > 1e-30, 127.0 / amax, torch.zeros_like(amax))
    q = torch.trunc(t + torch.copysign(torch.full_like(t, 0.5), t))
    return ((amax / 127.0).double() * q.double()).flatten(-2)


class _Exact:
    """The model in 64 bits."""

    def __init__(self, case):
        self.s, self.layers = MODELS[case["model"]], [{} for _ in range(case["layers"])]
        self.top = {}
        for layer, role, tt, rows, cols, raw in _weights(case["model"], case["layers"], case["vocab"]):
            m = (tt, torch.from_numpy(raw).cuda().double() if tt == G.F32 else _dequant(tt, raw, rows, cols))
            (self.top if role in ("TOKEN_EMBD", "OUTPUT_NORM") else self.layers[layer])[role] = m
        kv = [torch.zeros((self.s.n_kv_heads, 0, self.s.head_dim), dtype=torch.float64, device="cuda")] * 2
        self.kv = [list(kv) for _ in self.layers]

    def mul(self, m, x):
        tt, w = m
        return (_q8k(x) if tt in (G.Q4_K, G.Q6_K) else x) @ w.t().contiguous()

    def norm(self, x, w):
        return x / torch.sqrt(x.square().mean(-1, keepdim=True) + float(np.float32(self.s.rms_eps))) * w[1]

    def rope(self, x, pos):  # [positions, heads, head_dim]
        hd = self.s.head_dim
        f = self.s.rope_theta ** (-2.0 * torch.arange(hd // 2, dtype=torch.float64, device="cuda") / hd)
        a = (pos.double().unsqueeze(1) * f).unsqueeze(1)
        u, v = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([u * a.cos() - v * a.sin(), u * a.sin() + v * a.cos()], -1)

    def forward(self, toks, pos0):
        """normX of the last of `toks`, the first of which stands at pos0."""
        s, n, hd = self.s, len(toks), self.s.head_dim
        pos = torch.arange(pos0, pos0 + n, device="cuda")
        x = self.top["TOKEN_EMBD"][1][torch.as_tensor(np.asarray(toks), dtype=torch.long, device="cuda")]
        for L, kv in zip(self.layers, self.kv):
            a = self.norm(x, L["ATTN_NORM"])
            q, k, v = (self.mul(L["ATTN_" + r], a) + (L["ATTN_" + r + "_BIAS"][1] if "ATTN_" + r + "_BIAS" in L else 0)
                       for r in "QKV")
            q, k, v = (t.reshape(n, -1, hd) for t in (q, k, v))
            if "ATTN_Q_NORM" in L:
                q, k = self.norm(q, L["ATTN_Q_NORM"]), self.norm(k, L["ATTN_K_NORM"])
            q, k = self.rope(q, pos), self.rope(k, pos)
            for i, new in enumerate((k, v)):
                kv[i] = torch.cat([kv[i][:, :pos0], new.transpose(0, 1)], 1)
            per = s.n_heads // s.n_kv_heads
            mask = torch.arange(pos0 + n, device="cuda") > pos.unsqueeze(1)
            heads = []
            for h in range(s.n_heads):
                sc = q[:, h] @ kv[0][h // per].t().contiguous() / math.sqrt(hd)
                heads.append(torch.softmax(sc.masked_fill(mask, -math.inf), -1) @ kv[1][h // per])
            x = x + self.mul(L["ATTN_OUT"], torch.cat(heads, -1))
            a = self.norm(x, L["FFN_NORM"])
            g, u = self.mul(L["FFN_GATE"], a), self.mul(L["FFN_UP"], a)
            x = x + self.mul(L["FFN_DOWN"], g * torch.sigmoid(g) * u)
        return self.norm(x[-1], self.top["OUTPUT_NORM"])

    def logits(self, normx):
        return self.top["TOKEN_EMBD"][1] @ normx  # Q8_0: the f32 row as it is


def exact(case, seed):
    if case["kind"] == "op":
        tt, w, x = _op_input(case, seed)
        kq = case["op"] == "gemv" and tt in (G.Q4_K, G.Q6_K)
        x = torch.from_numpy(x).cuda()
        x = _q8k(x) if kq else x.double()
        W = _dequant(tt, w, case["rows"], case["cols"])
        y = W @ x[:W.shape[1]]
        return dict(y=y, q8k=None) if kq else dict(y=y)
    m, toks, pos, n = _Exact(case), _tokens(case, seed), case["pos"], _cached(case)
    if n > FILLED:
        kv = _restored_kv(case, seed).double()
        m.kv = [[kv[0, i], kv[1, i]] for i in range(case["layers"])]
    elif n > 0:
        m.forward(toks[:n], 0)
    if case["kind"] == "prefill":
        x = m.forward(toks[pos:], pos)
        return dict(normx=x, logits=m.logits(x))
    # the greedy stream after it turns on differences that 32 bits do not
    # tell apart, and what follows from it has no value of its own
    return dict(first=m.forward(toks[pos - 1:pos], pos - 1), tokens=None, normx=None, logits=None)
