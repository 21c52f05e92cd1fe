"""Prompts and decode steps take, at each size, the kernels that suit it: the
time of one against that of like work, with a bound between what the two
routes measure, and bit for bit what one forward per token leaves."""
import time

import numpy as np
import pytest

from c2slm_amd import _lib as H
from c2slm_amd import gguf as G

pytestmark = pytest.mark.gpu


def best_us(f, reps=7):
    t = []
    for _ in range(reps):
        t0 = time.perf_counter()
        f()
        t.append(time.perf_counter() - t0)
    return min(t) * 1e6


def open_model(path, shape, max_ctx, seed=71):
    G.write_synthetic_model(str(path), shape, seed=seed)
    gf = G.GGUFFile(str(path))
    ctx = H.Ctx(H.desc_from_gguf(gf, max_ctx=max_ctx))
    H.load_gguf_into(ctx, gf)
    return ctx


def fill(ctx, s, n, seed=72):
    kv = np.random.default_rng(seed).standard_normal((n, s.head_dim)).astype(np.float32)
    for which in range(2):
        for layer in range(s.n_layers):
            for h in range(s.n_kv_heads):
                ctx.set_kv(which, layer, h, 0, np.roll(kv, 17 * (which + 2 * layer + 5 * h), 0))


def check_prompt(ctx, s, toks, pos0):
    """normX, and K and V of every layer from pos0 on, as one forward per token leaves them."""
    n = pos0 + len(toks)
    got = ctx.prefill(toks, pos0)
    kv = [ctx.kv(w, layer, h, n)[pos0:] for w in (0, 1) for layer in range(s.n_layers) for h in range(s.n_kv_heads)]
    for i, t in enumerate(toks):
        want = ctx.forward(int(t), pos0 + i)
    ref = [ctx.kv(w, layer, h, n)[pos0:] for w in (0, 1) for layer in range(s.n_layers) for h in range(s.n_kv_heads)]
    for a, b in zip([got, *kv], [want, *ref]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


# Prompts late in a session: few tokens, and any number once a workgroup's
# LDS holds one token's scores, run the decode's long-context kernels.

LATE = 15700


@pytest.fixture(scope="module")
def late(tmp_path_factory):
    s = G.ModelShape(n_layers=2, n_vocab=2048)
    ctx = open_model(tmp_path_factory.mktemp("late") / "m.gguf", s, 16384)
    fill(ctx, s, LATE)
    yield s, ctx
    ctx.close()


# what the context adds to a prompt, in units of what it adds to a forward
# (whose attention is the same three launches for one token): 0.9, 1.3 and 21
# measured; with a workgroup per head and block of tokens 3.9, 4.3 and 59
@pytest.mark.parametrize("n,most", [(1, 2.0), (16, 2.7), (256, 44.0)])
def test_late_prompts_keep_up_with_decode(late, n, most):
    s, ctx = late
    toks = np.random.default_rng(n).integers(0, s.n_vocab, n).astype(np.int32)
    more = best_us(lambda: ctx.prefill(toks, LATE)) - best_us(lambda: ctx.prefill(toks, 100))
    one = best_us(lambda: ctx.forward(5, LATE)) - best_us(lambda: ctx.forward(5, 100))
    print(n, more, one, more / one, flush=True)
    assert more < most * one


# one sub-launch whole and in part, several with a part; an ordinary prompt
# beside them (37 tokens at 4,000 stay with k_pf_attn)
@pytest.mark.parametrize("pos0,n", [(1024, 1), (3000, 16), (4000, 5), (4000, 37), (7000, 17), (LATE, 37), (LATE, 1)])
def test_late_prompts_equal_forwards(late, pos0, n):
    s, ctx = late
    print(pos0, n, flush=True)
    check_prompt(ctx, s, np.random.default_rng(pos0 + n).integers(0, s.n_vocab, n).astype(np.int32), pos0)
    fill(ctx, s, LATE)


# Q5_0 projections of few tokens: a block per thread (k_pf_gemm_q50s,
# k_pf_gemm_f) where k_pf_gemm_q50's waves would wait out a load per block.

Q50 = dict(n_layers=2, n_vocab=2048, t_q=G.Q5_0, t_k=G.Q5_0, t_v=G.Q8_0, t_o=G.Q5_0, t_gate=G.Q5_0, t_up=G.Q5_0)


# the same prompt with Q5_0 matrices and with others beside them: rows of 28
# blocks against Q8_0 (a small FFN, so that q|k and o are much of the pass):
# 1.23 measured, 1.89 with k_pf_gemm_q50 for all; rows of 152 blocks against
# Q6_K: below 1, 1.52
@pytest.mark.parametrize("kind,n,most", [("narrow", 8, 1.5), ("wide", 1, 1.2)])
def test_few_q5_0_tokens_keep_up(kind, n, most, tmp_path):
    if kind == "narrow":
        a, b = (dict(Q50, n_ff=768, t_q=t, t_k=t, t_o=t, t_gate=t, t_up=t, t_down=t) for t in (G.Q5_0, G.Q8_0))
    else:
        a, b = (dict(Q50, t_down=t) for t in (G.Q5_0, G.Q6_K))
    us = []
    for i, kw in enumerate((a, b)):
        s = G.ModelShape(**dict(kw, n_layers=6))
        with open_model(tmp_path / f"{i}.gguf", s, 512) as ctx:
            toks = np.random.default_rng(n).integers(0, s.n_vocab, n).astype(np.int32)
            us.append(best_us(lambda: ctx.prefill(toks, 0), 9))
    print(kind, us, us[0] / us[1], flush=True)
    assert us[0] < most * us[1]


# each kernel's tokens and tiles, and the lines between them: 16 tokens per
# k_pf_gemm_q50s workgroup and 1,000 of those a launch (145 tokens of q|k,
# 17 of gate|up); 7 tokens of wide rows; ffn_down rows of 24, 32, 33 (a
# workgroup's 7 rows leave threads over), 152 and 280 blocks (past the 256 of
# a decode workgroup's threads)
@pytest.mark.parametrize("n_ff", [768, 1024, 1056, 4864, 8960])
@pytest.mark.parametrize("n", [1, 7, 8, 16, 17, 128, 145])
def test_q5_0_prompts_equal_forwards(n_ff, n, tmp_path):
    s = G.ModelShape(**dict(Q50, n_ff=n_ff, t_down=G.Q5_0))
    with open_model(tmp_path / "m.gguf", s, 256) as ctx:
        print(n_ff, n, flush=True)
        check_prompt(ctx, s, np.random.default_rng(n).integers(0, s.n_vocab, n).astype(np.int32), 0)


# Decode attention at head_dim 128 past the split: no slower than the one
# launch it replaces there (0.82 measured; with a workgroup per group of heads
# 1.13).

def test_h128_two_launches_no_slower_than_one(tmp_path, monkeypatch):
    s = G.ModelShape(n_layers=2, n_embd=1536, n_heads=12, n_kv_heads=2, n_ff=8960, n_vocab=2048)
    ctxs = []
    for split in (None, "2047"):
        if split is not None:
            monkeypatch.setenv("C2H_ATT_SPLIT", split)
        ctxs.append(open_model(tmp_path / "m.gguf", s, 2048))
        fill(ctxs[-1], s, 530)
        ctxs[-1].set_seq(520)
    two, one = np.min([[c.time_layer_kernel("attn", 200, True) * 1e3 for c in ctxs] for _ in range(6)], axis=0)
    print(two, one, two / one, flush=True)
    for c in ctxs:
        c.close()
    assert two < 1.05 * one
