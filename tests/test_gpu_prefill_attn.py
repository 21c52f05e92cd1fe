"""The prefill kernels (k_pf_qk, k_pf_attn and the batch around them) against
the device's own decode kernels, bit for bit: a prompt taken in as one batch
leaves the K and V rows of every layer and the normX that one forward per
token leaves (c2slm.go:103-114).  Layer 1's K and V rows are functions of
every token's layer-0 attention, so each token of a block is compared.

The decode side is itself compared with the oracle, here and elsewhere.  It
runs its chains in VALU fmas, but for head_dim 128 past 512 positions; the
batch runs them on v_mfma_f32_16x16x4_f32, so equal bits here also pin the
order and the single rounding per step that this instruction is relied on
for, with subnormal, infinite and NaN operands.  Where decode runs them on
that instruction too, the batch and the decode are each compared with the
oracle.  NaN results are compared as NaN: their sign and payload are those of the
operand the compiler put first."""
import os

import numpy as np
import pytest

from c2slm_amd import _lib as H
from c2slm_amd import gguf as G
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = {
    "hd64": G.ModelShape(n_layers=2, n_vocab=2048),
    "hd64-formats": G.ModelShape(n_layers=2, n_vocab=2048, t_q=G.Q5_0, t_k=G.Q5_0, t_v=G.Q8_0, t_o=G.Q5_0,
                                 t_gate=G.Q5_0, t_up=G.Q5_0),
    "hd64-1536": G.ModelShape(n_layers=2, n_embd=1536, n_heads=24, n_kv_heads=4, n_ff=1536, n_vocab=2048),
    "hd128-qknorm": G.ModelShape(n_layers=2, n_embd=2048, n_heads=16, n_kv_heads=8, n_ff=6144, n_vocab=2048,
                                 arch="qwen3"),
    "hd128-biases": G.ModelShape(n_layers=2, n_embd=1536, n_heads=12, n_kv_heads=2, n_ff=8960, n_vocab=2048),
}
MAX_CTX = 6000


@pytest.fixture(scope="module", params=list(SHAPES))
def model(request, tmp_path_factory):
    p = str(tmp_path_factory.mktemp("pfa") / "m.gguf")
    G.write_synthetic_model(p, SHAPES[request.param], seed=91)
    gf = G.GGUFFile(p)
    ctx = H.Ctx(H.desc_from_gguf(gf, max_ctx=MAX_CTX))
    H.load_gguf_into(ctx, gf)
    yield SHAPES[request.param], gf, ctx
    ctx.close()


def same(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return (a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))


def all_kv(ctx, s, n):
    return [ctx.kv(w, l, h, n) for w in (0, 1) for l in (0, 1) for h in range(s.n_kv_heads)]


def fill(ctx, s, n, rng, edit=lambda which, kv: None):
    """n positions of N(0,1) keys and values in both layers."""
    for which in (0, 1):
        for layer in (0, 1):
            for h in range(s.n_kv_heads):
                kv = rng.normal(0, 1, (n, s.n_embd // s.n_heads)).astype(np.float32)
                if layer == 0:
                    edit(which, kv)
                ctx.set_kv(which, layer, h, 0, kv)


def compare(ctx, s, toks, pos0):
    n = pos0 + len(toks)
    nx = ctx.prefill(toks, pos0)
    kv = all_kv(ctx, s, n)
    for p, t in enumerate(toks):  # (two-launch attention past 512 positions at head_dim 128)
        want = ctx.forward(int(t), pos0 + p)
    for got, ref in zip(kv, all_kv(ctx, s, n)):
        ok = same(got, ref)
        assert ok.all(), np.argwhere(~ok)[:4]
    assert same(nx, want).all()


# tiles of 16 positions, quads of 4, batches of 64 (AV and sums), in blocks of
# four tokens: these prompts are too short for more to fill the GPU.  At
# head_dim 64 the last runs the long-context kernels; at head_dim 128 one and
# two tokens run the forwards themselves.
@pytest.mark.parametrize("pos0,n", [(0, 1), (0, 2), (0, 3), (0, 16), (0, 17), (3, 33), (63, 1), (62, 37), (127, 20), (300, 75),
                                    (505, 12),
                                    (1000, 30), (2340, 18), (4700, 9)])
def test_prefill_equals_forwards(model, pos0, n):
    s, _, ctx = model
    print(s.n_embd, s.n_heads, pos0, n, flush=True)
    rng = np.random.default_rng(pos0 * 1000 + n)
    fill(ctx, s, max(pos0, 1), rng)
    compare(ctx, s, rng.integers(0, s.n_vocab, n).astype(np.int32), pos0)


@pytest.mark.parametrize("kind", ["subnormal", "inf-v", "nan-v", "nan-k0", "inf-k"])
def test_special_rows(model, kind):
    s, _, ctx = model
    rng = np.random.default_rng(17)

    def edit(which, kv):
        if kind == "subnormal":  # products and sums in the subnormal range
            kv *= np.float32(1e-3 if which == 0 else 2e-39)
        elif which == 1 and kind == "inf-v":
            kv[10, 5], kv[31, 6] = np.inf, -np.inf
        elif which == 1 and kind == "nan-v":
            kv[10, 5] = np.nan
        elif which == 0 and kind == "nan-k0":  # a NaN score 0 makes the max NaN
            kv[0] = np.nan
        elif which == 0 and kind == "inf-k":
            kv[12, 3] = -np.inf

    fill(ctx, s, 45, rng, edit)
    compare(ctx, s, rng.integers(0, s.n_vocab, 20).astype(np.int32), 45)


def test_non_finite_token_leaves_earlier_tokens(model):
    """A token whose embedding holds a NaN: where the projections read f32
    rows its K and V rows are NaN (the Q8_K quantiser makes numbers of them),
    and the tokens before it in the same block are untouched by them."""
    s, gf, ctx = model
    emb = gf.tensor_map["token_embd.weight"]
    raw = np.array(emb.data)
    row = s.n_embd // 32 * 34
    bad = raw.copy()
    bad[7 * row:7 * row + 2] = (0x00, 0x7e)  # fp16 NaN scale
    rng = np.random.default_rng(23)
    toks = rng.integers(100, s.n_vocab, 14).astype(np.int32)
    toks[9] = 7
    try:
        ctx.upload(0, "TOKEN_EMBD", G.Q8_0, s.n_vocab, s.n_embd, bad)
        compare(ctx, s, toks, 0)
        v0, k1 = ctx.kv(1, 0, 0, 14), ctx.kv(0, 1, 0, 14)
        before, own = bool(np.isfinite(k1[:9]).all()), bool(np.isnan(v0[9]).any())
        assert before and own == (s.t_v == G.Q8_0)
    finally:
        ctx.upload(0, "TOKEN_EMBD", G.Q8_0, s.n_vocab, s.n_embd, raw)


# k_pf_gemm_q50: 16 tokens per wave; 8, with the blocks of a row whole, in one
# round of two or four waves, and (4,864 columns) in five rounds.  5 and 100
# tokens run k_pf_gemm_q50s for q|k and o, 5 with 4,864 columns k_pf_gemm_f.
@pytest.mark.parametrize("down", [G.Q6_K, G.Q5_0])
@pytest.mark.parametrize("n", [5, 100, 150, 260])
def test_q5_0_prompts(down, n, tmp_path):
    s = G.ModelShape(n_layers=2, n_vocab=2048, t_q=G.Q5_0, t_k=G.Q5_0, t_v=G.Q8_0, t_o=G.Q5_0, t_gate=G.Q5_0,
                     t_up=G.Q5_0, t_down=down)
    G.write_synthetic_model(str(tmp_path / "m.gguf"), s, seed=92)
    gf = G.GGUFFile(str(tmp_path / "m.gguf"))
    with H.Ctx(H.desc_from_gguf(gf, max_ctx=512)) as ctx:
        H.load_gguf_into(ctx, gf)
        print("q5_0", down, n, flush=True)
        compare(ctx, s, np.random.default_rng(n).integers(0, s.n_vocab, n).astype(np.int32), 0)


# ---- each block size, and each reason for it

def block_tokens(heads, m, pmax):
    """k_pf_attn's tokens per workgroup and whether it stages K
    (pf_attn_tokens, pfa_lds_bytes)."""
    def lds(tb, stage):
        return tb * ((pmax + 1 + 63) // 64 * 64 + 4) * 4 + (8 * 16 * 68 * 4 if stage else 0)

    tb = 16
    while tb > 4 and heads * -(-m // tb) < 256:
        tb //= 2
    while tb > 1 and lds(tb, True) > 156 * 1024:
        tb //= 2
    return tb, lds(tb, True) <= 156 * 1024


def long_launches(s, m, pmax, tb):
    """Whether the long-context launches take the pass instead (pf_attn_split)."""
    T = pmax + 1
    whole = 8000 + -(-s.n_heads * -(-m // tb) // 256) * 18.2 * T
    split = -(-m // 16) * (18000 + 4.8 * T) + m * s.n_kv_heads * (220 + 0.07 * T)
    return s.head_dim == 64 and T > 1024 and split < 0.95 * whole


# 345 tokens fill the GPU in blocks of 16 at 12 heads and more; 1,919, 3,839
# and 7,743 are the last positions that leave 16, 8 and 4 tokens' scores room
@pytest.mark.parametrize("pos0,n,tb", [(131, 345, 16), (1570, 350, 16), (1571, 350, 8), (3489, 351, 8), (3490, 351, 4),
                                       (0, 350, 16), (510, 200, 8)])
def test_block_sizes(model, pos0, n, tb):
    s, _, ctx = model
    if (pos0, n) == (510, 200):  # (8 by the number of workgroups: 12 and 14 heads)
        tb = 8 if s.n_heads < 20 else 16
    assert block_tokens(s.n_heads, n, pos0 + n - 1) == (tb, True)
    assert not long_launches(s, n, pos0 + n - 1, tb)
    print(s.n_embd, s.n_heads, pos0, n, flush=True)
    rng = np.random.default_rng(pos0 * 1000 + n)
    fill(ctx, s, max(pos0, 1), rng)
    compare(ctx, s, rng.integers(0, s.n_vocab, n).astype(np.int32), pos0)


# a last pass of one and two tokens
@pytest.mark.parametrize("n", [513, 514])
def test_short_last_pass(model, n):
    s, _, ctx = model
    compare(ctx, s, np.random.default_rng(n).integers(0, s.n_vocab, n).astype(np.int32), 0)


def special(kind):
    def edit(which, kv):
        if kind == "subnormal":
            kv *= np.float32(1e-3 if which == 0 else 2e-39)
        elif which == 1 and kind == "inf-v":
            kv[10, 5], kv[31, 6] = np.inf, -np.inf
        elif which == 1 and kind == "nan-v":
            kv[10, 5] = np.nan
        elif which == 0 and kind == "nan-k0":
            kv[0] = np.nan
        elif which == 0 and kind == "inf-k":
            kv[12, 3] = -np.inf
    return edit


KINDS = ["subnormal", "inf-v", "nan-v", "nan-k0", "inf-k"]


@pytest.mark.parametrize("kind", KINDS)
def test_special_rows_blocks_of_16(model, kind):
    s, _, ctx = model
    assert block_tokens(s.n_heads, 345, 45 + 344) == (16, True)
    rng = np.random.default_rng(18)
    fill(ctx, s, 45, rng, special(kind))
    compare(ctx, s, rng.integers(0, s.n_vocab, 345).astype(np.int32), 45)


def test_non_finite_token_in_a_block_of_16(model):
    s, gf, ctx = model
    raw = np.array(gf.tensor_map["token_embd.weight"].data)
    row = s.n_embd // 32 * 34
    bad = raw.copy()
    bad[7 * row:7 * row + 2] = (0x00, 0x7e)  # fp16 NaN scale
    toks = np.random.default_rng(24).integers(100, s.n_vocab, 345).astype(np.int32)
    toks[203] = 7
    assert block_tokens(s.n_heads, 345, 344) == (16, True)
    try:
        ctx.upload(0, "TOKEN_EMBD", G.Q8_0, s.n_vocab, s.n_embd, bad)
        compare(ctx, s, toks, 0)
        assert np.isfinite(ctx.kv(0, 1, 0, 345)[:203]).all()
    finally:
        ctx.upload(0, "TOKEN_EMBD", G.Q8_0, s.n_vocab, s.n_embd, raw)


# ---- two, one and one unstaged token per workgroup: past 7,743, 15,551 and
# 31,167 positions, up to the longest session.  Head_dim 128 against the
# oracle; head_dim 64 with sixteen KV heads (few enough query heads for each
# that k_pf_attn keeps the prompt) against the decode's long-context kernels.

def test_head_dim_128_late_positions(tmp_path):
    s = SHAPES["hd128-biases"]
    G.write_synthetic_model(str(tmp_path / "m.gguf"), s, seed=93)
    gf = G.GGUFFile(str(tmp_path / "m.gguf"))
    ctx, orc = H.Ctx(H.desc_from_gguf(gf, max_ctx=38848)), O.OracleEngine(gf, max_ctx=38848, n_threads=16)
    H.load_gguf_into(ctx, gf)
    rng = np.random.default_rng(94)
    view = orc.kv_view()
    rows = rng.standard_normal((38848, 128), dtype=np.float32)
    for which in (0, 1):
        for layer in (0, 1):
            for h in (0, 1):
                view[which, layer, h, :38848] = np.roll(rows, 13 * (which + 2 * layer + 5 * h), 0)
                ctx.set_kv(which, layer, h, 0, view[which, layer, h, :38848])
    for pos0, n, want in ((7741, 6, (2, True)), (15549, 5, (1, True)), (31166, 5, (1, False)), (38845, 3, (1, False))):
        assert block_tokens(s.n_heads, n, pos0 + n - 1) == want
        print(pos0, n, flush=True)
        toks = rng.integers(0, s.n_vocab, n).astype(np.int32)
        orc.set_seq_len(pos0)
        got, ref = ctx.prefill(toks, pos0), orc.ingest_from(pos0, toks)
        assert same(got, ref).all(), pos0
        for which in (0, 1):
            for h in (0, 1):
                assert same(ctx.kv(which, 1, h, pos0 + n)[pos0:], view[which, 1, h, pos0:pos0 + n]).all(), pos0
    ctx.close()
    orc.close()


def test_head_dim_64_late_positions(tmp_path):
    s = G.ModelShape(n_layers=2, n_embd=1024, n_heads=16, n_kv_heads=16, n_ff=1024, n_vocab=2048)
    G.write_synthetic_model(str(tmp_path / "m.gguf"), s, seed=95)
    gf = G.GGUFFile(str(tmp_path / "m.gguf"))
    rng = np.random.default_rng(96)
    rows = rng.standard_normal((36864, 64), dtype=np.float32)
    with H.Ctx(H.desc_from_gguf(gf, max_ctx=36864)) as ctx:
        H.load_gguf_into(ctx, gf)
        for which in (0, 1):
            for layer in (0, 1):
                for h in range(16):
                    ctx.set_kv(which, layer, h, 0, np.roll(rows, 13 * (which + 2 * layer + 5 * h), 0))
        for pos0, n, want in ((7741, 16, (2, True)), (15549, 16, (1, True)), (31166, 16, (1, False)),
                              (36848, 16, (1, False))):
            assert block_tokens(s.n_heads, n, pos0 + n - 1) == want
            assert not long_launches(s, n, pos0 + n - 1, want[0])
            print(pos0, n, flush=True)
            toks = rng.integers(0, s.n_vocab, n).astype(np.int32)
            got = ctx.prefill(toks, pos0)
            kv = [ctx.kv(w, 1, h, pos0 + n)[pos0:] for w in (0, 1) for h in range(16)]
            for i, tok in enumerate(toks):
                ref = ctx.forward(int(tok), pos0 + i)
            assert same(got, ref).all(), pos0
            for a, b in zip(kv, [ctx.kv(w, 1, h, pos0 + n)[pos0:] for w in (0, 1) for h in range(16)]):
                assert same(a, b).all(), pos0


# ---- head_dim-128 decode past the split (k_attn_h128_scores, _sav) against
# the oracle, the split moved down: every remainder of the quads, the edges of
# the 16-position tiles and of a workgroup's 64, of four batches of V (256)

@pytest.fixture(scope="module", params=["hd128-qknorm", "hd128-biases"])
def split_pair(request, tmp_path_factory):
    s = SHAPES[request.param]
    p = str(tmp_path_factory.mktemp("split") / "m.gguf")
    G.write_synthetic_model(p, s, seed=97)
    gf = G.GGUFFile(p)
    old = os.environ.get("C2H_ATT_SPLIT")
    os.environ["C2H_ATT_SPLIT"] = "1"
    try:
        ctx = H.Ctx(H.desc_from_gguf(gf, max_ctx=600))
    finally:
        if old is None:
            del os.environ["C2H_ATT_SPLIT"]
        else:
            os.environ["C2H_ATT_SPLIT"] = old
    H.load_gguf_into(ctx, gf)
    orc = O.OracleEngine(gf, max_ctx=600, n_threads=16)
    yield s, ctx, orc
    ctx.close()
    orc.close()


def decode_against_oracle(s, ctx, orc, pos, steps, edit=lambda which, kv: None):
    rng = np.random.default_rng(pos)
    view = orc.kv_view()
    for which in (0, 1):
        for layer in (0, 1):
            for h in range(s.n_kv_heads):
                kv = rng.normal(0, 1, (max(pos, 1), s.head_dim)).astype(np.float32)
                if layer == 0:
                    edit(which, kv)
                view[which, layer, h, :len(kv)] = kv
                ctx.set_kv(which, layer, h, 0, kv)
    for i in range(steps):
        tok = int(rng.integers(0, s.n_vocab))
        assert same(ctx.forward(tok, pos + i), orc.forward(tok, pos + i)).all(), pos + i
    for which in (0, 1):
        for h in range(s.n_kv_heads):
            got = ctx.kv(which, 1, h, pos + steps)[pos:]
            assert same(got, view[which, 1, h, pos:pos + steps]).all(), (which, h)


@pytest.mark.parametrize("pos,steps", [(0, 20), (29, 6), (60, 8), (125, 6), (253, 6), (510, 6), (573, 6)])
def test_h128_split_decode(split_pair, pos, steps):
    s, ctx, orc = split_pair
    print(s.n_embd, pos, flush=True)
    decode_against_oracle(s, ctx, orc, pos, steps)


@pytest.mark.parametrize("kind", KINDS)
def test_h128_split_decode_special_rows(split_pair, kind):
    s, ctx, orc = split_pair
    print(s.n_embd, kind, flush=True)
    decode_against_oracle(s, ctx, orc, 45, 5, special(kind))
    decode_against_oracle(s, ctx, orc, 300, 4, special(kind))
