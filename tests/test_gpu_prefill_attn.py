"""The prefill kernels (k_pf_qk, k_pf_attn and the batch around them) against
the device's own decode kernels, bit for bit: a prompt taken in as one batch
leaves the K and V rows of every layer and the normX that one forward per
token leaves (c2slm.go:103-114).  Layer 1's K and V rows are functions of
every token's layer-0 attention, so each token of a block is compared.

The decode side runs its chains in VALU fmas and is itself compared with the
oracle elsewhere; the batch runs them on v_mfma_f32_16x16x4_f32, so equal
bits here also pin the order and the single rounding per step that this
instruction is relied on for, with subnormal, infinite and NaN operands.
NaN results are compared as NaN: their sign and payload are those of the
operand the compiler put first."""
import numpy as np
import pytest

from c2slm_amd import _lib as H
from c2slm_amd import gguf as G

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


# blocks of 16 tokens, tiles of 16 positions, quads of 4, batches of 64
# (AV and sums); 2,340 positions is past 16 tokens' scores in LDS, 4,700
# past eight's
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


# k_pf_gemm_q50: 16 tokens per wave; 8, with the blocks of a row whole, in
# one round of two or four waves, and (4,864 columns) in five rounds
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
