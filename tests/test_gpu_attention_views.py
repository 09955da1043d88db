"""Decode attention at the edges of its views: as many positions as a wave holds and one more or less,
the longest view of one launch and the first that is split, and the cached rows behind the position.

A decode step of a short-context model requests rows of the cache past its position before it knows the
position and drops them; the step must come out as if those rows held zeros, whatever they hold.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    import aesir_hip

    return aesir_hip


def f64_attention(q, K, V, hd, nq, nkv):
    """Output, and sum of probability times |V|, per query head and dim."""
    g = np.arange(nq) // (nq // nkv)
    qd = q.astype(np.float64).reshape(nq, hd)
    Kd, Vd = (x.astype(np.float64).reshape(-1, nkv, hd)[:, g] for x in (K, V))
    s = np.einsum("hd,shd->hs", qd, Kd) / np.sqrt(hd)
    p = np.exp(s - s.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    top = np.einsum("hd,shd->hs", np.abs(qd), np.abs(Kd)).max() / np.sqrt(hd)
    return np.einsum("hs,shd->hd", p, Vd).reshape(-1), np.einsum("hs,shd->hd", p, np.abs(Vd)).reshape(-1), top


# positions per wave 64 up to head_dim 32, 32 above; one launch up to 512 positions, 256 at head_dim 128
# (a decode step of head_dim 64 and 128: 96 and 128 cache rows, then rounds of 64 positions up to these)
VIEWS = {8: (1, 63, 64, 65, 511, 512, 513), 16: (1, 63, 64, 65, 511, 512, 513), 32: (1, 63, 64, 65, 511, 512, 513),
         64: (1, 31, 32, 33, 63, 64, 65, 511, 512, 513), 128: (1, 31, 32, 33, 127, 128, 129, 255, 256, 257)}


@pytest.mark.parametrize("hd,offset", [(8, 0), (16, 0), (32, 0), (64, 0), (128, 0), (8, 1), (16, 1), (32, 1)])
def test_view_edges(A, hd, offset):
    """offset 1: keys 2 bytes into an allocation (the kernels without 16-byte loads). The bound is one f16
    rounding of the output, and the f32 rounding of the dot products (each off by at most hd 2^-24 of the
    sum of |products|), probabilities and sums, doubled."""
    rng = np.random.default_rng(hd)
    for S in VIEWS[hd]:
        for nq, nkv in ((8, 2), (4, 4)):
            q = rng.standard_normal((1, nq * hd)).astype(np.float16)
            K, V = (rng.standard_normal((S, nkv * hd)).astype(np.float16) for _ in range(2))
            with A.Context(32 << 20) as ctx:
                kb = ctx.from_numpy(np.concatenate([np.zeros(offset, np.float16), K.reshape(-1)]).reshape(1, -1))
                out = ctx.tensor(1, nq * hd)
                A.flash_attention_gqa(ctx, ctx.from_numpy(q), kb.view(S, nkv * hd, offset), ctx.from_numpy(V), out, S, hd, nq, nkv)
                got = out.numpy().reshape(-1).astype(np.float64)
            want, mass, top = f64_attention(q, K, V, hd, nq, nkv)
            ulp = np.spacing(np.abs(want).astype(np.float16)).astype(np.float64)
            bound = ulp + ((hd + 8) * (1 + top) + S) * 2.0 ** -23 * mass
            assert np.all(np.abs(got - want) <= bound), (S, nq, nkv, float((np.abs(got - want) - bound).max()))


@pytest.mark.parametrize("heads,kv,hd,ctx_len", [(8, 4, 8, 200), (8, 4, 8, 512), (8, 2, 16, 140), (4, 2, 32, 200),
                                                 (4, 1, 64, 64), (4, 1, 64, 96), (4, 1, 64, 97), (4, 1, 64, 200), (4, 2, 64, 700),
                                                 (4, 4, 128, 64), (4, 4, 128, 128), (4, 1, 128, 128), (4, 1, 128, 200)])
def test_rows_behind_the_position_do_not_count(A, oracle, heads, kv, hd, ctx_len):
    """The cache behind the position holds infinities and NaN (steps of a token whose K and V overflow);
    the steps before them, on both sides of a wave's last position, equal those on a zeroed cache bit for
    bit."""
    dim = heads * hd
    cfg = oracle.Config(dim=dim, n_layers=2, n_heads=heads, n_kv_heads=kv, ffn=2 * dim, vocab=64, ctx_len=ctx_len)
    w = oracle.synthetic_weights(cfg, 3, norm_mean=1.0)
    bad = 63
    emb = w["token_embd.weight"]
    emb[:, 0] = 0.0
    emb[bad] = 0.0
    emb[bad, 0] = 1.0
    for i in range(cfg.n_layers):
        for t in ("attn_k", "attn_v"):
            w["blk.%d.%s.weight" % (i, t)][:, 0] = np.float16(60000.0)  # the other tokens have nothing at dim 0 ..
        for t in ("attn_output", "ffn_down"):
            w["blk.%d.%s.weight" % (i, t)][0] = 0.0  # .. in any layer
    prompt = [1 + (5 * i) % 60 for i in range(ctx_len)]
    positions = [p for p in range(ctx_len) if p < 3 or p in (31, 32, 33, 62, 63, 64, 65, 126, 127, 128, 129)]
    with A.Context(256 << 20) as ctx:
        logits = []
        for poison in (False, True):
            m = A.Model.create(ctx, A.ModelConfig(cfg.dim, cfg.n_layers, cfg.n_heads, cfg.n_kv_heads, cfg.ffn, cfg.vocab,
                                                  cfg.ctx_len, cfg.eps, cfg.theta, 1, -1))
            m.set_weights(w)
            if poison:
                for p in range(ctx_len):
                    m.forward_pass([bad] * (p + 1), p)
                assert not np.isfinite(m.logits().astype(np.float32)).all()
            out = []
            for p in range(min(ctx_len, 132)):
                m.forward_pass(prompt[:p + 1], p)
                if p in positions:
                    out.append(m.logits().view(np.uint16))
            logits.append(np.stack(out))
            m.close()
    assert np.isfinite(logits[0].view(np.float16).astype(np.float32)).all()
    assert np.array_equal(logits[0], logits[1])
