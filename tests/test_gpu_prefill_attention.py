"""The matrix-core prefill attention where its split of the work changes: chunks of a few rows after a
long history (key shares over workgroups and their merge), row blocks that straddle a key tile (rows
of one block that see no key of a tile other rows need), and every head_dim / query-group instance.

A two-layer model's logits after the last position depend on every row's attention in the first layer
(through the second layer's K and V). Compared with the per-position oracle on the forward pass's
bound (max-abs 2e-2 / rel 1e-2), which the oracle's own f16 attention accumulator sets.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    import aesir_hip

    return aesir_hip


@pytest.mark.parametrize("dim,heads,kv,first,n", [
    (512, 8, 1, 300, 1), (512, 8, 1, 610, 37), (512, 8, 1, 55, 300),   # head_dim 64, 8 query heads per KV head
    (512, 8, 2, 200, 17), (512, 8, 2, 50, 270), (512, 8, 4, 333, 5), (512, 8, 8, 447, 33),
    (1024, 8, 1, 520, 20), (1024, 8, 2, 500, 37), (1024, 8, 2, 57, 280), (1024, 8, 4, 260, 3), (1024, 8, 8, 130, 64),
])
def test_chunk_after_history(A, oracle, dim, heads, kv, first, n):
    total = first + n
    cfg = oracle.Config(dim=dim, n_layers=2, n_heads=heads, n_kv_heads=kv, ffn=2 * dim, vocab=512, ctx_len=total + 4)
    w = oracle.synthetic_weights(cfg, 78)
    om = oracle.Model(cfg, w)
    prompt = oracle.prompt_tokens(total, cfg.vocab, 5)
    okv = om.new_kv()
    for p in range(total):
        _, want = om.forward(okv, prompt, p)
    with A.Context(1 << 30) as ctx:
        m = A.Model.create(ctx, A.ModelConfig(cfg.dim, cfg.n_layers, cfg.n_heads, cfg.n_kv_heads, cfg.ffn, cfg.vocab,
                                              cfg.ctx_len, cfg.eps, cfg.theta, 1, -1))
        m.set_weights(w)
        m.prefill(prompt[:first])
        m.prefill(prompt[first:], start_pos=first)
        got = m.logits().astype(np.float64)
        m.close()
    want = np.asarray(want, np.float64)
    assert np.all(np.abs(got - want) <= 2e-2 + 1e-2 * np.abs(want))


@pytest.mark.parametrize("hd,heads,kv,first,n", [(64, 8, 1, 0, 202), (64, 8, 1, 600, 40), (64, 4, 4, 0, 202),
                                                 (128, 8, 2, 0, 202), (128, 4, 2, 300, 60), (128, 8, 1, 0, 300)])
def test_small_probabilities_are_kept(A, hd, heads, kv, first, n):
    """One key holds nearly all of the last query's weight and has V = 0; every other key holds 2^-26 of it
    and a large V, so the output is what the small probabilities carry. Everything else of the model is the
    identity or zero: norms of one-hot rows, RoPE at the pair that does not turn, no feed-forward. A whole
    position's worth of f32 sums stays far inside 1/64; f16 alone would drop every one of those keys."""
    dim, total = heads * hd, first + n
    names = ["attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down"]
    kvd, ffn, vocab = kv * hd, 256, 8
    shapes = dict(zip(names, [(dim, dim), (kvd, dim), (kvd, dim), (dim, dim), (ffn, dim), (ffn, dim), (dim, ffn)]))
    w = {"blk.0.%s.weight" % x: np.zeros(s, np.float16) for x, s in shapes.items()}
    for x in ("blk.0.attn_norm", "blk.0.ffn_norm", "output_norm"):
        w[x + ".weight"] = np.ones((1, dim), np.float16)
    emb, head = np.zeros((vocab, dim), np.float16), np.zeros((vocab, dim), np.float16)
    heavy, light, query = 1, 2, 3
    for t in (heavy, light, query):
        emb[t, t] = 1.0
    unit = np.float16(1.0 / np.sqrt(1.0 / dim + 1e-5))  # a one-hot row after its norm
    a = np.float16(np.sqrt(26 * np.log(2.0) * np.sqrt(hd)) / unit)
    w["blk.0.attn_q.weight"][hd - 2::hd, query] = a
    w["blk.0.attn_k.weight"][hd - 2::hd, heavy] = a
    w["blk.0.attn_v.weight"][:, light] = 40.0
    w["blk.0.attn_output.weight"][100, 0] = 1.0
    head[5, 100] = 1.0
    w["token_embd.weight"], w["output.weight"] = emb, head
    prompt = [heavy] + [light] * (total - 2) + [query]
    with A.Context(256 << 20) as ctx:
        m = A.Model.create(ctx, A.ModelConfig(dim, 1, heads, kv, ffn, vocab, total + 4, 1e-5, 1e12, 1, -1))
        m.set_weights(w)
        if first:
            m.prefill(prompt[:first])
        m.prefill(prompt[first:], start_pos=first)
        got = float(m.logits()[5])
        m.close()
    q = float(np.float16(unit * a))
    small = (total - 2) * np.exp(-q * q / np.sqrt(hd))
    out = small / (1.0 + small) * float(np.float16(unit * np.float16(40.0)))
    want = out / np.sqrt((1.0 + out * out) / dim + 1e-5)
    assert abs(got - want) <= want / 64, (got, want)


@pytest.mark.parametrize("hd,heads,kv,first,n,bad_at", [
    (64, 8, 1, 0, 40, 30), (64, 8, 1, 0, 300, 130), (64, 8, 1, 600, 37, 20), (64, 8, 2, 0, 70, 64), (64, 4, 2, 300, 33, 1),
    (64, 4, 4, 10, 64, 50), (128, 8, 1, 0, 40, 15), (128, 8, 2, 500, 37, 12), (128, 4, 2, 0, 100, 63), (128, 4, 4, 0, 270, 200),
    (32, 8, 2, 0, 40, 30),
])
def test_a_later_row_does_not_reach_earlier_ones(A, oracle, hd, heads, kv, first, n, bad_at):
    """A token of the chunk whose K and V overflow to infinity: the rows before it come out as with any other
    token there, bit for bit (their second-layer K and V are read back by a step at that position)."""
    total = first + n
    cfg = oracle.Config(dim=heads * hd, n_layers=2, n_heads=heads, n_kv_heads=kv, ffn=256, vocab=64, ctx_len=total + 4)
    w = oracle.synthetic_weights(cfg, 4, norm_mean=1.0)
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
    prompt = [1 + (5 * i) % 60 for i in range(total)]
    at = first + bad_at
    with A.Context(256 << 20) as ctx:
        m = A.Model.create(ctx, A.ModelConfig(cfg.dim, cfg.n_layers, cfg.n_heads, cfg.n_kv_heads, cfg.ffn, cfg.vocab,
                                              cfg.ctx_len, cfg.eps, cfg.theta, 1, -1))
        m.set_weights(w)
        got = []
        for tok in (prompt[at], bad):
            chunk = list(prompt)
            chunk[at] = tok
            if first:
                m.prefill(chunk[:first])
            m.prefill(chunk[first:], start_pos=first)
            last = m.logits().astype(np.float32)
            assert np.isfinite(last).all() == (tok != bad)  # later rows do see it
            m.forward_pass(prompt[:at + 1], at)
            got.append(m.logits())
        m.close()
    assert np.isfinite(got[0].astype(np.float32)).all()
    assert np.array_equal(got[0].view(np.uint16), got[1].view(np.uint16))
