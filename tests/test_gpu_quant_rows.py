"""The decode GEMVs of the repacked weight types at row lengths and row counts of full-size models, and prefill
chunks of 1 to 64 rows on every stored weight type, through one-layer models against the CPU oracle on the
weights' f16 values.

Decode: K of 14336 and 28672 (several rounds of a wave), 5632 and 2048 (a partial last round), and lm_heads of more
than 1024 16-row blocks (persistent workgroups) that end inside a block. Chunks: one to four 16-row activation tiles
and both sides of each, 4 and 8 waves per workgroup, K splits and none, an odd number of 128-wide segments, weight
rows that end inside a workgroup's share; with the store, residual and SwiGLU epilogues. A row of weights left out or taken twice
moves its logit, or through the residual stream all of them, by far more than the forward pass's bound (max-abs 2e-2 /
rel 1e-2): logits have a spread of 0.3 and more.
"""
import numpy as np
import pytest

from quant_tools import expected_f16, make_tensor, within_tol

pytestmark = pytest.mark.gpu

REPACKED = {"q4_0": 2, "q4_1": 3, "q5_0": 6, "q5_1": 7, "q2_k": 10, "q3_k": 11, "q4_k": 12, "q5_k": 13, "q6_k": 14}
STORED = dict(f16=1, q8_0=8, **REPACKED)


@pytest.fixture(scope="module")
def A():
    import aesir_hip

    return aesir_hip


def model(A, oracle, ctx, t, dim, heads, kv, ffn, vocab, ctx_len):
    cfg = oracle.Config(dim=dim, n_layers=1, n_heads=heads, n_kv_heads=kv, ffn=ffn, vocab=vocab, ctx_len=ctx_len)
    rng = np.random.default_rng(dim + ffn + t)
    w = {}
    for name, (r, c) in oracle.tensor_shapes(cfg).items():
        norm = name.endswith("norm.weight")
        std = 0.02 if t not in (10, 12, 13) else 0.006  # (types with minima: their weights have a mean as well)
        w[name] = (1.0 + 0.05 * rng.standard_normal(c)).astype(np.float16) if norm else make_tensor(A, t, r, c, rng, std)
    m = A.Model.create(ctx, A.ModelConfig(cfg.dim, cfg.n_layers, cfg.n_heads, cfg.n_kv_heads, cfg.ffn, cfg.vocab,
                                          cfg.ctx_len), t)
    m.set_weights(w)
    plain = {n: x if t == 1 or n.endswith("norm.weight") else expected_f16(oracle, t, x) for n, x in w.items()}
    return m, oracle.Model(cfg, plain), oracle.prompt_tokens(ctx_len, vocab, 5)


@pytest.mark.parametrize("kind", list(REPACKED))
@pytest.mark.parametrize("dim,heads,kv,ffn,vocab", [(1024, 8, 2, 14336, 40), (256, 4, 2, 28672, 18001), (2048, 16, 4, 5632, 33),
                                                    (512, 8, 2, 1536, 16401)])
def test_decode_rows(A, oracle, kind, dim, heads, kv, ffn, vocab):
    with A.Context(1 << 30) as ctx:
        m, om, prompt = model(A, oracle, ctx, REPACKED[kind], dim, heads, kv, ffn, vocab, 8)
        okv = om.new_kv()
        for p in range(3):
            _, want = om.forward(okv, prompt, p)
            m.forward_pass(prompt[:p + 1], p)
            got = m.logits()
            assert np.asarray(want, np.float64).std() > 0.25
            assert within_tol(got, want), (p, float(np.abs(got.astype(np.float64) - np.asarray(want, np.float64)).max()))
        m.close()


@pytest.mark.parametrize("kind", list(STORED))
@pytest.mark.parametrize("shape", ["wide", "ragged", "long_ffn"])
def test_short_chunks(A, oracle, kind, shape):
    t = STORED[kind]
    k256 = 10 <= t
    # wide: 8 waves with K splits; ragged: Q/K/V of 432 or 864 rows, three and five segments (six for the super-block
    # types); long_ffn: 8 waves without K splits in gate and up
    dim, heads, kv, ffn = {"wide": (3072, 48, 6, 256), "long_ffn": (256, 4, 2, 12544),
                           "ragged": (768, 16, 1, 768) if k256 else (384, 16, 1, 640)}[shape]
    with A.Context(1 << 30) as ctx:
        m, om, prompt = model(A, oracle, ctx, t, dim, heads, kv, ffn, 67, 80)
        okv = om.new_kv()
        want = [om.forward(okv, prompt, p)[1] for p in range(65)]
        for n in (1, 2, 15, 16, 17, 32, 33, 37, 48, 49, 64):
            m.prefill(prompt[:n])
            assert within_tol(m.logits(), want[n - 1]), n
        m.forward_pass(prompt[:65], 64)  # reads the rows that the chunk of 64 wrote
        assert within_tol(m.logits(), want[64])
        m.close()
