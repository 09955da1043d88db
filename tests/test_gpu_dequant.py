"""The f16 copies of quantized matrices that long prefill chunks multiply: whole 16 x 128 plane tiles per
wave (repacked types), and eight weights per thread (Q8_0), where rows end inside a tile and the weight
count ends inside a workgroup.

The copies are whole numbers of f16 rounding steps of the type's own rule, so they equal the oracle's bits.
"""
import numpy as np
import pytest

from quant_tools import expected_f16, make_tensor, same_token, within_tol

pytestmark = pytest.mark.gpu

TYPES = {"q4_0": 2, "q4_1": 3, "q5_0": 6, "q5_1": 7, "q2_k": 10, "q3_k": 11, "q4_k": 12, "q5_k": 13, "q6_k": 14}


@pytest.fixture(scope="module")
def A():
    import aesir_hip

    return aesir_hip


@pytest.fixture(scope="module")
def ctx(A):
    c = A.Context(1 << 30)
    yield c
    c.close()


def weights(A, oracle, cfg, t, seed):
    rng = np.random.default_rng(seed)
    w = {}
    for name, (r, c) in oracle.tensor_shapes(cfg).items():
        norm = name.endswith("norm.weight")
        w[name] = (1.0 + 0.05 * rng.standard_normal(c)).astype(np.float16) if norm else make_tensor(A, t, r, c, rng)
    return w


def make(A, ctx, cfg, t, w):
    m = A.Model.create(ctx, A.ModelConfig(cfg.dim, cfg.n_layers, cfg.n_heads, cfg.n_kv_heads, cfg.ffn, cfg.vocab,
                                          cfg.ctx_len), t)
    m.set_weights(w)
    return m


@pytest.mark.parametrize("kind", list(TYPES))
@pytest.mark.parametrize("vocab", [1, 17, 1003])
def test_tiles_equal_the_rule(A, ctx, oracle, kind, vocab):
    """Vocabulary rows that end inside a row block, the parts of the fused Q/K/V, and the interleaved gate
    and up rows (gathered record by record), read back bit for bit."""
    cfg = oracle.Config(dim=256, n_layers=1, n_heads=32, n_kv_heads=2, ffn=512, vocab=vocab, ctx_len=32)
    w = weights(A, oracle, cfg, TYPES[kind], vocab)
    m = make(A, ctx, cfg, TYPES[kind], w)
    for name, shape in oracle.tensor_shapes(cfg).items():
        if not name.endswith("norm.weight"):
            want = expected_f16(oracle, TYPES[kind], w[name])
            assert np.array_equal(m.get_tensor(name, shape).view(np.uint16), want.view(np.uint16)), name
    m.close()


def test_q8_0_long_chunk_with_a_ragged_weight_count(A, ctx, oracle):
    """260 rows on matrices of 61440 and 36864 weights: half a workgroup's share is past the end."""
    cfg = oracle.Config(dim=192, n_layers=2, n_heads=3, n_kv_heads=1, ffn=192, vocab=70, ctx_len=272)
    w = weights(A, oracle, cfg, 8, 3)
    om = oracle.Model(cfg, {n: x if n.endswith("norm.weight") else expected_f16(oracle, 8, x) for n, x in w.items()})
    m = make(A, ctx, cfg, 8, w)
    prompt = oracle.prompt_tokens(260, cfg.vocab, 5)
    kv, cur = om.new_kv(), list(prompt)
    for p in range(len(prompt)):
        want, logits = om.forward(kv, cur, p)
    got = m.prefill(prompt)
    assert within_tol(m.logits(), logits)
    assert same_token(got, want, logits)
    m.close()
