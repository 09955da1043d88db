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
