"""The sampler's top-k selection and token lists where their route changes: more ties at the k-th logit
than the sorting workgroup holds (constant logits, three levels), fewer ties but more together with the
candidates above them, exactly as many candidates as top_k
leaves, token lists on both sides of the length that the prepare kernel scans itself, ids outside the
vocabulary, vocabularies around a workgroup's 1024 entries. Token and RuneRNG state equal the oracle's
(exact: both sides run the reference's f32 sums in the reference's order)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    import aesir_hip

    return aesir_hip


@pytest.mark.parametrize("vocab,levels,top_k,n_context,n_suppress", [
    (128256, 1, 40, 0, 0), (128256, 1, 4096, 5, 0), (128256, 3, 1000, 300, 2), (60000, 2, 3000, 8192, 0),
    (60000, 200, 64, 8190, 3), (1023, 1, 1000, 10, 0), (1024, 60, 1023, 0, 1), (1025, 60, 40, 2000, 10),
    (4097, 1, 4096, 1, 1), (2, 1, 1, 0, 0),
    # more gathered than the workgroup holds, of which those that share the k-th key's bits are fewer
    (60000, 200, 4090, 10, 0), (60000, 200, 4096, 0, 2), (60000, 20, 4096, 0, 0), (128256, 4000, 4096, 256, 0),
    (30000, 8, 4000, 0, 0), (8192, 2, 4095, 0, 0), (8193, 2, 4096, 0, 0),
])
def test_selection(A, oracle, vocab, levels, top_k, n_context, n_suppress):
    rng = np.random.default_rng(vocab + top_k + n_context)
    cfg = dict(temperature=0.8, top_k=top_k, top_p=0.97, repetition_penalty=1.2)
    g_rng = A.RuneRNG(99)
    o_state = oracle.rune_rng_state(99)
    with A.Context(64 << 20) as ctx:
        for d in range(4):
            logits = (rng.integers(0, levels, vocab) * 0.5 + 1.0).astype(np.float16)
            context = rng.integers(-3, vocab + 3, n_context).tolist()
            suppress = rng.integers(0, vocab + 1, n_suppress).tolist()
            got = A.sample_token(ctx, ctx.from_numpy(logits.reshape(1, -1)), A.SamplerConfig(**cfg), g_rng, context, suppress)
            want, o_state = oracle.sample_token_f16(logits, oracle.SamplerConfig(**cfg), o_state, context, suppress)
            assert got == want, d
            assert g_rng.state == o_state, d


@pytest.mark.parametrize("top_p,min_p", [(0.9, 0.0), (1.0, 0.02), (0.97, 0.1), (1.0, 0.0), (1e-6, 0.0), (1.0, 0.999)])
@pytest.mark.parametrize("top_k", [2, 63, 255, 256, 257, 1025, 4096])
def test_truncations_of_the_selection(A, oracle, top_k, top_p, min_p):
    """Both sorts of the selecting workgroup (by rank up to 256 gathered candidates, bitonic above) with
    each truncation behind them; infinities and NaN among the logits are sanitized first."""
    rng = np.random.default_rng(top_k)
    cfg = dict(temperature=0.7, top_k=top_k, top_p=top_p, min_p=min_p)
    g_rng = A.RuneRNG(5)
    o_state = oracle.rune_rng_state(5)
    with A.Context(64 << 20) as ctx:
        for d in range(3):
            logits = (rng.standard_normal(9000) * (0.3, 2.5, 8.0)[d]).astype(np.float16)
            logits[rng.integers(0, 9000, 4)] = [np.inf, -np.inf, np.nan, -0.0]
            got = A.sample_token(ctx, ctx.from_numpy(logits.reshape(1, -1)), A.SamplerConfig(**cfg), g_rng, [], [])
            want, o_state = oracle.sample_token_f16(logits, oracle.SamplerConfig(**cfg), o_state, [], [])
            assert got == want, d
            assert g_rng.state == o_state, d


@pytest.mark.parametrize("vocab,live,top_k", [(128256, 10, 40), (128256, 0, 40), (32000, 60, 1000), (4097, 3, 4), (4100, 1, 4096),
                                              (20000, 39, 40), (20000, 40, 40)])
def test_masked_logits(A, oracle, vocab, live, top_k):
    """Nearly all logits masked to -inf (sanitized to one value): the selection is filled up with the masked ones
    of the lowest indices."""
    rng = np.random.default_rng(vocab + live)
    cfg = dict(temperature=0.8, top_k=top_k, top_p=1.0, min_p=0.0, repetition_penalty=1.1)
    g_rng, o_state = A.RuneRNG(4), oracle.rune_rng_state(4)
    with A.Context(64 << 20) as ctx:
        for d in range(3):
            logits = np.full(vocab, -np.inf, np.float16)
            logits[rng.permutation(vocab)[:live]] = rng.standard_normal(live).astype(np.float16) if d else np.float16(-6e4)
            context = rng.integers(0, vocab, 5).tolist()
            got = A.sample_token(ctx, ctx.from_numpy(logits.reshape(1, -1)), A.SamplerConfig(**cfg), g_rng, context, [])
            want, o_state = oracle.sample_token_f16(logits, oracle.SamplerConfig(**cfg), o_state, context, [])
            assert got == want, d
            assert g_rng.state == o_state, d


@pytest.mark.parametrize("plain,top_k", [(50, 40), (50, 50), (50, 51), (50, 100), (12000, 64), (12000, 4096)])
def test_ties_that_differ_in_their_last_bits(A, oracle, plain, top_k):
    """More logits than the selecting workgroup holds share all but the last bits of their key: equal ones, part of
    them moved by a repetition penalty next to 1."""
    vocab = 20000
    rng = np.random.default_rng(plain + top_k)
    cfg = dict(temperature=1.0, top_k=top_k, top_p=1.0, min_p=0.0, repetition_penalty=1.00001)
    g_rng, o_state = A.RuneRNG(6), oracle.rune_rng_state(6)
    logits = np.full(vocab, -1.6, np.float16)
    with A.Context(64 << 20) as ctx:
        for d in range(3):
            context = rng.permutation(vocab)[plain:].tolist()
            got = A.sample_token(ctx, ctx.from_numpy(logits.reshape(1, -1)), A.SamplerConfig(**cfg), g_rng, context, [])
            want, o_state = oracle.sample_token_f16(logits, oracle.SamplerConfig(**cfg), o_state, context, [])
            assert got == want, d
            assert g_rng.state == o_state, d
