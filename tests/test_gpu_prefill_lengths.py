"""Long chunks at the lengths where the library refuses the algorithm that it proposes first: the chunk runs
on the next one (or the framework's own kernels) instead of failing. One layer at the TinyLlama and Llama-3
widths; the logits equal those of the same prompt in chunks below 256 rows, which never reach the library,
within the forward pass's bound (max-abs 2e-2 / rel 1e-2).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    import aesir_hip

    return aesir_hip


@pytest.mark.parametrize("dim,heads,kv,ffn,lengths", [
    (4096, 32, 8, 14336, (256, 345, 408, 426, 453, 471, 513, 525, 678, 804, 822)),
    (2048, 32, 4, 5632, (256, 678, 705, 714, 804, 831, 858)),
    (3072, 24, 8, 8192, (561, 570, 687, 714, 777, 867)),
])
def test_long_chunk_lengths(A, dim, heads, kv, ffn, lengths):
    with A.Context(3 << 30) as ctx:
        m = A.Model.create(ctx, A.ModelConfig(dim, 1, heads, kv, ffn, 512, 900, 1e-5, 10000.0, 1, -1))
        m.init_random(3, norm_mean=1.0)
        for n in lengths:
            prompt = [(7 * i + 3 * n) % 512 for i in range(n)]
            m.prefill(prompt)
            got = m.logits().astype(np.float64)
            for p in range(0, n, 200):
                m.prefill(prompt[p:p + 200], start_pos=p)
            want = m.logits().astype(np.float64)
            assert np.all(np.abs(got - want) <= 2e-2 + 1e-2 * np.abs(want)), n
        m.close()
