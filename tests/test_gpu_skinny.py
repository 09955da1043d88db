"""The per-op products of 1 to 64 activation rows at the edges of their tiles, on f16 rows and on packed
GGUF blocks of every type, and the repacked route above 64 rows on the same blocks.

f16: the 32-row kernel, and from 33 rows on 8129 weight rows or more the short-chunk GEMM. Blocks: the short-chunk
GEMM where it pays (every type but Q8_0, Q3_K and Q6_K always; see the cases of the lines between), else Q8_0's
GEMV per row and an f16 copy for the other two.

Rows on both sides of the 16-row activation tiles, weight rows that end inside a 16-row block, a
workgroup (64 or 128 rows) or a group of 4, one and an odd number of 128-wide K segments, and K splits.
The bound is that of one f16 rounding of an f32 sum: 1 ulp, or 2^-17 of the sum of |products| (summation
order over at most 2^14 terms in f32, taken generously) where cancellation leaves less.
"""
import numpy as np
import pytest

from quant_tools import expected_f16, make_tensor

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(77)


@pytest.fixture(scope="module")
def A():
    import aesir_hip

    return aesir_hip


@pytest.fixture(scope="module")
def ctx(A):
    c = A.Context(1 << 30)
    yield c
    c.close()


@pytest.fixture(autouse=True)
def well_scope(ctx):
    off = ctx.offset
    yield
    ctx.synchronize()
    ctx.reset(off)


def check(got, a, w):
    a, w = a.astype(np.float64), w.astype(np.float64)
    want = a @ w.T
    ulp = np.spacing(np.abs(want).astype(np.float16)).astype(np.float64)
    err = np.abs(got.astype(np.float64) - want)
    noise = 2.0 ** -17 * (np.abs(a) @ np.abs(w).T)
    assert np.all(err <= np.maximum(ulp, noise)), float((err - np.maximum(ulp, noise)).max())


@pytest.mark.parametrize("M,K,N", [(2, 128, 1), (15, 128, 17), (16, 256, 64), (17, 384, 130), (32, 4096, 62),
                                   (33, 2176, 300), (48, 256, 4100), (49, 640, 1023), (64, 4096, 4096),
                                   (64, 14336, 70), (5, 5632, 2048)])
def test_f16_edges(A, ctx, M, K, N):
    a = RNG.standard_normal((M, K)).astype(np.float16)
    b = (RNG.standard_normal((N, K)) * 0.02).astype(np.float16)
    c = ctx.tensor(M + 1, N)  # a guard row behind the product
    c.upload(np.full((M + 1, N), 7.0, np.float16))
    A.gemm_f16(ctx, ctx.from_numpy(a), ctx.from_numpy(b), c.view(M, N))
    got = c.numpy()
    check(got[:M], a, b)
    assert np.all(got[M] == 7.0)


TYPES = {"q4_0": 2, "q4_1": 3, "q5_0": 6, "q5_1": 7, "q8_0": 8, "q2_k": 10, "q3_k": 11, "q4_k": 12, "q5_k": 13,
         "q6_k": 14}


@pytest.mark.parametrize("kind", list(TYPES))
@pytest.mark.parametrize("M,K,N", [(1, 256, 17), (2, 512, 66), (17, 768, 130), (33, 4096, 70), (64, 1280, 4099),
                                   (70, 768, 50)])
@pytest.mark.parametrize("offset", [0, 2])
def test_packed_blocks(A, ctx, oracle, kind, M, K, N, offset):
    """Blocks at the start of an allocation and 2 bytes into it (the loads' smallest alignment)."""
    if kind == "q8_0":
        d = (0.5 + RNG.random((N, K // 32))) * 0.02 / 73.6
        t = A.Q8_0Tensor.from_parts(d.astype(np.float16), RNG.integers(-127, 128, (N, K)).astype(np.int8))
        w = t.dequantize()
    else:
        t = make_tensor(A, TYPES[kind], N, K, RNG, 0.02)
        w = expected_f16(oracle, TYPES[kind], t)
    raw = np.concatenate([np.zeros(offset, np.uint8), t.blocks.reshape(-1)])
    raw = np.concatenate([raw, np.zeros(len(raw) % 2, np.uint8)])
    buf = ctx.from_numpy(raw.view(np.float16))
    a = RNG.standard_normal((M, K)).astype(np.float16)
    c = ctx.tensor(M + 1, N)
    c.upload(np.full((M + 1, N), 7.0, np.float16))
    A.gemm_quant(ctx, ctx.from_numpy(a), buf.ptr + offset, TYPES[kind], N, c.view(M, N))
    got = c.numpy()
    check(got[:M], a, w)
    assert np.all(got[M] == 7.0)


@pytest.mark.parametrize("M,K,N", [(32, 1024, 8130), (33, 1024, 8128), (33, 1024, 8129), (48, 1152, 8200), (64, 2176, 8191),
                                   (64, 896, 8200)])
def test_f16_rule(A, ctx, M, K, N):
    """Both sides of the lines between the 32-row kernel and the short-chunk GEMM."""
    test_f16_edges(A, ctx, M, K, N)


@pytest.mark.parametrize("kind,M,K,N", [
    # Q8_0: rows times weight rows below and above the line, one launch without K splits, several passes of 64 rows
    ("q8_0", 12, 768, 2047), ("q8_0", 13, 768, 1900), ("q8_0", 2, 256, 33), ("q8_0", 17, 128, 65), ("q8_0", 33, 256, 130),
    ("q8_0", 48, 640, 515), ("q8_0", 64, 640, 386), ("q8_0", 65, 256, 100), ("q8_0", 65, 1024, 770), ("q8_0", 130, 512, 700),
    # Q3_K and Q6_K: the copy for short rows, one row, few bytes; the blocks in 4 and in 8 waves
    ("q6_k", 16, 768, 341), ("q6_k", 17, 768, 341), ("q6_k", 16, 768, 342), ("q6_k", 1, 1792, 2400), ("q6_k", 1, 2048, 2049),
    ("q6_k", 2, 1024, 2047), ("q6_k", 2, 1024, 2049), ("q6_k", 33, 1280, 1700), ("q6_k", 32, 1280, 1700), ("q6_k", 64, 2816, 1001),
    ("q6_k", 40, 1024, 8192), ("q6_k", 40, 1024, 8200),
    ("q3_k", 16, 768, 341), ("q3_k", 17, 768, 341), ("q3_k", 1, 2048, 2047), ("q3_k", 1, 2048, 2049), ("q3_k", 33, 1280, 1700),
    ("q3_k", 64, 2816, 1001), ("q4_k", 1, 512, 700), ("q4_0", 1, 512, 700),
])
def test_packed_blocks_rule(A, ctx, oracle, kind, M, K, N):
    """Both sides of the lines between the routes of packed blocks."""
    test_packed_blocks(A, ctx, oracle, kind, M, K, N, 0)


def test_q8_0_row_limit(A, ctx):
    """More than 65535 rows of A are refused whatever the alignment."""
    a, c = ctx.tensor(65536, 32), ctx.tensor(65536, 1)
    a256 = ctx.tensor(65536, 256)
    blocks = ctx.tensor(1, 8 * 17)
    for x, rows in ((a, 1), (a256, 1)):
        with pytest.raises(A.AesirError, match="more than 65535 rows"):
            A.gemm_q8_0(ctx, x, blocks.ptr, rows, c)
    wide = ctx.tensor(65536, 1024)
    with pytest.raises(A.AesirError, match="more than 65535 rows"):
        A.gemm_q8_0(ctx, a256, ctx.tensor(1024, 8 * 17).ptr, 1024, wide)
