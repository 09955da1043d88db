// gemm_skinny_kernel on packed GGUF blocks (raw_tile.hpp): the per-op products of a few rows, which
// read each block once as it lies in memory instead of repacking or dequantizing the matrix first.
// Measured on MI355X, 14336 x 4096, us per call: Q4_K 1 row 78.5 -> 16.3 (repack 72 + GEMV 10 before), 64
// rows 104 -> 30; Q4_0 43 -> 20, Q5_K 61 -> 24, Q6_K 74 -> 39 (210-byte blocks: its loads straddle the
// most lines); Q8_0 at 128 rows of 4096 x 4096 379 -> 39 (one pass over the blocks per row before).
#include "skinny_launch.hpp"

namespace aesir {

int32_t launch_gemm_skinny_raw(hipStream_t s, int epi, const SkinnyMat &w, const void *A, int64_t M, int64_t K, int64_t N,
                               void *C, int64_t ldc, float *part, int64_t ldp, const SkinnyPlan &p) {
    if (w.type == AESIR_GGML_Q8_0) return launch_m<kRawType + AESIR_GGML_Q8_0>(s, epi, w, A, M, K, N, C, ldc, part, ldp, p);
    if (!qf_type(w.type)) return fail(AESIR_ERR_UNSUPPORTED, "gemm_skinny: weight type %d", (int)w.type);
    int32_t rc = AESIR_OK;
    qf_switch(w.type, [&](auto t) {
        rc = launch_m<kRawType + decltype(t)::value>(s, epi, w, A, M, K, N, C, ldc, part, ldp, p);
    });
    return rc;
}

}  // namespace aesir
