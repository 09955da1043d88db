// Launch of gemm_skinny_kernel for one weight type (skinny.hip: types a model stores; skinny_raw.hip:
// packed GGUF blocks).
#pragma once

#include "common.hpp"
#include "kernels.hpp"
#include "skinny.hpp"

namespace aesir {

template <int T, int MT, int NW>
int32_t launch_t(hipStream_t s, int epi, const SkinnyMat &w, const void *A, int64_t M, int64_t K, int64_t N, void *C,
                        int64_t ldc, float *part, int64_t ldp, int64_t splits) {
    constexpr int lds = 2 * kSkSegs * MT * 4096;
    static_assert(lds <= 64 * 1024, "within the default LDS limit");
    const dim3 grid((unsigned)((N + 16 * NW - 1) / (16 * NW)), (unsigned)splits);
    hipLaunchKernelGGL((gemm_skinny_kernel<T, MT, NW>), grid, dim3(NW * kWave), lds, s, (const h16 *)A, (int)M,
                       (int)K, w, (int)N, epi, (h16 *)C, ldc, part, ldp);
    AESIR_LAUNCH_CHECK("gemm_skinny_kernel");
    return AESIR_OK;
}

template <int T>
int32_t launch_m(hipStream_t s, int epi, const SkinnyMat &w, const void *A, int64_t M, int64_t K, int64_t N, void *C,
                        int64_t ldc, float *part, int64_t ldp, const SkinnyPlan &p) {
#define AESIR_SK(MTV)                                                                                       \
    if constexpr (T != AESIR_GGML_F16) /* (skinny_plan gives f16 4 waves) */                                \
        if (p.nw == 8) return launch_t<T, MTV, 8>(s, epi, w, A, M, K, N, C, ldc, part, ldp, p.splits);      \
    return launch_t<T, MTV, 4>(s, epi, w, A, M, K, N, C, ldc, part, ldp, p.splits)
    switch ((M + 15) / 16) {
        case 1: AESIR_SK(1);
        case 2: AESIR_SK(2);
        case 3: AESIR_SK(3);
        default: AESIR_SK(4);
    }
#undef AESIR_SK
}

}  // namespace aesir
