// Short-chunk GEMM (2 to 64 activation rows) for every weight type: plan, dispatch and launch of
// gemm_skinny_kernel.
#include "common.hpp"
#include "device.hpp"
#include "kernels.hpp"
#include "mfma_gemm.hpp"
#include "skinny_launch.hpp"

namespace aesir {

// Waves per workgroup (16 weight rows each) and K splits. 8 waves re-read the activations half as
// often as 4 and 4 fill the chip where the rows are few, so 8 where they reach about a workgroup
// per CU (with splits, or by themselves where the epilogue is applied in the kernel). The splits
// bring the grid to at most kSkinnyWgTarget workgroups, with at least two segments each, at most 8
// (the fused row kernels' count). Measured on MI355X, 37 rows, weights past the MALL, us per launch,
// 8 waves / 4 waves: Q4_K gate/up 28672 x 4096 27.0 / 28, O 4096 x 4096 6.8 / 7.5, down 4096 x 14336
// 12.9 / 17.3, 11264 x 2048 14.7 / 11.5, 2048 x 2048 4.7 / 4.3; f16 54.7 / 52.6, 11.7 / 10.0, 26.5 /
// 25.7, 24.1 / 15.6, 6.8 / 5.0 (f16 always takes 4: its own bytes outweigh the activations').
constexpr int64_t kSkinnyWgTarget = 256;

SkinnyPlan skinny_plan(int64_t M, int64_t K, int64_t N, int32_t type, SkinnySplit split, bool raw) {
    const int64_t lim = (int64_t)1 << 31;
    if (M < 1 || M > kSkinnyMaxRows || K % kSeg != 0 || K * M >= lim || N < 1 || N >= lim / 2) return {};
    if (!raw && qf_type(type) && (K % gguf_block_elems(type) != 0 || mul_checked(qf_rows_alloc(N), K) >= lim)) return {};
    if (raw && K % gguf_block_elems(type) != 0) return {};
    SkinnyPlan p;
    const int64_t t8 = (N + 127) / 128;
    // a sum launch costs more than it gains once 4-wave workgroups alone reach most CUs
    const bool may_split = split == kSplitFree || (split == kSplitPaid && (N + 63) / 64 < kSkinnyWgTarget * 5 / 8);
    p.nw = type != AESIR_GGML_F16 && t8 * (may_split ? 8 : 1) >= kSkinnyWgTarget * 3 / 4 ? 8 : 4;
    // packed Q6_K blocks with 33 rows or more: 4 waves and their splits up to 8192 weight rows (us per call, 8 / 4
    // waves, 64 rows: 4096 x 4096 23.9 / 19.7, 6144 x 4096 32.9 / 28.8, 3072 x 3072 24.3 / 18.0, 8000 x 6144 38.8 /
    // 39.7, 32000 x 2048 41.8 / 44.2)
    if (raw && type == AESIR_GGML_Q6_K && M > 32 && N <= 8192) p.nw = 4;
    if (may_split) {
        const int64_t tiles = (N + 16 * p.nw - 1) / (16 * p.nw), most = K / (2 * kSeg);
        int64_t s = kSkinnyWgTarget / tiles;
        if (s > 8) s = 8;
        if (s > most) s = most;
        p.splits = s < 1 ? 1 : s;
    }
    return p;
}

int32_t launch_gemm_skinny(hipStream_t s, int epi, const SkinnyMat &w, const void *A, int64_t M, int64_t K, int64_t N,
                           void *C, int64_t ldc, float *part, int64_t ldp, const SkinnyPlan &p) {
    if (!p.nw || M < 1 || M > kSkinnyMaxRows || K % kSeg != 0 || p.splits < 1 || p.splits > K / kSeg ||
        (p.splits > 1 && !part) || (epi == kEpiSwiglu && (N & 1)) || w.qf.row0 % 16 != 0 ||
        (w.raw && ((uintptr_t)w.w & 1)))
        return fail(AESIR_ERR_INVALID, "gemm_skinny: unsupported arguments");
    if (((uintptr_t)A & 15) || ((uintptr_t)part & 15)) return fail(AESIR_ERR_INVALID, "gemm_skinny: operand is not 16-byte aligned");
    int32_t rc = AESIR_OK;
    if (w.raw) rc = launch_gemm_skinny_raw(s, epi, w, A, M, K, N, C, ldc, part, ldp, p);
    else if (w.type == AESIR_GGML_F16) rc = launch_m<AESIR_GGML_F16>(s, epi, w, A, M, K, N, C, ldc, part, ldp, p);
    else if (w.type == AESIR_GGML_Q8_0) rc = launch_m<AESIR_GGML_Q8_0>(s, epi, w, A, M, K, N, C, ldc, part, ldp, p);
    else if (qf_type(w.type))
        qf_switch(w.type, [&](auto t) { rc = launch_m<decltype(t)::value>(s, epi, w, A, M, K, N, C, ldc, part, ldp, p); });
    else rc = fail(AESIR_ERR_UNSUPPORTED, "gemm_skinny: weight type %d", (int)w.type);
    return rc;
}

}  // namespace aesir
