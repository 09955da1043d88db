// Kernel body of the short-chunk GEMM (skinny.hip): C = epilogue(A W^T) for a few tens of
// activation rows and a weight matrix of any type, on v_mfma_f32_16x16x32_f16.
#pragma once

#include "mfma_gemm.hpp"
#include "qf_tile.hpp"
#include "raw_tile.hpp"

namespace aesir {

// One lane's share of a 16-row x 128-k weight tile: row lane % 16, k = 32 (lane / 16) .. + 31.
// T: f16 rows, Q8_0 planes, a repacked type's planes, or (kRawType + GGML type) packed GGUF blocks.
constexpr int kRawType = 256;
template <int T>
struct SkTile {
    std::conditional_t<(T >= kRawType), RawTile<T % kRawType>, QTile<T % kRawType>> q;
};
template <>
struct SkTile<AESIR_GGML_F16> {
    u32x4 v[4];
};
template <>
struct SkTile<AESIR_GGML_Q8_0> {
    u32x4 v[2];
    h16 d;
};
template <>
struct SkTile<kRawType + AESIR_GGML_Q8_0> {
    RawTile<AESIR_GGML_Q8_0> q;
};
// The 8 k values of A operand j in lane group g of a segment are granule sk_granule(g, j) (k
// 8 granule .. + 7): 32 consecutive weights per lane for the repacked tiles (their layout) and for
// Q8_0 rows (one block, so one scale); f16 rows by 64 contiguous bytes of a row per load (16-byte
// pieces 64 bytes apart took 85 us for gate/up against 53).
template <int T>
__device__ __forceinline__ constexpr int sk_granule(int g, int j) {
    return T == AESIR_GGML_F16 ? 4 * j + g : 4 * g + j;
}

// Grid (ceil(N / (16 NB NW)), splits), NW waves. Wave w owns the NB row blocks
// (blockIdx.x NW + w) NB .. of 16 weight rows and all MT 16-row activation tiles; the K range of
// split z goes by in steps of SG 128-wide segments. A step's weight tiles go straight from memory
// into registers and are dequantized there (they are the MFMA A operand: every weight byte is read
// once by one wave), D - 1 steps ahead of their use; its activations are requested equally far
// ahead, each by one thread of the workgroup, and stored to one of two LDS stages in B-operand
// order, where every wave reads them. So the HBM stream is the weights in their stored form and
// the activations cost one L2 read per 16 NB NW weight rows.
// LDS stage: granule p of lane group g's operand j (p = sk_granule(g, j)) of activation row 16 mt + c,
// segment u, at ((u MT + mt) 4 + j) 1024 + g 256 + 16 (c ^ ((8 u + p / 2) & 15)): a fragment read
// covers 256 contiguous bytes per lane group, and the 16 records of a row that neighbouring
// threads store fall into different banks.
// Rows past M and weight rows past N re-read the last one; their results are not stored.
// With one split the epilogue is applied here, else split z writes f32 partials P[z][M][ldp].
// Bound: HBM for f16 weights (4.5 TB/s), the LDS reads of the activations (every wave reads all of
// them: 4 us per 16 rows of 28672 x 4096) and the dequantization beside the weight stream for the
// quantized types. Measured on MI355X at 37 rows (weights past the MALL, us per launch): Q4_K gate/up
// 28672 x 4096 26 where dequantizing to f16 and multiplying on the 32-row kernel took 163 (96 + 67),
// down 4096 x 14336 12.9 (of 80); Q8_0 gate/up 41.5; f16 gate/up 52.7 against 67 for the 32-row
// kernel, O 10.0 against 19. 37 rows after 500 positions on the Llama-3-8B shape in Q4_K_M: 11.9 ->
// 3.8 ms. Not faster: three steps of weights in flight, two K groups of waves per workgroup, two row
// blocks per wave (34 us: too few workgroups).
constexpr int kSkSegs = 2;  // segments per step
template <int T, int MT, int NW>
__global__ __launch_bounds__(NW *kWave) void gemm_skinny_kernel(const h16 *__restrict__ A, int M, int K, SkinnyMat w,
                                                              int N, int epi, h16 *__restrict__ C, int64_t ldc,
                                                              float *__restrict__ P, int64_t ldp) {
    constexpr int NB = 1, SG = kSkSegs, D = 2;     // row blocks per wave, segments per step, steps in flight
    constexpr int NT = NW * kWave;
    constexpr int STAGE = SG * MT * 4096;
    constexpr int RECS = SG * MT * 128;            // 16-element activation records of a step
    constexpr int XL = (RECS + NT - 1) / NT;       // records per thread
    constexpr bool RAW = T >= kRawType, QF = T != AESIR_GGML_F16 && T != AESIR_GGML_Q8_0 && !RAW;
    constexpr int TR = T % kRawType;
    static_assert(SG <= 2, "the store swizzle covers 16 records per row");
    extern __shared__ __align__(16) uint8_t lds[];  // two stages
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int nseg = K >> 7, splits = gridDim.y, z = blockIdx.y;
    const int sg0 = (int)((int64_t)nseg * z / splits), sg1 = (int)((int64_t)nseg * (z + 1) / splits);
    const int steps = (sg1 - sg0 + SG - 1) / SG;
    const int nblk = (N + 15) >> 4;
    const int blk0 = ((int)blockIdx.x * NW + wave) * NB;  // first row block of the wave

    // ---- activations: thread's records of a step, global offset and LDS slot
    auto slot = [&](int u, int row, int p) {  // granule p of segment u of activation row `row`
        const int gg = T == AESIR_GGML_F16 ? p & 3 : p >> 2, j = T == AESIR_GGML_F16 ? p >> 2 : p & 3;
        return ((u * MT + (row >> 4)) * 4 + j) * 1024 + gg * 256 + (((row & 15) ^ ((8 * u + (p >> 1)) & 15)) << 4);
    };
    const h16 *xp[XL];
    int xs[XL];
    bool xlive[XL];
#pragma unroll
    for (int i = 0; i < XL; i++) {
        const int rec = tid + NT * i;
        xlive[i] = rec < RECS;
        const int row = xlive[i] ? rec / (8 * SG) : 0, q = rec % (8 * SG);  // record q of the step: segment q / 8
        xp[i] = A + (int64_t)(row < M ? row : M - 1) * K + 16 * q;
        xs[i] = slot(q >> 3, row, 2 * (q & 7));
    }
    struct XBuf {
        u32x4 v[XL][2];
    };
    auto xload = [&](XBuf &b, int st) {
        int seg = sg0 + (st < steps ? st : steps - 1) * SG;
#pragma unroll
        for (int i = 0; i < XL; i++) {
            // a last step's segments past K re-read the row's first ones
            const int u = ((tid + NT * i) % (8 * SG)) >> 3;
            const int sg = SG == 1 || seg + u < nseg ? seg : seg - u;
            const h16 *p = xp[i] + sg * 128;
            b.v[i][0] = ld16(p);
            b.v[i][1] = ld16(p + 8);
        }
    };
    auto xstore = [&](const XBuf &b, uint8_t *stage) {
#pragma unroll
        for (int i = 0; i < XL; i++) {
            u32x4 o[2] = {b.v[i][0], b.v[i][1]};
            if constexpr (QF) qf_perm_rec(b.v[i], o);  // the nibble words' element order
            if (RECS % NT == 0 || xlive[i]) {
                st16(stage + xs[i], o[0]);
                st16(stage + xs[i] + (T == AESIR_GGML_F16 ? 256 : 1024), o[1]);
            }
        }
    };

    // ---- weights
    struct WBuf {
        SkTile<T> t[SG][NB];
    };
    constexpr int es1 = (qf_kq<T>() || T == AESIR_GGML_Q2_K) ? 4 : 2;
    QfRsrc rs;
    if constexpr (QF) rs = qf_rsrc(w.qf, T, w.qf.row0 + (int64_t)nblk * 16, K);
    const int sbr = K >> 8, s1v = c * es1;
    const uint8_t *wr[NB];  // packed blocks of the lane's row
    const h16 *wf[NB];
    const int8_t *wq[NB];
    const h16 *wd[NB];
    int pb[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int blk = blk0 + b < nblk ? blk0 + b : nblk - 1;
        pb[b] = (int)(w.qf.row0 >> 4) + blk;
        const int row = blk * 16 + c < N ? blk * 16 + c : N - 1;
        if constexpr (T == AESIR_GGML_F16) wf[b] = (const h16 *)w.w + (int64_t)row * K + 8 * g;
        if constexpr (RAW) wr[b] = (const uint8_t *)w.w + (int64_t)row * (K / (raw_super(TR) ? 256 : 32)) * raw_block_bytes(TR);
        if constexpr (T == AESIR_GGML_Q8_0) {
            wq[b] = (const int8_t *)w.w + (int64_t)row * K + 32 * g;
            wd[b] = (const h16 *)w.s + (int64_t)row * (K / 32) + g;
        }
    }
    auto wload = [&](WBuf &buf, int st) {
        const int first = sg0 + (st < steps ? st : steps - 1) * SG;
#pragma unroll
        for (int u = 0; u < SG; u++) {
            const int sg = first + u < sg1 ? first + u : sg1 - 1;  // surplus: the split's last segment again
#pragma unroll
            for (int b = 0; b < NB; b++) {
                SkTile<T> &t = buf.t[u][b];
                if constexpr (T == AESIR_GGML_F16) {
#pragma unroll
                    for (int j = 0; j < 4; j++) t.v[j] = ld16(wf[b] + sg * 128 + 32 * j);
                } else if constexpr (T == AESIR_GGML_Q8_0) {
                    t.v[0] = ld16(wq[b] + sg * 128);
                    t.v[1] = ld16(wq[b] + sg * 128 + 16);
                    t.d = wd[b][sg * 4];
                } else if constexpr (RAW) {
                    raw_load<TR>(t.q, wr[b] + (raw_super(TR) ? sg >> 1 : 4 * sg + g) * raw_block_bytes(TR), sg & 1, g);
                } else {
                    t.q = qf_tile_load<T>(rs, pb[b] * nseg + sg, lane, s1v, (pb[b] * sbr + (sg >> 1)) * 16 * es1);
                }
            }
        }
    };

    f32x4 acc[NB][MT];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int m = 0; m < MT; m++) acc[b][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    WBuf wb[D];
    XBuf xb[D];
#pragma unroll
    for (int j = 0; j + 1 < D; j++) {
        xload(xb[j], j);
        wload(wb[j], j);
    }
    xstore(xb[0], lds);
    __syncthreads();
    QfRegs kr;
    if constexpr (QF) kr = QfRegs::make();
    auto step = [&](int st, const WBuf &cur, WBuf &wnew, XBuf &xnew, const XBuf &xnext) {
        xload(xnew, st + D - 1);
        wload(wnew, st + D - 1);
        const uint8_t *stage = lds + (st & 1) * STAGE;
        const int first = sg0 + st * SG;
#pragma unroll
        for (int u = 0; u < SG; u++) {
            if (SG > 1 && first + u >= sg1) break;  // uniform
            u32x4 a[NB][4];
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const SkTile<T> &t = cur.t[u][b];
                if constexpr (T == AESIR_GGML_F16) {
#pragma unroll
                    for (int j = 0; j < 4; j++) a[b][j] = t.v[j];
                } else if constexpr (T == AESIR_GGML_Q8_0) {
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        unsigned o[8];
                        dequant_q8x4(t.v[h].x, t.d, o[0], o[1]);
                        dequant_q8x4(t.v[h].y, t.d, o[2], o[3]);
                        dequant_q8x4(t.v[h].z, t.d, o[4], o[5]);
                        dequant_q8x4(t.v[h].w, t.d, o[6], o[7]);
                        a[b][2 * h] = u32x4{o[0], o[1], o[2], o[3]};
                        a[b][2 * h + 1] = u32x4{o[4], o[5], o[6], o[7]};
                    }
                } else if constexpr (RAW) {
                    raw_tile_a<TR>(t.q, (first + u) & 1, g, a[b]);
                } else {
                    qf_tile_a<T>(t.q, kr, a[b]);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint8_t *xj = stage + (u * MT * 4 + j) * 1024 + g * 256 +
                                    ((c ^ ((8 * u + (sk_granule<T>(g, j) >> 1)) & 15)) << 4);
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    const u32x4 x = ld16(xj + m * 4096);
#pragma unroll
                    for (int b = 0; b < NB; b++) acc[b][m] = mfma16x16x32(a[b][j], x, acc[b][m]);
                }
            }
        }
        if (st + 1 < steps) {
            xstore(xnext, lds + ((st + 1) & 1) * STAGE);
            __syncthreads();
        }
    };
    // unrolled D times so that every buffer keeps its registers
    for (int base = 0; base < steps; base += D) {
#pragma unroll
        for (int j = 0; j < D; j++)
            if (base + j < steps) step(base + j, wb[j], wb[(j + D - 1) % D], xb[(j + D - 1) % D], xb[(j + 1) % D]);
    }

    // lane: rows 16 blk + 4 g + e (outputs n), activation row 16 m + c
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int n = (blk0 + b) * 16 + 4 * g;
        if (n >= N) continue;
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const int row = 16 * m + c;
            if (row >= M) continue;
            const f32x4 v = acc[b][m];
            const int left = N - n < 4 ? N - n : 4;
            if (splits > 1) {
                float *p = P + ((int64_t)z * M + row) * ldp + n;
                if (left == 4 && (ldp & 3) == 0) *reinterpret_cast<f32x4 *>(p) = v;
                else
                    for (int e = 0; e < left; e++) p[e] = v[e];
            } else if (epi == kEpiSwiglu) {  // N even: pairs (gate, up)
                h16 *o = C + row * ldc + n / 2;
                o[0] = hmul((h16)v[1], silu_h((h16)v[0]));
                if (left == 4) o[1] = hmul((h16)v[3], silu_h((h16)v[2]));
            } else {
                h16 *o = C + row * ldc + n;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (e < left) o[e] = epi == kEpiResidual ? hadd((h16)v[e], o[e]) : (h16)v[e];
            }
        }
    }
}

}  // namespace aesir
