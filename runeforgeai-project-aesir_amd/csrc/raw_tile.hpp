// One lane's share of a 16-row x 128-k tile read straight from packed GGUF blocks: row lane % 16,
// weights 32 (lane / 16) .. + 31 of the segment, dequantized to the four natural-order A operands
// (weights 8 j .. + 7 of the share) with the weight rules of qf_tile.hpp, so the f16 values are those
// of the repacked planes and of gguf_dequant_kernel. Every 32-weight share lies in one block (or one
// 32-weight part of a super-block), so a lane reads its quants with 8- and 16-byte loads at the
// block's own alignment (2 bytes and up; gfx950 global loads take any) and its scales beside them.
#pragma once

#include "qf_tile.hpp"

namespace aesir {

struct __attribute__((packed, aligned(2))) RawU16 { uint16_t v; };
struct __attribute__((packed, aligned(2))) RawU32 { uint32_t v; };
struct __attribute__((packed, aligned(2))) RawU64 { uint64_t v; };
struct __attribute__((packed, aligned(2))) RawU128 { u32x4 v; };
__device__ __forceinline__ unsigned raw16(const uint8_t *p) { return reinterpret_cast<const RawU16 *>(p)->v; }
__device__ __forceinline__ unsigned raw32(const uint8_t *p) { return reinterpret_cast<const RawU32 *>(p)->v; }
__device__ __forceinline__ u32x4 raw128(const uint8_t *p) { return reinterpret_cast<const RawU128 *>(p)->v; }

constexpr int raw_block_bytes(int t) {
    switch (t) {
        case AESIR_GGML_Q4_0: return 18;
        case AESIR_GGML_Q4_1: return 20;
        case AESIR_GGML_Q5_0: return 22;
        case AESIR_GGML_Q5_1: return 24;
        case AESIR_GGML_Q8_0: return 34;
        case AESIR_GGML_Q2_K: return 84;
        case AESIR_GGML_Q3_K: return 110;
        case AESIR_GGML_Q4_K: return 144;
        case AESIR_GGML_Q5_K: return 176;
        default: return 210;  // Q6_K
    }
}
constexpr bool raw_super(int t) {  // blocks of 256 weights
    return t == AESIR_GGML_Q2_K || t == AESIR_GGML_Q3_K || t == AESIR_GGML_Q4_K || t == AESIR_GGML_Q5_K || t == AESIR_GGML_Q6_K;
}

// As loaded: quant bytes (16 or 32), high-bit bytes, and the scale words.
template <int T>
struct RawTile {
    u32x4 q[2];   // Q4_0 .. Q5_1: q[0] only
    u32x4 h[2];   // Q5_K / Q6_K / Q3_K: high-bit bytes of the 32 weights; Q5_0 / Q5_1: h[0].x
    u32x4 s;      // scale fields
};

// blk: the block holding the share (the super-block of segment sg, or block 4 sg + g); half: sg & 1.
template <int T>
__device__ __forceinline__ void raw_load(RawTile<T> &t, const uint8_t *blk, int half, int g) {
    if constexpr (T == AESIR_GGML_Q4_0) {
        t.s.x = raw16(blk);
        t.q[0] = raw128(blk + 2);
    } else if constexpr (T == AESIR_GGML_Q4_1) {
        t.s.x = raw32(blk);
        t.q[0] = raw128(blk + 4);
    } else if constexpr (T == AESIR_GGML_Q5_0) {
        t.s.x = raw16(blk);
        t.h[0].x = raw32(blk + 2);
        t.q[0] = raw128(blk + 6);
    } else if constexpr (T == AESIR_GGML_Q5_1) {
        t.s.x = raw32(blk);
        t.h[0].x = raw32(blk + 4);
        t.q[0] = raw128(blk + 8);
    } else if constexpr (T == AESIR_GGML_Q8_0) {
        t.s.x = raw16(blk);
        t.q[0] = raw128(blk + 2);
        t.q[1] = raw128(blk + 18);
    } else if constexpr (T == AESIR_GGML_Q4_K || T == AESIR_GGML_Q5_K) {
        // part 4 half + g of eight: nibble bytes 32 (part / 2) .., low or high
        const uint8_t *qs = blk + (T == AESIR_GGML_Q4_K ? 16 : 48) + 64 * half + 32 * (g >> 1);
        t.s = raw128(blk);
        if constexpr (T == AESIR_GGML_Q5_K) {
            t.h[0] = raw128(blk + 16);
            t.h[1] = raw128(blk + 32);
        }
        t.q[0] = raw128(qs);
        t.q[1] = raw128(qs + 16);
    } else if constexpr (T == AESIR_GGML_Q6_K) {
        const uint8_t *ql = blk + 64 * half + 32 * (g & 1), *qh = blk + 128 + 32 * half;
        t.q[0] = raw128(ql);
        t.q[1] = raw128(ql + 16);
        t.h[0] = raw128(qh);
        t.h[1] = raw128(qh + 16);
        t.s.x = raw16(blk + 192 + 8 * half + 2 * g);  // int8 scales of the two 16-weight parts
        t.s.y = raw16(blk + 208);
    } else if constexpr (T == AESIR_GGML_Q2_K) {
        const uint8_t *qs = blk + 16 + 32 * half;
        t.q[0] = raw128(qs);
        t.q[1] = raw128(qs + 16);
        t.s.x = raw16(blk + 8 * half + 2 * g);  // scale | min << 4 bytes of the two parts
        t.s.y = raw32(blk + 80);
    } else {  // Q3_K
        const uint8_t *qs = blk + 32 + 32 * half;
        t.h[0] = raw128(blk);
        t.h[1] = raw128(blk + 16);
        t.q[0] = raw128(qs);
        t.q[1] = raw128(qs + 16);
        t.s.x = raw32(blk + 96);
        t.s.y = raw32(blk + 100);
        t.s.z = raw32(blk + 104);
        t.s.w = raw16(blk + 108);
    }
}

// Word i (0..7) of the share's unsigned quantized values, one byte per weight 4 i .. + 3.
template <int T>
__device__ __forceinline__ unsigned raw_qword(const RawTile<T> &t, int i, int half, int g) {
    if constexpr (T == AESIR_GGML_Q4_0 || T == AESIR_GGML_Q4_1 || T == AESIR_GGML_Q5_0 || T == AESIR_GGML_Q5_1) {
        unsigned v = (i < 4 ? t.q[0][i] : t.q[0][i - 4] >> 4) & 0x0f0f0f0fu;
        if constexpr (T == AESIR_GGML_Q5_0 || T == AESIR_GGML_Q5_1)  // four fifth bits, one per byte at bit 4
            v |= ((((t.h[0].x >> (4 * i)) & 15u) * 0x00204081u) & 0x01010101u) << 4;
        return v;
    } else if constexpr (T == AESIR_GGML_Q4_K || T == AESIR_GGML_Q5_K) {
        unsigned v = (t.q[i >> 2][i & 3] >> (4 * (g & 1))) & 0x0f0f0f0fu;
        if constexpr (T == AESIR_GGML_Q5_K) v |= ((t.h[i >> 2][i & 3] >> (4 * half + g)) & 0x01010101u) << 4;
        return v;
    } else if constexpr (T == AESIR_GGML_Q6_K) {
        const unsigned lo = (t.q[i >> 2][i & 3] >> (4 * (g >> 1))) & 0x0f0f0f0fu;
        return lo | (((t.h[i >> 2][i & 3] >> (2 * g)) & 0x03030303u) << 4);
    } else if constexpr (T == AESIR_GGML_Q2_K) {
        return (t.q[i >> 2][i & 3] >> (2 * g)) & 0x03030303u;
    } else if constexpr (T == AESIR_GGML_Q3_K) {  // q + 4
        return ((t.q[i >> 2][i & 3] >> (2 * g)) & 0x03030303u) |
               (((t.h[i >> 2][i & 3] >> (4 * half + g)) & 0x01010101u) << 2);
    } else {
        return 0u;
    }
}

// 6-bit scale and min of part sb of a Q4_K / Q5_K super-block from its header words (d | dmin << 16,
// then the 12 packed bytes), as the pair (scale, min) of exact f16 values.
__device__ __forceinline__ h16x2 raw_k_scale_min(u32x4 s, int sb) {
    const int sh = 8 * (sb & 3);
    const unsigned a = s.y >> sh, b = s.z >> sh, c = s.w >> sh;  // bytes sb % 4, 4 + sb % 4, 8 + sb % 4
    const unsigned sc = sb < 4 ? a & 63u : (c & 15u) | (((a >> 6) & 3u) << 4);
    const unsigned mn = sb < 4 ? b & 63u : ((c >> 4) & 15u) | (((b >> 6) & 3u) << 4);
    return as_h2((sc | (mn << 16)) | kMagic) - h16x2{(h16)1024.0f, (h16)1024.0f};
}

template <int T>
__device__ __forceinline__ void raw_tile_a(const RawTile<T> &t, int half, int g, u32x4 (&a)[4]) {
    unsigned w[16];  // natural pairs
    if constexpr (T == AESIR_GGML_Q8_0) {
        const h16 d = bits_to_h((uint16_t)t.s.x);
#pragma unroll
        for (int i = 0; i < 8; i++) dequant_q8x4(t.q[i >> 2][i & 3], d, w[2 * i], w[2 * i + 1]);
    } else {
        // per 16-weight part r: the scale pair and the negated offset (or added min) pair
        h16x2 aa[2], nbb[2];
        if constexpr (T == AESIR_GGML_Q4_0 || T == AESIR_GGML_Q5_0) {
            const h16 d = bits_to_h((uint16_t)t.s.x);
            aa[0] = aa[1] = h16x2{d, d};
        } else if constexpr (qf_dm<T>()) {
            const h16x2 dm = as_h2(t.s.x);
            aa[0] = aa[1] = h16x2{dm.x, dm.x};
            nbb[0] = nbb[1] = h16x2{dm.y, dm.y};
        } else if constexpr (qf_kq<T>()) {
            const h16x2 ab = q4k_scales(as_h2(t.s.x), raw_k_scale_min(t.s, 4 * half + g));
            aa[0] = aa[1] = h16x2{ab.x, ab.x};
            nbb[0] = nbb[1] = h16x2{-ab.y, -ab.y};
        } else if constexpr (T == AESIR_GGML_Q2_K) {
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const unsigned x = t.s.x >> (8 * r);
                const h16x2 ab = q4k_scales(as_h2(t.s.y), h16x2{(h16)(float)(x & 15u), (h16)(float)((x >> 4) & 15u)});
                aa[r] = h16x2{ab.x, ab.x};
                nbb[r] = h16x2{-ab.y, -ab.y};
            }
        } else if constexpr (T == AESIR_GGML_Q3_K) {
            // 6-bit scales of parts 8 half + 2 g + r: low 4 bits in bytes 0-7 (low nibbles of parts 0-7,
            // high of 8-15), high 2 bits in bytes 8-11
            const h16 d = bits_to_h((uint16_t)t.s.w);
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int is = 2 * g + r;  // part within its half
                const unsigned lo = ((is < 4 ? t.s.x : t.s.y) >> (8 * (is & 3) + 4 * half)) & 15u;
                const unsigned hi = (t.s.z >> (8 * (is & 3) + 4 * half + 2 * (is >> 2))) & 3u;
                const h16 x = q6k_scale(d, (int)(lo | (hi << 4)) - 32);
                aa[r] = h16x2{x, x};
            }
        } else {  // Q6_K
            const h16 d = bits_to_h((uint16_t)t.s.y);
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const h16 x = q6k_scale(d, (int)(int8_t)(t.s.x >> (8 * r)));
                aa[r] = h16x2{x, x};
            }
        }
        constexpr float off = T == AESIR_GGML_Q4_0 ? 1032.0f : T == AESIR_GGML_Q5_0 ? 1040.0f : T == AESIR_GGML_Q6_K ? 1056.0f
                              : T == AESIR_GGML_Q3_K ? 1028.0f : 1024.0f;
        const h16x2 bias = {(h16)off, (h16)off};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const unsigned q = raw_qword<T>(t, i, half, g);
#pragma unroll
            for (int p = 0; p < 2; p++) {  // two bytes under the f16 exponent of 1024: exact
                const h16x2 v = as_h2(__builtin_amdgcn_perm(0x64646464u, q, p == 0 ? 0x04010400u : 0x04030402u)) - bias;
                const int r = i >> 2;
                if constexpr (T == AESIR_GGML_Q4_0 || T == AESIR_GGML_Q5_0) w[2 * i + p] = h2_bits(q4_0_w2(v, aa[r]));
                else if constexpr (qf_dm<T>()) w[2 * i + p] = h2_bits(q4_1_w2(v, aa[r], nbb[r]));
                else if constexpr (qf_kq<T>() || T == AESIR_GGML_Q2_K) w[2 * i + p] = h2_bits(q4k_w2(v, aa[r], nbb[r]));
                else w[2 * i + p] = h2_bits(q6k_w2(v, aa[r]));
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) a[j] = u32x4{w[4 * j], w[4 * j + 1], w[4 * j + 2], w[4 * j + 3]};
}

}  // namespace aesir
