// One lane's share of the repacked 2- to 6-bit weight planes and its dequantization, shared by the
// decode GEMV and wide-tile GEMM (quant.hip) and the short-chunk GEMM (skinny.hip): the type
// families, the weight rules, records, matrix-core tiles (QTile) and their A operands.
#pragma once

#include <type_traits>

#include "device.hpp"
#include "kernels.hpp"

namespace aesir {

constexpr int kRec = 16;                  // weights per record
constexpr int kSeg = 128;                 // weights per tile row (8 records)
constexpr unsigned kMagic = 0x64006400u;  // f16 1024 in both halves


// Type families of the repacked layout: a fifth-bit word per record pair (Q5_0, Q5_1, Q5_K); an
// f16 (d, m) pair per 32 weights (Q4_1, Q5_1); the K-quant 6-bit (scale, min) bytes with a
// super-block (d, dmin) pair (Q4_K, Q5_K).
template <int T>
constexpr bool qf_hb5() {
    return T == AESIR_GGML_Q5_0 || T == AESIR_GGML_Q5_1 || T == AESIR_GGML_Q5_K;
}
template <int T>
constexpr bool qf_dm() {
    return T == AESIR_GGML_Q4_1 || T == AESIR_GGML_Q5_1;
}
template <int T>
constexpr bool qf_kq() {
    return T == AESIR_GGML_Q4_K || T == AESIR_GGML_Q5_K;
}
template <int T>
constexpr bool qf_crumb() {
    return T == AESIR_GGML_Q2_K || T == AESIR_GGML_Q3_K;
}

// Crumb records (Q2_K, Q3_K). Nibble i of a record's crumb word holds the low 2 bits of nibble i
// of its two nibble words (bits 0-1: word 0, bits 2-3: word 1), so each word is one shift and mask
// away. The Q3_K third bits of a record pair share one word: nibble i holds them for nibble i of
// the odd record's words 0 and 1 (bits 0, 1) and the even record's (bits 2, 3); shifting the word
// left by 2 for the odd record puts its bits where the even record's are.
constexpr unsigned kCrumbMask = 0x33333333u, kThirdMask = 0x44444444u;
__host__ __device__ __forceinline__ unsigned crumb_word(unsigned w0, unsigned w1) {
    return (w0 & kCrumbMask) | ((w1 & kCrumbMask) << 2);
}
__host__ __device__ __forceinline__ unsigned third_bits(unsigned w0, unsigned w1, int odd) {
    return odd ? ((w0 & kThirdMask) >> 2) | ((w1 & kThirdMask) >> 1) : (w0 & kThirdMask) | ((w1 & kThirdMask) << 1);
}
// Nibble words of a crumb record; h: the pair's third-bit word shifted to the even record's
// positions (0 for Q2_K).
__device__ __forceinline__ u32x2 crumb_nibbles(unsigned c, unsigned h) {
    return u32x2{(c & kCrumbMask) | (h & kThirdMask), ((c >> 2) & kCrumbMask) | ((h >> 1) & kThirdMask)};
}


// Nibble pair f of a record holds weights a and a + 2, a = {0, 1, 4, 5, 8, 9, 12, 13}[f]: pairs
// 0-3 are low nibbles, 4-7 high nibbles. In the Q6_K high-bit word, pair f's two 2-bit fields sit
// 16 bits apart at qf_hb_off(f) = {0, 2, 8, 10}[f & 3] + 4 (f >> 2) and 16 above, so that one
// shift by 4 - {0, 2, 8, 10}[f & 3] serves a low pair (fields to bits 4, 20, above its nibbles)
// and a high pair (to bits 8, 24, above its 16-scaled nibbles).
__host__ __device__ __forceinline__ int qf_hb_off(int f) { return ((f & 1) << 1) + ((f & 2) << 2) + ((f >> 2) << 2); }
// The 5-bit types keep a record pair's fifth bits in one word: the even record's at the low bit
// of each Q6_K field position, the odd record's one above, so that shifting the word right by
// the record's parity turns it into a Q6_K word whose fields hold only their low bit.

// ------------------------------------------------------------------ weight arithmetic

// Scales of the f16 weight rules from the block fields (correctly rounded f16 products of exact
// operands): Q4_K (f16(d sc), f16(dmin m)), Q6_K f16(d sc).
__device__ __forceinline__ h16x2 q4k_scales(h16x2 d_dmin, h16x2 sc_m) { return d_dmin * sc_m; }
__device__ __forceinline__ h16 q6k_scale(h16 d, int sc) { return hmul(d, (h16)(float)sc); }
// Weight pairs from exact f16 pairs of quantized values: Q4_0 q - 8 (times d), Q4_K q (a q - b,
// one fused rounding), Q6_K q - 32 (times a).
__device__ __forceinline__ h16x2 q4_0_w2(h16x2 q8, h16x2 dd) { return q8 * dd; }
__device__ __forceinline__ h16x2 q4k_w2(h16x2 q, h16x2 aa, h16x2 nbb) { return __builtin_elementwise_fma(q, aa, nbb); }
__device__ __forceinline__ h16x2 q6k_w2(h16x2 q32, h16x2 aa) { return q32 * aa; }
// Q4_1 / Q5_1 weight pairs f16(f16(q d) + m): two roundings, the reference's f16 multiply then
// add (the library is built without multiply-add contraction).
__device__ __forceinline__ h16x2 q4_1_w2(h16x2 q, h16x2 dd, h16x2 mm) { return q * dd + mm; }

// ------------------------------------------------------------------ one record

template <int T>
struct QRec;
template <>
struct QRec<AESIR_GGML_Q4_0> {
    u32x2 nib;
    h16 d;
};
template <>
struct QRec<AESIR_GGML_Q4_K> {
    u32x2 nib;
    unsigned scm;  // scale | min << 8
    unsigned dd;   // f16 d | f16 dmin << 16
};
template <>
struct QRec<AESIR_GGML_Q6_K> {
    u32x2 nib;
    unsigned hb;
    int sc;
    h16 d;
};
template <>
struct QRec<AESIR_GGML_Q4_1> {
    u32x2 nib;
    unsigned dm;  // f16 d | f16 m << 16
    unsigned hb;  // unused
};
template <>
struct QRec<AESIR_GGML_Q5_1> {
    u32x2 nib;
    unsigned dm;
    unsigned hb;  // the fifth bits, shifted to the even record's positions
};
template <>
struct QRec<AESIR_GGML_Q5_0> {
    u32x2 nib;
    h16 d;
    unsigned hb;
};
template <>
struct QRec<AESIR_GGML_Q5_K> {
    u32x2 nib;
    unsigned scm;
    unsigned dd;
    unsigned hb;
};
template <>
struct QRec<AESIR_GGML_Q2_K> {
    u32x2 nib;
    unsigned scm;  // GGML's byte: scale | min << 4
    unsigned dd;   // f16 d | f16 dmin << 16
};
template <>
struct QRec<AESIR_GGML_Q3_K> {
    u32x2 nib;
    int sc;
    h16 d;
};

// Record `rec` of plane row `prow`.
template <int T>
__device__ __forceinline__ QRec<T> qf_load(const QFMat &w, int64_t prow, int64_t rec, int64_t K) {
    QRec<T> q;
    if constexpr (qf_crumb<T>()) {
        const uint8_t *pr = (const uint8_t *)w.nib + qf_qlane_off(prow, rec, K, qf_lane_bytes(T));
        const unsigned c = *reinterpret_cast<const uint32_t *>(pr + 4 * (rec & 1));
        unsigned h = 0u;
        if constexpr (T == AESIR_GGML_Q3_K) h = *reinterpret_cast<const uint32_t *>(pr + 8) << (2 * (rec & 1));
        q.nib = crumb_nibbles(c, h);
    } else {
        q.nib = *reinterpret_cast<const u32x2 *>((const uint8_t *)w.nib + qf_nib_off(prow, rec, K));
    }
    const uint8_t *s0 = (const uint8_t *)w.s0 + qf_s0_off(prow, rec, K, qf_s0_bytes(T));
    if constexpr (qf_hb5<T>())
        q.hb = *reinterpret_cast<const uint32_t *>((const uint8_t *)w.hb + qf_hb_pair_off(prow, rec, K, 4)) >> (rec & 1);
    if constexpr (T == AESIR_GGML_Q4_0 || T == AESIR_GGML_Q5_0) {
        q.d = *reinterpret_cast<const h16 *>(s0);
    } else if constexpr (qf_dm<T>()) {
        q.dm = *reinterpret_cast<const uint32_t *>(s0);
    } else if constexpr (qf_kq<T>()) {
        q.scm = *reinterpret_cast<const uint16_t *>(s0);
        q.dd = *reinterpret_cast<const uint32_t *>((const uint8_t *)w.s1 + qf_s1_off(prow, rec, K, 4));
    } else if constexpr (T == AESIR_GGML_Q2_K) {
        q.scm = s0[rec & 1];
        q.dd = *reinterpret_cast<const uint32_t *>((const uint8_t *)w.s1 + qf_s1_off(prow, rec, K, 4));
    } else if constexpr (T == AESIR_GGML_Q3_K) {
        q.sc = *reinterpret_cast<const int8_t *>(s0 + (rec & 1));
        q.d = *reinterpret_cast<const h16 *>((const uint8_t *)w.s1 + qf_s1_off(prow, rec, K, 2));
    } else {
        q.hb = *reinterpret_cast<const uint32_t *>((const uint8_t *)w.hb + qf_hbw_off(prow, rec, K));
        q.sc = *reinterpret_cast<const int8_t *>(s0 + (rec & 1));
        q.d = *reinterpret_cast<const h16 *>((const uint8_t *)w.s1 + qf_s1_off(prow, rec, K, 2));
    }
    return q;
}

// f16 pair (1024 + q_a, 1024 + q_b) of nibble pair f (weights a, a + 2 of the record), with the
// Q6_K high bits OR-ed in when given.
__device__ __forceinline__ unsigned qf_pair(u32x2 nib, int f) {
    const int sh = (f & 1) * 8 + (f >> 2) * 4;
    return (((f >> 1) & 1 ? nib.y : nib.x) >> sh) & 0x000F000Fu;
}
__device__ __forceinline__ unsigned qf_hb_pair(unsigned hb, int f) {
    const int s = 4 - qf_hb_off(f);
    return (s >= 0 ? hb << s : hb >> -s) & 0x00300030u;
}
// The fifth bits of nibble pair f (value 16) from a 5-bit record's shifted word.
__device__ __forceinline__ unsigned qf_hb5_pair(unsigned hb, int f) {
    const int s = 4 - qf_hb_off(f);
    return (s >= 0 ? hb << s : hb >> -s) & 0x00100010u;
}

// Exact f16 pairs of the record's quantized values, pair order: Q4_0 q - 8, Q5_0 q - 16, Q4_1 /
// Q5_1 / Q4_K / Q5_K q, Q6_K q - 32.
template <int T>
__device__ __forceinline__ h16x2 qf_qpair(const QRec<T> &q, int f) {
    if constexpr (T == AESIR_GGML_Q4_0) {
        const h16x2 bias = {(h16)1032.0f, (h16)1032.0f};
        return as_h2(qf_pair(q.nib, f) | kMagic) - bias;
    } else if constexpr (qf_hb5<T>()) {
        const float b = T == AESIR_GGML_Q5_0 ? 1040.0f : 1024.0f;
        const h16x2 bias = {(h16)b, (h16)b};
        return as_h2(qf_pair(q.nib, f) | qf_hb5_pair(q.hb, f) | kMagic) - bias;
    } else if constexpr (T == AESIR_GGML_Q4_1 || T == AESIR_GGML_Q4_K || T == AESIR_GGML_Q2_K) {
        const h16x2 bias = {(h16)1024.0f, (h16)1024.0f};
        return as_h2(qf_pair(q.nib, f) | kMagic) - bias;
    } else if constexpr (T == AESIR_GGML_Q3_K) {
        const h16x2 bias = {(h16)1028.0f, (h16)1028.0f};
        return as_h2(qf_pair(q.nib, f) | kMagic) - bias;
    } else {
        const h16x2 bias = {(h16)1056.0f, (h16)1056.0f};
        return as_h2(qf_pair(q.nib, f) | qf_hb_pair(q.hb, f) | kMagic) - bias;
    }
}

// Natural-order weights from pair-order pairs: o[0] holds weights 0..7, o[1] 8..15.
__device__ __forceinline__ void qf_unpair(const unsigned (&wp)[8], u32x4 (&o)[2]) {
#pragma unroll
    for (int c = 0; c < 2; c++) {
        o[c].x = __builtin_amdgcn_perm(wp[4 * c + 1], wp[4 * c + 0], 0x05040100u);
        o[c].y = __builtin_amdgcn_perm(wp[4 * c + 1], wp[4 * c + 0], 0x07060302u);
        o[c].z = __builtin_amdgcn_perm(wp[4 * c + 3], wp[4 * c + 2], 0x05040100u);
        o[c].w = __builtin_amdgcn_perm(wp[4 * c + 3], wp[4 * c + 2], 0x07060302u);
    }
}

// The record's 16 f16 weights in natural order.
template <int T>
__device__ __forceinline__ void qf_deq16(const QRec<T> &q, u32x4 (&o)[2]) {
    unsigned wp[8];
    h16x2 aa, nbb;
    if constexpr (T == AESIR_GGML_Q4_0 || T == AESIR_GGML_Q5_0) {
        aa = h16x2{q.d, q.d};
    } else if constexpr (qf_dm<T>()) {
        const h16x2 dm = as_h2(q.dm);
        aa = h16x2{dm.x, dm.x};
        nbb = h16x2{dm.y, dm.y};  // the added min
    } else if constexpr (T == AESIR_GGML_Q2_K) {
        const h16x2 ab = q4k_scales(as_h2(q.dd), h16x2{(h16)(float)(q.scm & 15u), (h16)(float)(q.scm >> 4)});
        aa = h16x2{ab.x, ab.x};
        nbb = h16x2{-ab.y, -ab.y};
    } else if constexpr (T == AESIR_GGML_Q3_K) {
        const h16 a = q6k_scale(q.d, q.sc);
        aa = h16x2{a, a};
    } else if constexpr (qf_kq<T>()) {
        const h16x2 sm = {(h16)(float)(q.scm & 0xffu), (h16)(float)(q.scm >> 8)};
        const h16x2 ab = q4k_scales(as_h2(q.dd), sm);
        aa = h16x2{ab.x, ab.x};
        nbb = h16x2{-ab.y, -ab.y};
    } else {
        const h16 a = q6k_scale(q.d, q.sc);
        aa = h16x2{a, a};
    }
#pragma unroll
    for (int f = 0; f < 8; f++) {
        const h16x2 v = qf_qpair(q, f);
        if constexpr (T == AESIR_GGML_Q4_0 || T == AESIR_GGML_Q5_0) wp[f] = h2_bits(q4_0_w2(v, aa));
        else if constexpr (qf_dm<T>()) wp[f] = h2_bits(q4_1_w2(v, aa, nbb));
        else if constexpr (qf_kq<T>() || T == AESIR_GGML_Q2_K) wp[f] = h2_bits(q4k_w2(v, aa, nbb));
        else wp[f] = h2_bits(q6k_w2(v, aa));
    }
    qf_unpair(wp, o);
}

// Runs F<T>() for the repacked type `type` (one of qf_type's).
template <class F>
inline void qf_switch(int32_t type, F &&f) {
    switch (type) {
        case AESIR_GGML_Q4_0: f(std::integral_constant<int, AESIR_GGML_Q4_0>{}); break;
        case AESIR_GGML_Q4_1: f(std::integral_constant<int, AESIR_GGML_Q4_1>{}); break;
        case AESIR_GGML_Q5_0: f(std::integral_constant<int, AESIR_GGML_Q5_0>{}); break;
        case AESIR_GGML_Q5_1: f(std::integral_constant<int, AESIR_GGML_Q5_1>{}); break;
        case AESIR_GGML_Q2_K: f(std::integral_constant<int, AESIR_GGML_Q2_K>{}); break;
        case AESIR_GGML_Q3_K: f(std::integral_constant<int, AESIR_GGML_Q3_K>{}); break;
        case AESIR_GGML_Q4_K: f(std::integral_constant<int, AESIR_GGML_Q4_K>{}); break;
        case AESIR_GGML_Q5_K: f(std::integral_constant<int, AESIR_GGML_Q5_K>{}); break;
        default: f(std::integral_constant<int, AESIR_GGML_Q6_K>{}); break;
    }
}

// Register-held constants: the and-or and packed-f16 forms below take a mask or bias from a
// register (one VOP3 instruction holds at most one literal), which the compiler does not arrange
// by itself; without them every nibble pair costs a shift, an AND and an OR.
__device__ __forceinline__ unsigned sreg(unsigned v) {
    unsigned r;
    asm("s_mov_b32 %0, %1" : "=s"(r) : "i"(v));
    return r;
}
__device__ __forceinline__ unsigned vreg(unsigned v) {
    unsigned r;
    asm("v_mov_b32 %0, %1" : "=v"(r) : "i"(v));
    return r;
}

struct QfRegs {
    unsigned lo, hi, magic;  // nibble masks 0x000F000F / 0x00F000F0, f16 1024 in both halves
    unsigned hlo, hhi;       // Q6_K high-bit masks 0x00300030 / 0x03000300
    unsigned flo, fhi;       // fifth-bit masks 0x00100010 / 0x01000100
    __device__ __forceinline__ static QfRegs make() {
        return QfRegs{sreg(0x000F000Fu), sreg(0x00F000F0u), vreg(kMagic), sreg(0x00300030u),
                      sreg(0x03000300u), sreg(0x00100010u), sreg(0x01000100u)};
    }
};

// One lane's share of a tile as loaded.
template <int T>
struct QTile;
template <>
struct QTile<AESIR_GGML_Q4_0> {
    u32x4 nib;
    unsigned s0;  // f16 d in the low half
};
template <>
struct QTile<AESIR_GGML_Q4_K> {
    u32x4 nib;
    unsigned s0;  // scale | min << 8
    unsigned s1;  // f16 d | f16 dmin << 16
};
template <>
struct QTile<AESIR_GGML_Q6_K> {
    u32x4 nib;
    u32x2 hb;     // high-bit words of the two records
    unsigned s0;  // int8 scales of the two records
    unsigned s1;  // f16 super-block d in the low half
};
template <>
struct QTile<AESIR_GGML_Q5_0> {
    u32x4 nib;
    unsigned s0;  // f16 d in the low half
    unsigned hb;  // fifth bits of the two records
};
template <>
struct QTile<AESIR_GGML_Q4_1> {
    u32x4 nib;
    unsigned s0;  // f16 d | f16 m << 16
};
template <>
struct QTile<AESIR_GGML_Q5_1> {
    u32x4 nib;
    unsigned s0;  // f16 d | f16 m << 16
    unsigned hb;
};
template <>
struct QTile<AESIR_GGML_Q5_K> {
    u32x4 nib;
    unsigned s0;  // scale | min << 8
    unsigned s1;  // f16 d | f16 dmin << 16
    unsigned hb;
};
template <>
struct QTile<AESIR_GGML_Q2_K> {
    u32x2 cr;     // crumb words of the two records
    unsigned s0;  // the two records' scale | min << 4 bytes
    unsigned s1;  // f16 d | f16 dmin << 16
};
template <>
struct QTile<AESIR_GGML_Q3_K> {
    u32x2 cr;     // crumb words of the two records
    unsigned hb;  // third bits of the record pair
    unsigned s0;  // int8 scales of the two records
    unsigned s1;  // f16 super-block d in the low half
};

// Buffer resources of a matrix's planes (range-checked loads, tile offsets in SGPRs).
struct QfRsrc {
    __amdgpu_buffer_rsrc_t nib, hb, s0, s1;
};

__device__ __forceinline__ QfRsrc qf_rsrc(const QFMat &w, int32_t type, int64_t prows, int64_t K) {
    QfRsrc r;
    r.nib = __builtin_amdgcn_make_buffer_rsrc((void *)w.nib, 0, (int)(prows * qf_plane_row_bytes(type, 0, K)), 0x00020000);
    r.hb = __builtin_amdgcn_make_buffer_rsrc((void *)w.hb, 0, (int)(prows * qf_plane_row_bytes(type, 1, K)), 0x00020000);
    r.s0 = __builtin_amdgcn_make_buffer_rsrc((void *)w.s0, 0, (int)(prows * qf_plane_row_bytes(type, 2, K)), 0x00020000);
    r.s1 = __builtin_amdgcn_make_buffer_rsrc((void *)w.s1, 0, (int)(prows * qf_plane_row_bytes(type, 3, K)), 0x00020000);
    return r;
}

// Tile `tile` (wave-uniform); s1v / s1s: the lane's and the tile's byte offsets in the s1 plane.
template <int T>
__device__ __forceinline__ QTile<T> qf_tile_load(const QfRsrc &r, int tile, int lane, int s1v, int s1s) {
    QTile<T> q;
    if constexpr (T == AESIR_GGML_Q2_K) {
        q.cr = __builtin_amdgcn_raw_buffer_load_b64(r.nib, lane * 8, tile * 512, 2);
    } else if constexpr (T == AESIR_GGML_Q3_K) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b96(r.nib, lane * 12, tile * 768, 2);
        q.cr = u32x2{(unsigned)v[0], (unsigned)v[1]};
        q.hb = (unsigned)v[2];
    } else {
        q.nib = __builtin_amdgcn_raw_buffer_load_b128(r.nib, lane * 16, tile * 1024, 2);
    }
    if constexpr (qf_dm<T>())
        q.s0 = __builtin_amdgcn_raw_buffer_load_b32(r.s0, lane * 4, tile * 256, 0);
    else
        q.s0 = __builtin_amdgcn_raw_buffer_load_b16(r.s0, lane * 2, tile * 128, 0);
    if constexpr (qf_hb5<T>()) q.hb = __builtin_amdgcn_raw_buffer_load_b32(r.hb, lane * 4, tile * 256, 0);
    if constexpr (qf_kq<T>() || T == AESIR_GGML_Q2_K) q.s1 = __builtin_amdgcn_raw_buffer_load_b32(r.s1, s1v, s1s, 0);
    if constexpr (T == AESIR_GGML_Q3_K) q.s1 = __builtin_amdgcn_raw_buffer_load_b16(r.s1, s1v, s1s, 0);
    if constexpr (T == AESIR_GGML_Q6_K) {
        q.hb = __builtin_amdgcn_raw_buffer_load_b64(r.hb, lane * 8, tile * 512, 2);
        q.s1 = __builtin_amdgcn_raw_buffer_load_b16(r.s1, s1v, s1s, 0);
    }
    return q;
}

// The four A operands of a lane's tile share: operand j from nibble word j (record j / 2, bytes
// 4 (j % 2) .. + 3), as the pairs (v & lo), (v >> 8 & lo), (v & hi), (v >> 8 & hi), i.e. the
// weights {0, 2, 1, 3, 8, 10, 9, 11} + 4 (j % 2) of the record. Values exact in f16 until the
// weight rule's single rounding: Q4_0 turns 1024 + q into q - 8 by adding -1032 and 1024 + 16 q
// by (.) / 16 - 72; Q4_K into q by -1024 and (.) / 16 - 64; Q6_K into q - 32 by -1056 and
// (.) / 16 - 96, its high bits OR-ed in from the record's hb word (shifted by 4, 2, -4, -6 for
// the four pair positions of the record).
template <int T>
__device__ __forceinline__ void qf_tile_a(const QTile<T> &q, const QfRegs &k, u32x4 (&a)[4]) {
    unsigned nw[4];
    if constexpr (qf_crumb<T>()) {  // spread the crumbs (and Q3_K's third bits) into nibble words
        unsigned h = 0u;
        if constexpr (T == AESIR_GGML_Q3_K) h = q.hb;
        const u32x2 e = crumb_nibbles(q.cr.x, h), o = crumb_nibbles(q.cr.y, h << 2);
        nw[0] = e.x;
        nw[1] = e.y;
        nw[2] = o.x;
        nw[3] = o.y;
    } else {
        nw[0] = q.nib.x;
        nw[1] = q.nib.y;
        nw[2] = q.nib.z;
        nw[3] = q.nib.w;
    }
    const h16x2 s16 = {(h16)0.0625f, (h16)0.0625f};
    if constexpr (T == AESIR_GGML_Q4_0) {
        const h16 d = bits_to_h((uint16_t)(q.s0 & 0xffffu));
        const h16x2 dd = {d, d};
        const h16x2 blo = {(h16)-1032.0f, (h16)-1032.0f}, bhi = {(h16)-72.0f, (h16)-72.0f};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const unsigned v = nw[j], t = v >> 8;
            a[j].x = h2_bits(q4_0_w2(as_h2((v & k.lo) | k.magic) + blo, dd));
            a[j].y = h2_bits(q4_0_w2(as_h2((t & k.lo) | k.magic) + blo, dd));
            a[j].z = h2_bits(q4_0_w2(__builtin_elementwise_fma(as_h2((v & k.hi) | k.magic), s16, bhi), dd));
            a[j].w = h2_bits(q4_0_w2(__builtin_elementwise_fma(as_h2((t & k.hi) | k.magic), s16, bhi), dd));
        }
    } else if constexpr (T == AESIR_GGML_Q2_K || T == AESIR_GGML_Q3_K) {
        // a scale per record (16 weights): the lane's two records have their own; the values are
        // q (Q2_K) or q - 4 (Q3_K, its nibble holding q + 4), then Q4_K's or Q6_K's rule
        constexpr float off = T == AESIR_GGML_Q3_K ? 4.0f : 0.0f;
        const h16x2 blo = {(h16)(-1024.0f - off), (h16)(-1024.0f - off)}, bhi = {(h16)(-64.0f - off), (h16)(-64.0f - off)};
        h16x2 aa[2], nbb[2];
        if constexpr (T == AESIR_GGML_Q2_K) {
            const h16x2 b1024 = {(h16)-1024.0f, (h16)-1024.0f};
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const unsigned x = q.s0 >> (8 * r);  // scale | min << 4
                const h16x2 sm = as_h2(((x & 15u) | ((x & 0xF0u) << 12)) | k.magic) + b1024;
                const h16x2 ab = q4k_scales(as_h2(q.s1), sm);
                aa[r] = h16x2{ab.x, ab.x};
                nbb[r] = h16x2{-ab.y, -ab.y};
            }
        } else {
            const h16x2 b1152 = {(h16)-1152.0f, (h16)-1152.0f};
            const h16x2 sc = as_h2(__builtin_amdgcn_perm(0u, q.s0 ^ 0x8080u, 0x0c010c00u) | k.magic) + b1152;
            const h16 d = bits_to_h((uint16_t)(q.s1 & 0xffffu));
            const h16x2 a01 = h16x2{d, d} * sc;  // (f16(d sc0), f16(d sc1))
            aa[0] = h16x2{a01.x, a01.x};
            aa[1] = h16x2{a01.y, a01.y};
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = j >> 1;
            auto rule = [&](h16x2 v) {
                if constexpr (T == AESIR_GGML_Q2_K) return q4k_w2(v, aa[r], nbb[r]);
                else return q6k_w2(v, aa[r]);
            };
            const unsigned v = nw[j], t = v >> 8;
            a[j].x = h2_bits(rule(as_h2((v & k.lo) | k.magic) + blo));
            a[j].y = h2_bits(rule(as_h2((t & k.lo) | k.magic) + blo));
            a[j].z = h2_bits(rule(__builtin_elementwise_fma(as_h2((v & k.hi) | k.magic), s16, bhi)));
            a[j].w = h2_bits(rule(__builtin_elementwise_fma(as_h2((t & k.hi) | k.magic), s16, bhi)));
        }
    } else if constexpr (T != AESIR_GGML_Q6_K) {
        // Q4_1, Q5_0, Q5_1, Q4_K, Q5_K: the exact quantized pairs (q - 16 for Q5_0, else q), the
        // fifth bits OR-ed in at value 16 (low nibbles) or 256 (16-scaled high nibbles), then the
        // weight rule with the record pair's scales
        constexpr bool h5 = qf_hb5<T>();
        constexpr float off = T == AESIR_GGML_Q5_0 ? 16.0f : 0.0f;
        const h16x2 blo = {(h16)(-1024.0f - off), (h16)(-1024.0f - off)}, bhi = {(h16)(-64.0f - off), (h16)(-64.0f - off)};
        h16x2 aa, nbb;
        if constexpr (qf_kq<T>()) {
            const h16x2 b1024 = {(h16)-1024.0f, (h16)-1024.0f};
            // (scale, min) bytes into the low byte of each half, then exact through the 1024 exponent
            const h16x2 sm = as_h2(__builtin_amdgcn_perm(0u, q.s0, 0x0c010c00u) | k.magic) + b1024;
            const h16x2 ab = q4k_scales(as_h2(q.s1), sm);
            aa = h16x2{ab.x, ab.x};
            nbb = h16x2{-ab.y, -ab.y};
        } else if constexpr (qf_dm<T>()) {
            const h16x2 dm = as_h2(q.s0);
            aa = h16x2{dm.x, dm.x};
            nbb = h16x2{dm.y, dm.y};
        } else {
            const h16 d = bits_to_h((uint16_t)(q.s0 & 0xffffu));
            aa = h16x2{d, d};
        }
        auto rule = [&](h16x2 v) {
            if constexpr (qf_kq<T>()) return q4k_w2(v, aa, nbb);
            else if constexpr (qf_dm<T>()) return q4_1_w2(v, aa, nbb);
            else return q4_0_w2(v, aa);
        };
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const unsigned v = nw[j], t = v >> 8;
            unsigned fa = 0u, fb = 0u, ga = 0u, gb = 0u;  // fifth bits of the four pairs
            if constexpr (h5) {
                const unsigned h = (j >> 1) ? q.hb >> 1 : q.hb;  // the record's bits at the even positions
                const unsigned ha = (j & 1) == 0 ? h << 4 : h >> 4, hb = (j & 1) == 0 ? h << 2 : h >> 6;
                fa = ha & k.flo;
                ga = ha & k.fhi;
                fb = hb & k.flo;
                gb = hb & k.fhi;
            }
            a[j].x = h2_bits(rule(as_h2(fa | ((v & k.lo) | k.magic)) + blo));
            a[j].y = h2_bits(rule(as_h2(fb | ((t & k.lo) | k.magic)) + blo));
            a[j].z = h2_bits(rule(__builtin_elementwise_fma(as_h2(ga | ((v & k.hi) | k.magic)), s16, bhi)));
            a[j].w = h2_bits(rule(__builtin_elementwise_fma(as_h2(gb | ((t & k.hi) | k.magic)), s16, bhi)));
        }
    } else {
        const h16x2 blo = {(h16)-1056.0f, (h16)-1056.0f}, bhi = {(h16)-96.0f, (h16)-96.0f};
        const h16x2 b1152 = {(h16)-1152.0f, (h16)-1152.0f};
        // int8 scales of the two records: byte ^ 0x80 under the 1024 exponent reads 1152 + sc
        const h16x2 sc = as_h2(__builtin_amdgcn_perm(0u, q.s0 ^ 0x8080u, 0x0c010c00u) | k.magic) + b1152;
        const h16 d = bits_to_h((uint16_t)(q.s1 & 0xffffu));
        const h16x2 a01 = h16x2{d, d} * sc;  // (f16(d sc0), f16(d sc1))
        const unsigned hw[2] = {q.hb.x, q.hb.y};
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const h16x2 aa = r == 0 ? h16x2{a01.x, a01.x} : h16x2{a01.y, a01.y};
            const unsigned h = hw[r];
#pragma unroll
            for (int wd = 0; wd < 2; wd++) {
                const int j = 2 * r + wd;
                const unsigned v = nw[j], t = v >> 8;
                const unsigned ha = wd == 0 ? h << 4 : h >> 4, hb = wd == 0 ? h << 2 : h >> 6;
                a[j].x = h2_bits(q6k_w2(as_h2((ha & k.hlo) | ((v & k.lo) | k.magic)) + blo, aa));
                a[j].y = h2_bits(q6k_w2(as_h2((hb & k.hlo) | ((t & k.lo) | k.magic)) + blo, aa));
                a[j].z = h2_bits(q6k_w2(__builtin_elementwise_fma(as_h2((ha & k.hhi) | ((v & k.hi) | k.magic)), s16, bhi), aa));
                a[j].w = h2_bits(q6k_w2(__builtin_elementwise_fma(as_h2((hb & k.hhi) | ((t & k.hi) | k.magic)), s16, bhi), aa));
            }
        }
    }
}

// x of one record (natural order, x[0]: elements 0..7, x[1]: 8..15) -> the B operands of its two
// nibble words: o[0] = elements {0, 2, 1, 3, 8, 10, 9, 11}, o[1] = the same + 4.
__device__ __forceinline__ void qf_perm_rec(const u32x4 (&x)[2], u32x4 (&o)[2]) {
    const unsigned e[8] = {x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w};
#pragma unroll
    for (int c = 0; c < 2; c++) {
        o[c].x = __builtin_amdgcn_perm(e[2 * c + 1], e[2 * c], 0x05040100u);
        o[c].y = __builtin_amdgcn_perm(e[2 * c + 1], e[2 * c], 0x07060302u);
        o[c].z = __builtin_amdgcn_perm(e[2 * c + 5], e[2 * c + 4], 0x05040100u);
        o[c].w = __builtin_amdgcn_perm(e[2 * c + 5], e[2 * c + 4], 0x07060302u);
    }
}

// qf_perm_rec's inverse: a record's operands 2 h and 2 h + 1 of qf_tile_a to its 16 weights in order.
__device__ __forceinline__ void qf_unperm_rec(const u32x4 &p, const u32x4 &q, u32x4 (&o)[2]) {
    o[0] = u32x4{__builtin_amdgcn_perm(p.y, p.x, 0x05040100u), __builtin_amdgcn_perm(p.y, p.x, 0x07060302u),
                 __builtin_amdgcn_perm(q.y, q.x, 0x05040100u), __builtin_amdgcn_perm(q.y, q.x, 0x07060302u)};
    o[1] = u32x4{__builtin_amdgcn_perm(p.w, p.z, 0x05040100u), __builtin_amdgcn_perm(p.w, p.z, 0x07060302u),
                 __builtin_amdgcn_perm(q.w, q.z, 0x05040100u), __builtin_amdgcn_perm(q.w, q.z, 0x07060302u)};
}

}  // namespace aesir
