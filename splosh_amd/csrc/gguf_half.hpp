// gguf_half.hpp -- half a 256-element unit of one column of a GGUF weight, held and decoded by one lane
// (skinny_gguf.hip, and the native formats in prefill.hip).
#pragma once
#include "common.hpp"
#include "gguf_decode.hpp"

namespace splosh {

// The byte offset of a unit past the range: the loads at it and the few hundred bytes after read past
// the buffer (the host keeps weights under it), that is zeros.
constexpr uint32_t kSgOut = 0xFFFF0000u;

// A weight as the halves read it: native blocks, or the planes.
struct GgufSource {
    const uint8_t *w, *plane1, *meta;
    uint32_t w_bytes, p1_bytes, meta_bytes, row_bytes;
    int rows32;
    int units;  // 256-element units of K
};

// Half a unit of one column: raw bytes as loaded (load), the same aligned (take), group j's scales
// and code words (group), and elements 8 piece(i) .. + 7 of the group as bf16 (operand). kLoads: the
// vector loads load() issues once the compiler has merged what it can (the loop's waits count them; a
// test checks them against the assembly).
struct HalfNative {
    static constexpr int kTbl = 0;
    static constexpr int piece(int i) { return i; }
    rsrc_t rs;
    GgufRow row;
    int h;
    float s0, s1;
    uint32_t wd[8];
    template <int TYPE>
    __device__ void start(const GgufSource &args, uint32_t col, int h_) {
        h = h_;
        rs = make_rsrc(args.w, args.w_bytes);
        row = gguf_row<TYPE>(col, args.row_bytes, args.rows32);
    }
    __device__ uint32_t base(uint32_t u, bool live) const { return live ? row.base + u * row.ustride : kSgOut; }
    __device__ static void build(char *, int, int) {}
    __device__ void table(const char *) {}
};
// Codes 0 .. 255 of group word pair 2 i: s (code - zero), the difference exact, in one rounding (and with
// the decoder's infinities and NaN, which an fma with an offset of -zero s would not keep).
__device__ __forceinline__ bf16x8 sg_bytes(const uint32_t (&wd)[8], int i, float s, float zero) {
    u32x4 d;
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 2; ++e)
            d[2 * q + e] = f32x2_to_bf16x2(s * (cvt_byte(wd[2 * i + q], 2 * e) - zero),
                                           s * (cvt_byte(wd[2 * i + q], 2 * e + 1) - zero));
    return as_bf16x8(d);
}
// Dword k of bytes that start 2 bytes into a.
template <int W>
__device__ __forceinline__ uint32_t mid(const uint32_t (&a)[W], int k) {
    return __builtin_amdgcn_alignbyte(a[k + 1], a[k], 2);
}

template <int TYPE>
struct Half;

template <>
struct Half<8> : HalfNative {  // Q8_0: four blocks of fp16 d and 32 int8 codes (GgufQuant.swift:172-175)
    static constexpr int kLoads = 10;
    Span<34> raw;
    uint32_t x[34];
    __device__ void start(const GgufSource &a, uint32_t col, int h_) { HalfNative::start<8>(a, col, h_); }
    __device__ void load(uint32_t u, bool live) { raw = fetch_span<34>(rs, base(u, live) + 136u * (uint32_t)h); }
    __device__ void take() { align_span(raw, x); }
    __device__ void group(int j) {  // the block starts at byte 34 j
        s0 = half_bits_to_f32(j & 1 ? x[34 * j / 4] >> 16 : x[34 * j / 4]);
#pragma unroll
        for (int q = 0; q < 8; ++q) wd[q] = (j & 1 ? x[(34 * j + 2) / 4 + q] : mid(x, 34 * j / 4 + q)) ^ 0x80808080u;
    }
    __device__ bf16x8 operand(int i) const { return sg_bytes(wd, i, s0, 128.0f); }
};

template <>
struct Half<14> : HalfNative {  // Q6_K: ql[128], qh[64], scales[16], d (:218-230)
    static constexpr int kLoads = 11;
    Span<16> ql;
    Span<8> qh;
    Span<4> sc;
    uint32_t d;
    uint32_t xl[16], xh[8], xs[2];
    float df;
    __device__ void start(const GgufSource &a, uint32_t col, int h_) { HalfNative::start<14>(a, col, h_); }
    __device__ void load(uint32_t u, bool live) {
        const uint32_t b = base(u, live);
        ql = fetch_span<16>(rs, b + 64u * (uint32_t)h);
        qh = fetch_span<8>(rs, b + 128u + 32u * (uint32_t)h);
        sc = fetch_span<4>(rs, b + 192u);
        d = ld16(rs, b + 208u);
    }
    __device__ void take() {
        align_span(ql, xl);
        align_span(qh, xh);
        uint32_t s[4];
        align_span(sc, s);
        xs[0] = h ? s[2] : s[0];
        xs[1] = h ? s[3] : s[1];
        df = half_bits_to_f32(d);
    }
    __device__ void group(int j) {
        const uint32_t s = xs[j >> 1] >> (16 * (j & 1));
        s0 = df * (float)(int8_t)(s & 0xFF);
        s1 = df * (float)(int8_t)((s >> 8) & 0xFF);
#pragma unroll
        for (int q = 0; q < 8; ++q)
            wd[q] = ((xl[8 * (j & 1) + q] >> (4 * (j >> 1))) & 0x0F0F0F0Fu) | (((xh[q] >> (2 * j)) & 0x03030303u) << 4);
    }
    __device__ bf16x8 operand(int i) const {
        const float s = i < 2 ? s0 : s1;
        return sg_bytes(wd, i, s, 32.0f);
    }
};

template <>
struct Half<11> : HalfNative {  // Q3_K: hmask[32], qs[64], scales[12], d (:238-256)
    static constexpr int kLoads = 9;
    Span<8> hm, qs;
    Span<3> sc;
    uint32_t d;
    uint32_t xh[8], xq[8], xs[3];
    float df;
    __device__ void start(const GgufSource &a, uint32_t col, int h_) { HalfNative::start<11>(a, col, h_); }
    __device__ void load(uint32_t u, bool live) {
        const uint32_t b = base(u, live);
        hm = fetch_span<8>(rs, b);
        qs = fetch_span<8>(rs, b + 32u + 32u * (uint32_t)h);
        sc = fetch_span<3>(rs, b + 96u);
        d = ld16(rs, b + 108u);
    }
    __device__ void take() {
        align_span(hm, xh);
        align_span(qs, xq);
        align_span(sc, xs);
#pragma unroll
        for (int q = 0; q < 8; ++q) xh[q] >>= 4 * h;  // bit j: group 4 h + j's high bits
        df = half_bits_to_f32(d);
    }
    __device__ void group(int j) {
        // Scales 8 h + 2 j, + 1: nibble h of bytes 2 j, 2 j + 1, and bits 2 (2 h + j / 2) of bytes
        // 8 + 2 (j % 2), + 1.
        const uint32_t lo = xs[j >> 1] >> (16 * (j & 1) + 4 * h), hi = xs[2] >> (16 * (j & 1) + 4 * h + 2 * (j >> 1));
        s0 = df * ((float)((lo & 15) | ((hi & 3) << 4)) - 32.0f);
        s1 = df * ((float)(((lo >> 8) & 15) | (((hi >> 8) & 3) << 4)) - 32.0f);
#pragma unroll
        for (int q = 0; q < 8; ++q)
            wd[q] = ((xq[q] >> (2 * j)) & 0x03030303u) | (((xh[q] >> j) & 0x01010101u) << 2);
    }
    __device__ bf16x8 operand(int i) const {
        const float s = i < 2 ? s0 : s1;
        return sg_bytes(wd, i, s, 4.0f);
    }
};

// IQ4 operand (IQ4_NL, IQ4_XS): element e < 16 of the group is the low nibble of byte e, element e >= 16
// the high nibble of byte e - 16, looked up in the value table.
__device__ __forceinline__ bf16x8 sg_iq4(const uint32_t (&wd)[8], int i, float s) {
    u32x4 d;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const uint32_t x = wd[2 * (i & 1) + q];
        const uint32_t v = iq4_lookup4(i >> 1 ? (x >> 4) & 0x0F0F0F0Fu : x & 0x0F0F0F0Fu);
#pragma unroll
        for (int e = 0; e < 2; ++e)
            d[2 * q + e] = f32x2_to_bf16x2(s * (float)(int8_t)((v >> (16 * e)) & 0xFF),
                                           s * (float)(int8_t)((v >> (16 * e + 8)) & 0xFF));
    }
    return as_bf16x8(d);
}

template <>
struct Half<20> : HalfNative {  // IQ4_NL: four blocks of fp16 d and 16 bytes of codes (:179-185)
    static constexpr int kLoads = 6;
    Span<18> raw;
    uint32_t x[18];
    __device__ void start(const GgufSource &a, uint32_t col, int h_) { HalfNative::start<20>(a, col, h_); }
    __device__ void load(uint32_t u, bool live) { raw = fetch_span<18>(rs, base(u, live) + 72u * (uint32_t)h); }
    __device__ void take() { align_span(raw, x); }
    __device__ void group(int j) {  // the block starts at byte 18 j
        s0 = half_bits_to_f32(j & 1 ? x[18 * j / 4] >> 16 : x[18 * j / 4]);
#pragma unroll
        for (int q = 0; q < 4; ++q) wd[q] = j & 1 ? x[(18 * j + 2) / 4 + q] : mid(x, 18 * j / 4 + q);
    }
    __device__ bf16x8 operand(int i) const { return sg_iq4(wd, i, s0); }
};

template <>
struct Half<23> : HalfNative {  // IQ4_XS: d, scales_h, scales_l[4], qs[128] (:261-275)
    static constexpr int kLoads = 5;
    u32x4 head, raw[4], x[4];
    uint32_t sl, sh;
    float df;
    __device__ void start(const GgufSource &a, uint32_t col, int h_) { HalfNative::start<23>(a, col, h_); }
    __device__ void load(uint32_t u, bool live) {
        const uint32_t b = base(u, live);
        head = buffer_load16(rs, b, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) raw[j] = buffer_load16(rs, b + 8u + 64u * (uint32_t)h + 16u * j, 0);
    }
    __device__ void take() {
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = raw[j];
        df = half_bits_to_f32(head[0]);
        sh = head[0] >> (16 + 8 * h);
        sl = head[1] >> (16 * h);
    }
    __device__ void group(int j) {
        s0 = df * ((float)(((sl >> (4 * j)) & 15) | (((sh >> (2 * j)) & 3) << 4)) - 32.0f);
#pragma unroll
        for (int q = 0; q < 4; ++q) wd[q] = x[j][q];
    }
    __device__ bf16x8 operand(int i) const { return sg_iq4(wd, i, s0); }
};

template <>
struct Half<21> : HalfNative {  // IQ3_S: d, qs[64], qh[8], signs[32], scales[4] (:283-300)
    static constexpr int kLoads = 9;
    static constexpr int kTbl = 512 * 4;  // the codebook's four magnitudes an entry, as bytes
    const uint32_t *tbl;
    Span<8> cb;
    Span<4> sg;
    Span<1> nb;
    uint32_t d, sc;
    uint32_t xc[8], xg[4], xn[1], xsc;
    float df;
    uint32_t sign, ninth;
    __device__ static void build(char *t, int tid, int threads) {
        for (int e = tid; e < 512; e += threads) {
            const uint32_t packed = kIq3sPacked[e];
            uint32_t m = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) m |= (2u * ((packed >> (3 * q)) & 7u) + 1u) << (8 * q);
            ((uint32_t *)t)[e] = m;
        }
    }
    __device__ void table(const char *t) { tbl = (const uint32_t *)t; }
    __device__ void start(const GgufSource &a, uint32_t col, int h_) { HalfNative::start<21>(a, col, h_); }
    __device__ void load(uint32_t u, bool live) {
        const uint32_t b = base(u, live);
        d = ld16(rs, b);
        cb = fetch_span<8>(rs, b + 2u + 32u * (uint32_t)h);
        nb = fetch_span<1>(rs, b + 66u + 4u * (uint32_t)h);
        sg = fetch_span<4>(rs, b + 74u + 16u * (uint32_t)h);
        sc = ld16(rs, b + 106u + 2u * (uint32_t)h);
    }
    __device__ void take() {
        align_span(cb, xc);
        align_span(sg, xg);
        align_span(nb, xn);
        xsc = sc;
        df = half_bits_to_f32(d);
    }
    __device__ void group(int j) {
        s0 = df * (1.0f + 2.0f * (float)((xsc >> (4 * j)) & 15));
        wd[0] = xc[2 * j];
        wd[1] = xc[2 * j + 1];
        sign = xg[j];
        ninth = (xn[0] >> (8 * j)) & 0xFF;
    }
    __device__ bf16x8 operand(int i) const {
        float v[8];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int k = 2 * i + q;
            const uint32_t m = tbl[((wd[k >> 2] >> (8 * (k & 3))) & 0xFF) | (((ninth >> k) & 1) << 8)];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t s = ((sign >> (4 * k + e)) & 1u) << 31;
                v[4 * q + e] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, s0 * cvt_byte(m, e)) ^ s);
            }
        }
        u32x4 o;
#pragma unroll
        for (int p = 0; p < 4; ++p) o[p] = f32x2_to_bf16x2(v[2 * p], v[2 * p + 1]);
        return as_bf16x8(o);
    }
};

// Q4_K (FIFTH = false) and Q5_K planes (GgufPlanes.swift:8-20, 62-74; the nibbles' chunk order and the
// fifth bits' table as Q5Format in mma.hip).
template <bool FIFTH>
struct HalfPlane {
    static constexpr int kLoads = FIFTH ? 9 : 5;
    static constexpr int kTbl = FIFTH ? 256 * 8 : 0;
    static constexpr int piece(int i) { return ((i & 1) << 1) | (i >> 1); }
    rsrc_t r0, r1, rm;
    uint32_t rec, mrec;
    int h;
    const u32x2 *tbl;
    u32x4 raw[4], m, x[4];
    uint32_t rawh[4], xh[4], scw, mnw, dw;
    float s0, s1;
    u32x4 w;
    uint32_t wh, lo[2], hi[2];
    __device__ static void build(char *t, int tid, int threads) {
        if constexpr (FIFTH)
            for (uint32_t v = (uint32_t)tid; v < 256; v += (uint32_t)threads)
                ((u32x2 *)t)[v] = u32x2{((v & 0x33u) * 0x880110u) & 0x10101010u, (((v >> 2) & 0x33u) * 0x880110u) & 0x10101010u};
    }
    __device__ void table(const char *t) { tbl = (const u32x2 *)t; }
    __device__ void start(const GgufSource &args, uint32_t col, int h_) {
        h = h_;
        r0 = make_rsrc(args.w, args.w_bytes);
        r1 = make_rsrc(FIFTH ? (const void *)args.plane1 : (const void *)args.w, FIFTH ? args.p1_bytes : 0u);
        rm = make_rsrc(args.meta, args.meta_bytes);
        rec = ((col >> 7) * (uint32_t)args.units * 8u + 4u * (uint32_t)h) * 128u + (col & 127u);
        mrec = (col >> 7) * (uint32_t)args.units * 128u + (col & 127u);
    }
    __device__ void load(uint32_t u, bool live) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t at = rec + (8u * u + j) * 128u;
            raw[j] = buffer_load16_cp<2>(r0, live ? at * 16u : kSgOut, 0);
            if constexpr (FIFTH) rawh[j] = buffer_load_u32(r1, live ? at * 4u : kSgOut, 0);
        }
        m = buffer_load16(rm, live ? (mrec + u * 128u) * 16u : kSgOut, 0);
    }
    __device__ void take() {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x[j] = raw[j];
            if constexpr (FIFTH) xh[j] = rawh[j];
        }
        // The half's four scales and minimums (GgufQuant.swift:196-203), a byte each.
        scw = h ? (m[3] & 0x0F0F0F0Fu) | ((m[1] >> 2) & 0x30303030u) : m[1] & 0x3F3F3F3Fu;
        mnw = h ? ((m[3] >> 4) & 0x0F0F0F0Fu) | ((m[2] >> 2) & 0x30303030u) : m[2] & 0x3F3F3F3Fu;
        dw = m[0];
    }
    __device__ void group(int j) {
        s0 = half_bits_to_f32(dw) * cvt_byte(scw, j);
        s1 = -(half_bits_to_f32(dw >> 16) * cvt_byte(mnw, j));
        w = x[j];
        if constexpr (FIFTH) wh = xh[j];
    }
    __device__ bf16x8 operand(int i) {
        if ((i & 1) == 0) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                lo[e] = w[i + e] & 0x0F0F0F0Fu;
                hi[e] = (w[i + e] >> 4) & 0x0F0F0F0Fu;
                if constexpr (FIFTH) {
                    const u32x2 f = tbl[__builtin_amdgcn_ubfe(wh, 8 * (i + e), 8)];
                    lo[e] |= f[0];
                    hi[e] |= f[1];
                }
            }
        }
        const int b = i & 1;
        u32x4 d;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            d[2 * e] = f32x2_to_bf16x2(__builtin_fmaf(cvt_byte(lo[e], b), s0, s1), __builtin_fmaf(cvt_byte(lo[e], b + 2), s0, s1));
            d[2 * e + 1] = f32x2_to_bf16x2(__builtin_fmaf(cvt_byte(hi[e], b), s0, s1), __builtin_fmaf(cvt_byte(hi[e], b + 2), s0, s1));
        }
        return as_bf16x8(d);
    }
};
template <>
struct Half<12> : HalfPlane<false> {};
template <>
struct Half<13> : HalfPlane<true> {};

}  // namespace splosh
