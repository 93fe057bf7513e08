// skinny_gguf.hip -- GEMM for up to 32 activation rows over GGUF weights (native blocks of Q8_0, Q3_K,
// Q6_K, IQ4_NL, IQ3_S, IQ4_XS; Q4_K / Q5_K planes) on v_mfma_f32_32x32x16_bf16, with no barrier in
// its loop: the shape of skinny.hip with the weights decoded in registers.
//
// The M <= 64 kernel of mma.hip gives every lane one 32-element group a step. In the native
// formats the groups of a super-block share bytes (a Q3_K block's 32 bytes of high bits serve all
// eight groups, a Q6_K block's 64 bytes of low nibbles four), and each lane's load lies in a cache line
// of its own, so those steps are bound by the load instructions: Q6_K eight a group, 64 lines each.
// Here a wave's step is a unit of 256 elements of K: lane (r, h) = (lane & 31, lane >> 5) takes half h
// (four groups) of column r's unit, so shared bytes are read once a half (Q6_K 11 loads for four
// groups, Q3_K 9, Q8_0 11) a whole unit ahead of their use.
//
// A workgroup of four waves owns 32 columns; its waves take every fourth unit. The activations
// stream past in four tiles a unit (group j of both halves: RM rows of 128 bytes), straight into LDS of
// the wave's own, a unit ahead; the waits are counted vmcnt, uniform over the loop. Group j's
// weights become MFMA operands with the decoder's fp32 operations (GgufQuant.swift) and one rounding
// to bf16, as in mma.hip. The waves' sums meet in LDS in wave order; K slices as in skinny.hip.
#include "common.hpp"
#include "gguf_decode.hpp"
#include "launch.hpp"

namespace splosh {

struct SkinnyGgufArgs {
    const uint8_t *w, *plane1, *meta;  // native blocks, or the planes
    uint32_t w_bytes, p1_bytes, meta_bytes, row_bytes;
    int rows32;
    int64_t n;
    int units;  // 256-element units of K
    const uint16_t *a;
    int64_t lda;
    uint32_t a_bytes;
    void *out;
    int64_t ldc;
    const void *residual;
    int rows;
    int out_dtype;
    int nwhole, tail, slices;
    float *partial;
    int *counters;
    uint32_t partial_bytes;
};

constexpr int kSgWaves = 4, kSgCols = 32;
// The byte offset of a unit past the range: the loads at it and the few hundred bytes after read past
// the buffer (the host keeps weights under it), that is zeros.
constexpr uint32_t kSgOut = 0xFFFF0000u;

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
    __device__ void start(const SkinnyGgufArgs &args, uint32_t col, int h_) {
        h = h_;
        rs = make_rsrc(args.w, args.w_bytes);
        row = gguf_row<TYPE>(col, args.row_bytes, args.rows32);
    }
    __device__ uint32_t base(uint32_t u, bool live) const { return live ? row.base + u * row.ustride : kSgOut; }
    __device__ static void build(char *, int) {}
    __device__ void table(const char *) {}
};
// Codes 0 .. 255 of group word pair 2 i with scale s and offset o: s code + o in one rounding.
__device__ __forceinline__ bf16x8 sg_bytes(const uint32_t (&wd)[8], int i, float s, float o) {
    u32x4 d;
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 2; ++e)
            d[2 * q + e] = f32x2_to_bf16x2(__builtin_fmaf(cvt_byte(wd[2 * i + q], 2 * e), s, o),
                                           __builtin_fmaf(cvt_byte(wd[2 * i + q], 2 * e + 1), s, o));
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
    __device__ void start(const SkinnyGgufArgs &a, uint32_t col, int h_) { HalfNative::start<8>(a, col, h_); }
    __device__ void load(uint32_t u, bool live) { raw = fetch_span<34>(rs, base(u, live) + 136u * (uint32_t)h); }
    __device__ void take() { align_span(raw, x); }
    __device__ void group(int j) {  // the block starts at byte 34 j
        s0 = half_bits_to_f32(j & 1 ? x[34 * j / 4] >> 16 : x[34 * j / 4]);
#pragma unroll
        for (int q = 0; q < 8; ++q) wd[q] = (j & 1 ? x[(34 * j + 2) / 4 + q] : mid(x, 34 * j / 4 + q)) ^ 0x80808080u;
    }
    // d c as d (c + 128) - 128 d: the product's one rounding (128 d is exact).
    __device__ bf16x8 operand(int i) const { return sg_bytes(wd, i, s0, -128.0f * s0); }
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
    __device__ void start(const SkinnyGgufArgs &a, uint32_t col, int h_) { HalfNative::start<14>(a, col, h_); }
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
    // ds (c - 32) as one fma (-32 ds is exact).
    __device__ bf16x8 operand(int i) const {
        const float s = i < 2 ? s0 : s1;
        return sg_bytes(wd, i, s, -32.0f * s);
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
    __device__ void start(const SkinnyGgufArgs &a, uint32_t col, int h_) { HalfNative::start<11>(a, col, h_); }
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
        return sg_bytes(wd, i, s, -4.0f * s);
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
    __device__ void start(const SkinnyGgufArgs &a, uint32_t col, int h_) { HalfNative::start<20>(a, col, h_); }
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
    __device__ void start(const SkinnyGgufArgs &a, uint32_t col, int h_) { HalfNative::start<23>(a, col, h_); }
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
    __device__ static void build(char *t, int tid) {
        for (int e = tid; e < 512; e += kSgWaves * 64) {
            const uint32_t packed = kIq3sPacked[e];
            uint32_t m = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) m |= (2u * ((packed >> (3 * q)) & 7u) + 1u) << (8 * q);
            ((uint32_t *)t)[e] = m;
        }
    }
    __device__ void table(const char *t) { tbl = (const uint32_t *)t; }
    __device__ void start(const SkinnyGgufArgs &a, uint32_t col, int h_) { HalfNative::start<21>(a, col, h_); }
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
    __device__ static void build(char *t, int tid) {
        if constexpr (FIFTH) {
            const uint32_t v = (uint32_t)tid;  // 256 threads
            ((u32x2 *)t)[tid] = u32x2{((v & 0x33u) * 0x880110u) & 0x10101010u, (((v >> 2) & 0x33u) * 0x880110u) & 0x10101010u};
        }
    }
    __device__ void table(const char *t) { tbl = (const u32x2 *)t; }
    __device__ void start(const SkinnyGgufArgs &args, uint32_t col, int h_) {
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

// RM: activation rows staged (8, 16 or 32; rows past the last read zeros); E: accumulator values a lane
// keeps at the end (as skinny.hip).
template <int TYPE, int RM>
struct SgShape {
    static constexpr int kE = RM / 2;
    static constexpr int kThreads = kSgWaves * 64;
    static constexpr int kTile = RM * 128;
    static constexpr size_t kRing = (size_t)kSgWaves * 4 * kTile;
    static constexpr size_t kRed = (size_t)kSgWaves * kE * 64 * 4;
    static constexpr size_t kTblAt = kRing > kRed ? kRing : kRed;
    static constexpr size_t kLds = kTblAt + Half<TYPE>::kTbl;
    static constexpr int kVals = (kE + kSgWaves - 1) / kSgWaves;
    static constexpr int kActive = kE * 64 < kThreads ? kE * 64 : kThreads;
};

template <int TYPE, int RM>
__global__ void __launch_bounds__(kSgWaves * 64, 2)
gguf_skinny_kernel(SkinnyGgufArgs args) {
    using S = SgShape<TYPE, RM>;
    constexpr int E = S::kE, NA = RM / 8, NW = Half<TYPE>::kLoads;
    extern __shared__ __align__(16) char lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, h = lane >> 5;
    int blk, ua, ub, tb, sl;
    balance_block(blockIdx.x, gridDim.x, args.nwhole, args.tail, args.slices, args.units, blk, ua, ub, tb, sl);
    const int64_t n0 = (int64_t)blk * kSgCols;
    Half<TYPE> wt;
    if constexpr (Half<TYPE>::kTbl > 0) {
        Half<TYPE>::build(lds + S::kTblAt, tid);
        __syncthreads();
        wt.table(lds + S::kTblAt);
    }
    wt.start(args, (uint32_t)(n0 + r < args.n ? n0 + r : args.n - 1), h);
    const rsrc_t a_rsrc = make_rsrc(args.a, args.a_bytes);
    // Tile j of a unit: row m's 16-byte piece p (p < 4: elements 32 j + 8 p of half 0; else 32 j + 8 (p - 4)
    // of half 1) at slot p ^ (m % 8); load q brings rows 8 q .. + 7. Out-of-range offsets as skinny.hip.
    constexpr uint32_t kRowOut = 0x40000000u, kUnitOut = 0x80000000u;
    uint32_t src[NA];
#pragma unroll
    for (int q = 0; q < NA; ++q) {
        const int m = 8 * q + (lane >> 3), p = (lane & 7) ^ (lane >> 3);
        src[q] = m < args.rows ? (uint32_t)((m * args.lda + (p >> 2) * 128 + 8 * (p & 3)) * 2) : kRowOut;
    }
    char *ring = lds + wave * 4 * S::kTile;
    const int steps = (ub - ua + kSgWaves - 1) / kSgWaves;
    auto unit_of = [&](int t) { return ua + t * kSgWaves + wave; };
    auto load_a = [&](int t, int j) {
        const int u = unit_of(t);
        const uint32_t off = u < ub ? (uint32_t)u * 512u + 64u * j : kUnitOut;
#pragma unroll
        for (int q = 0; q < NA; ++q) buffer_load_lds16(a_rsrc, ring + j * S::kTile + q * 1024, src[q] + off);
    };
    auto load_w = [&](int t) {
        asm volatile("; splosh-unit-loads %0" ::"n"(NW));
        wt.load((uint32_t)unit_of(t), unit_of(t) < ub);
    };

    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
    load_w(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        load_a(0, j);
        __builtin_amdgcn_sched_barrier(0);
    }
    const uint32_t arow = (uint32_t)(r & (RM - 1)) * 128u;
    // Unit t: its raw bytes are aligned and the next unit's loads issued; then tile j is multiplied
    // once it has landed (younger: three tiles and the next unit's weights) and its slot refilled with
    // the next unit's tile j.
    for (int t = 0; t < steps; ++t) {
        wt.take();
        __builtin_amdgcn_sched_barrier(0);
        load_w(t + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            wait_vmcnt<3 * NA + NW>();
            asm volatile("" ::: "memory");
            wt.group(j);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int p = 4 * h + Half<TYPE>::piece(i);
                const bf16x8 x = as_bf16x8(*(const u32x4 *)(ring + j * S::kTile + arow + ((p ^ (r & 7)) << 4)));
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, wt.operand(i), acc, 0, 0, 0);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the tile is read before its refill
            load_a(t + 1, j);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    wait_vmcnt<0>();
    __syncthreads();  // every load into LDS has landed: the sums take its place
    float *red = (float *)lds;
#pragma unroll
    for (int e = 0; e < E; ++e) red[(wave * E + e) * 64 + lane] = acc[e];
    __syncthreads();
    constexpr int V = S::kVals;
    float v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int o = tid + j * S::kThreads;
        float x = 0.0f;
        if (o < E * 64) {
#pragma unroll
            for (int s = 0; s < kSgWaves; ++s) x += red[s * E * 64 + o];
        }
        v[j] = x;
    }
    if (tb >= 0 && !balance_merge<V>(v, tid, S::kActive, tb, sl, args.slices, args.partial, args.partial_bytes,
                                     args.counters))
        return;  // a slice whose block another slice finishes
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int o = tid + j * S::kThreads;
        const int e = o >> 6, l = o & 63;
        const int m = 8 * (e >> 2) + 4 * (l >> 5) + (e & 3);
        const int64_t n = n0 + (l & 31);
        if (o >= E * 64 || m >= args.rows || n >= args.n) continue;
        const int64_t index = m * args.ldc + n;
        float value = v[j];
        if (args.out_dtype == SPLOSH_F32) {
            if (args.residual) value += ((const float *)args.residual)[index];
            ((float *)args.out)[index] = value;
        } else {
            if (args.residual) value += bf16_bits_to_f32(((const uint16_t *)args.residual)[index]);
            ((uint16_t *)args.out)[index] = f32_to_bf16(value);
        }
    }
}

// K slices of the blocks of 32 columns: the last round of many blocks (plan_balance); one workgroup a
// CU for at most half a block a CU (K5120 -> N1024 9.8 -> 8.9 us); two a CU for fewer blocks than CUs
// and long K (K17408 -> N5120, Q6_K 27.6 -> 25.8 us, Q8_0 30.8 -> 27.5; the merge costs about 3 us, which
// K5120 -> N5120 does not win back: 11.1 -> 15).
constexpr int kSgLong = 32;  // units of K
static BalanceSplit plan_sg(int64_t blocks, int units) {
    const int cus = device_cus();
    BalanceSplit p = plan_balance(blocks, cus, units);
    int s = 1;
    if (2 * blocks <= cus) s = (int)(cus / blocks) * (units >= kSgLong ? 2 : 1);
    else if (blocks < cus && units >= kSgLong) s = (int)(2 * cus / blocks);
    s = s < kBalanceMaxSlices ? s : kBalanceMaxSlices;
    while (s >= 2 && (units < 2 * s * kSgWaves || blocks * s % 8 != 0)) --s;
    if (s >= 2) p = BalanceSplit{0, (int)blocks, s};
    return p;
}
static int sg_rows(int64_t rows) { return rows <= 8 ? 8 : rows <= 16 ? 16 : 32; }
static size_t sg_need(const BalanceSplit &p, int64_t rows) {
    if (p.slices < 2) return 0;
    const int e = sg_rows(rows) / 2, vals = (e + kSgWaves - 1) / kSgWaves;
    const int active = e * 64 < kSgWaves * 64 ? e * 64 : kSgWaves * 64;
    return kBalanceCounterBytes + (size_t)p.tail * p.slices * vals * active * sizeof(float);
}

// Shapes the kernel takes: whole units of K, 32-bit offsets, activations under 1 GiB.
static bool sg_shape(int64_t rows, int64_t columns, int64_t inner, int64_t lda) {
    return rows >= 1 && rows <= 32 && columns > 0 && inner >= 256 && inner % 256 == 0 &&
           (rows * lda + inner) * 2 < ((int64_t)1 << 30);
}

// And the calls it is the fastest for (us, K17408 -> N5120, file order, this kernel against the kernel
// before it): 5 to 16 rows of every type (8 rows: Q8_0 30.3 / 33.1, Q6_K 27.9 / 43.0, Q3_K 21.6 /
// 46.1, IQ3_S 26.2 / 42.4, IQ4_NL 23.3 / 27.2, IQ4_XS 23.0 / 30.0, Q4_K 18.7 / 21.8, Q5_K 21.4 /
// 23.8); two to four rows, and one of Q3_K (20.5 / 22.0), from about the size of K5120 -> N3328 (8.9
// against 8.3 on the streaming kernel at N1024, 11.4 against 14.2 at N5120); 17 to 32 rows, where
// the activations' traffic grows, of the types whose loads weigh most in mma.hip (32 rows: Q6_K 39.2 /
// 43.2, Q3_K 31.8 / 46.3, IQ3_S 35.4 / 42.8, IQ4_XS in the file's order 32.3 / 34.1; not Q8_0 41.0 / 38.6).
bool gguf_skinny_fits(int type, int64_t rows, int64_t columns, int64_t inner, int64_t lda, int64_t weight_bytes) {
    if (!sg_shape(rows, columns, inner, lda) || weight_bytes >= (int64_t)kSgOut - 65536) return false;
    const bool rows32 = gguf_layout(type);
    if (rows <= 4)
        return (rows > 1 || type == 11) && (columns + kSgCols - 1) / kSgCols * (inner / 256) >= 2048;
    return rows <= 16 || type == 14 || type == 11 || type == 21 || (type == 23 && !rows32);
}

size_t gguf_skinny_workspace_bytes(int64_t rows, int64_t columns, int64_t inner) {
    if (!sg_shape(rows, columns, inner, inner)) return 0;
    return sg_need(plan_sg((columns + kSgCols - 1) / kSgCols, (int)(inner / 256)), rows);
}

template <int TYPE, int RM>
static hipError_t launch_sg_v(const SkinnyGgufArgs &args, int64_t blocks, hipStream_t stream) {
    using S = SgShape<TYPE, RM>;
    auto kernel = gguf_skinny_kernel<TYPE, RM>;
    if constexpr (S::kLds > 64 * 1024) {
        static const bool once = [&] {
            (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
            return true;
        }();
        (void)once;
    }
    const int64_t grid = args.slices > 1 ? args.nwhole + (int64_t)args.tail * args.slices : blocks;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kSgWaves * 64), S::kLds, stream, args);
    return hipGetLastError();
}
template <int TYPE>
static hipError_t launch_sg(const SkinnyGgufArgs &args, int64_t blocks, hipStream_t stream) {
    switch (sg_rows(args.rows)) {
        case 8: return launch_sg_v<TYPE, 8>(args, blocks, stream);
        case 16: return launch_sg_v<TYPE, 16>(args, blocks, stream);
        default: return launch_sg_v<TYPE, 32>(args, blocks, stream);
    }
}

hipError_t launch_gguf_skinny(int type, const uint8_t *w, const uint8_t *plane1, const uint8_t *meta, int64_t columns,
                              int64_t inner, const uint16_t *a, int64_t lda, void *out, int64_t ldc, int out_dtype,
                              const void *residual, int64_t rows, void *workspace, size_t workspace_bytes,
                              hipStream_t stream) {
    SkinnyGgufArgs args = {};
    args.rows32 = gguf_layout(type);
    args.w = w;
    args.plane1 = plane1;
    args.meta = meta;
    args.n = columns;
    args.units = (int)(inner / 256);
    if (meta) {
        args.w_bytes = (uint32_t)(columns * args.units * 8 * 16);
        args.p1_bytes = (uint32_t)(columns * args.units * 8 * 4);
        args.meta_bytes = (uint32_t)(columns * args.units * 16);
    } else {
        int elems = 0, bytes = 0;
        gguf_native_block(type, &elems, &bytes);
        args.row_bytes = (uint32_t)(inner / elems * bytes);
        args.w_bytes = (uint32_t)((args.rows32 ? (columns + 31) / 32 * 32 : columns) * args.row_bytes);
    }
    args.a = a;
    args.lda = lda;
    args.a_bytes = (uint32_t)(((rows - 1) * lda + inner) * 2);
    args.out = out;
    args.ldc = ldc;
    args.residual = residual;
    args.rows = (int)rows;
    args.out_dtype = out_dtype;
    const int64_t blocks = (columns + kSgCols - 1) / kSgCols;
    const BalanceSplit p = plan_sg(blocks, args.units);
    const size_t need = sg_need(p, rows);
    args.slices = 1;
    if (need > 0 && workspace && workspace_bytes >= need) {
        args.nwhole = p.nwhole;
        args.tail = p.tail;
        args.slices = p.slices;
        args.counters = (int *)workspace;
        args.partial = (float *)((char *)workspace + kBalanceCounterBytes);
        args.partial_bytes = (uint32_t)(need - kBalanceCounterBytes);
    }
    switch (type) {
        case 8: return launch_sg<8>(args, blocks, stream);
        case 11: return launch_sg<11>(args, blocks, stream);
        case 12: return launch_sg<12>(args, blocks, stream);
        case 13: return launch_sg<13>(args, blocks, stream);
        case 14: return launch_sg<14>(args, blocks, stream);
        case 20: return launch_sg<20>(args, blocks, stream);
        case 21: return launch_sg<21>(args, blocks, stream);
        default: return launch_sg<23>(args, blocks, stream);
    }
}

}  // namespace splosh
