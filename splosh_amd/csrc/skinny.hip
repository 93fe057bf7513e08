// skinny.hip -- q4 GEMM for a few activation rows (3 to 32; a grouped call from one) over tiled weights on
// v_mfma_f32_32x32x16_bf16, with no barrier in its loop.
//
// At these row counts a call reads its weight once and is bound by HBM and by fixed latencies
// (the stream-K kernel of mma.hip streams as fast, but spends 8 to 13 us a call on its set-up,
// pipeline fill, K-wave reduction and fix-up). So this kernel has the decode kernel's shape: a
// workgroup of KW waves owns 32 output columns of each of NW weights (NW = 2: fused gate+up), its
// waves take every KW-th 64-group of K, and several workgroups share a CU and hide each other's
// latencies.
//
//  * Lane (r, h) = (lane & 31, lane >> 5) feeds column r with the group's words 4 h .. 4 h + 3 (one
//    16-byte load; a wave reads 32 consecutive records, a contiguous kilobyte) and row r.
//  * The wave's activations of a group (RM rows of 128 bytes) go straight from memory into LDS of
//    its own, eight rows a load, and are read back as MFMA operands; codes and sidecars go to a
//    register ring. All of a group's loads are issued D groups before its arithmetic and waited
//    for with a counted vmcnt: no wave waits for another before the end.
//  * Raw codes: a code word becomes four bf16 pairs (128 + q_j, 128 + q_{j+4}) with one v_and_or_b32
//    each, and the activation pairs are permuted to match ((x_j, x_{j+4}), shared by both weights).
//    Per group, P = sum x (128 + q) and the row sums S = sum x (the same operands times ones, one
//    chain for both weights) come from the matrix cores, and acc += s P + (b - 128 s) S takes two
//    FMAs a value: the weights are exact, where rounding them to bf16 in registers takes 19
//    instructions per 8 weights (7 here). The cost of the scaling grows with the rows; at 64 the
//    two are equal. P and S cancel to a thirtieth, which left the fp32 sums of three and four rows further
//    from 64 bits than the decode kernel's: calls of up to eight rows, but for grouped ones, use 16 + q, a shift
//    more a word (1 to 3% of the time).
//  * At the end the waves' sums meet in LDS in wave order. Where the blocks do not fill the CUs
//    evenly, or are few, K is cut into slices merged by the last to arrive in slice order
//    (balance_merge, common.hpp).
#include "common.hpp"
#include "launch.hpp"
#include "mix.hpp"

namespace splosh {

constexpr int kSkinnyCols = 32;  // output columns a workgroup
constexpr int kSkinnyMaxGroup = SPLOSH_MAX_GROUP;

struct SkinnyArgs {
    const uint32_t *packed[2];
    const uint16_t *scales[2], *biases[2];
    int groups;
    const uint16_t *a;
    int64_t lda;
    void *out;
    int64_t ldc;
    const void *residual;
    int rows;
    int64_t half;  // a split weight's columns a half
    int out_dtype;
    uint32_t code_bytes, sidecar_bytes, a_bytes;
    // K slices (slices > 1): blocks [0, nwhole) whole, nwhole + [0, tail) in `slices` slices each.
    int nwhole, tail, slices;
    float *partial;
    int *counters;
    uint32_t partial_bytes;
    // A grouped call: weight i owns blocks [gblk[i], gblk[i + 1]) and writes its own output.
    int ngroup;
    int gblk[kSkinnyMaxGroup + 1];
    const uint32_t *gpacked[kSkinnyMaxGroup];
    const uint16_t *gscales[kSkinnyMaxGroup], *gbiases[kSkinnyMaxGroup];
    void *gout[kSkinnyMaxGroup];
    int64_t gldc[kSkinnyMaxGroup];
};

// (a & mask) | c, one v_and_or_b32 with the mask in an SGPR and c in a VGPR. Not inline asm: what it
// returns feeds an MFMA, and the compiler leaves the wait states that a VALU write needs before an
// MFMA reads it only after instructions it knows.
__device__ __forceinline__ uint32_t sk_and_or(uint32_t a, uint32_t mask, uint32_t c) { return (a & mask) | c; }

// RM: activation rows staged (8, 16 or 32; rows past the last read zeros). E: accumulator values a
// lane keeps of the MFMA's 16 (row 8 (e / 4) + 4 h + e % 4: the first RM / 2 cover RM rows).
template <int RM, int KW, int D>
struct SkinnyShape {
    static constexpr int kE = RM / 2;
    static constexpr int kThreads = KW * 64;
    static constexpr int kTile = RM * 128;  // a group's activations of a wave
    static constexpr size_t ring() { return (size_t)KW * D * kTile; }
    static constexpr size_t lds(int nw) {
        const size_t red = (size_t)KW * nw * kE * 64 * 4;
        return ring() > red ? ring() : red;
    }
    static constexpr int kVals = (kE + KW - 1) / KW;                      // outputs a thread and weight
    static constexpr int kActive = kE * 64 < kThreads ? kE * 64 : kThreads;  // threads with outputs
};

// What a workgroup's NW weights are: one weight; one weight of a grouped call; the two column
// halves of one weight (each stored to its own columns); gate and up.
enum SkinnyMode { kSkinnyOne, kSkinnyGroup, kSkinnySplit, kSkinnyMlp };
constexpr int skinny_nw(SkinnyMode mode) { return mode >= kSkinnySplit ? 2 : 1; }

// (Registers: two workgroups of eight waves a CU up to 16 rows, which the K slices of a long K count on; K17408
// -> N5120 at 12 to 16 rows 22.9 us with one, 18.4 with two.)
template <SkinnyMode MODE, int RM, int KW, int D>
__global__ void __launch_bounds__(KW * 64, skinny_nw(MODE) == 2 && RM == 32 ? 3 : 4)
q4_skinny_kernel(SkinnyArgs args) {
    constexpr int NW = skinny_nw(MODE);
    using S = SkinnyShape<RM, KW, D>;
    constexpr int E = S::kE, NA = RM / 8;
    constexpr bool kNear = RM == 8 && MODE != kSkinnyGroup;  // codes as 16 + q, else 128 + q
    constexpr float kOffset = kNear ? 16.0f : 128.0f;
    constexpr int kLoads = 3 * NW + NA;  // loads a wave and group
    static_assert((D - 1) * kLoads <= 63, "vmcnt holds 6 bits");
    extern __shared__ __align__(16) char lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, h = lane >> 5;
    const int G = args.groups;
    int blk, ga, gb, tb, sl;
    balance_block(blockIdx.x, gridDim.x, args.nwhole, args.tail, args.slices, G, blk, ga, gb, tb, sl);
    void *out = args.out;
    int64_t ldc = args.ldc;
    rsrc_t q_rsrc[NW], s_rsrc[NW], b_rsrc[NW];
    if constexpr (MODE == kSkinnyGroup) {
        int gi = 0;
        for (int i = 1; i < args.ngroup; ++i) gi = blk >= args.gblk[i] ? i : gi;
        const uint32_t recs = (uint32_t)(args.gblk[gi + 1] - args.gblk[gi]) * kSkinnyCols * (uint32_t)G;
        blk -= args.gblk[gi];
        q_rsrc[0] = make_rsrc(args.gpacked[gi], recs * 32u);
        s_rsrc[0] = make_rsrc(args.gscales[gi], recs * 2u);
        b_rsrc[0] = make_rsrc(args.gbiases[gi], recs * 2u);
        out = args.gout[gi];
        ldc = args.gldc[gi];
    } else {
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            q_rsrc[w] = make_rsrc(args.packed[w], args.code_bytes);
            s_rsrc[w] = make_rsrc(args.scales[w], args.sidecar_bytes);
            b_rsrc[w] = make_rsrc(args.biases[w], args.sidecar_bytes);
        }
    }
    const rsrc_t a_rsrc = make_rsrc(args.a, args.a_bytes);
    const uint32_t n0 = (uint32_t)blk * kSkinnyCols;
    const uint32_t rec0 = (n0 >> 7) * (uint32_t)G * 128u + (n0 & 127u) + (uint32_t)r;
    // Activation load j: lane l brings row 8 j + l / 8, slot l % 8, holding the row's 16-byte piece
    // (l % 8) ^ (l / 8) (so that the operand reads of 8 consecutive rows hit eight slots). Rows past
    // the last and groups past the range read past the buffer (the host keeps it under 1 GiB, so
    // that these offsets cannot wrap): zeros, no traffic.
    constexpr uint32_t kRowOut = 0x40000000u, kGroupOut = 0x80000000u;
    uint32_t src[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) {
        const int m = 8 * j + (lane >> 3);
        src[j] = m < args.rows ? (uint32_t)((m * args.lda + 8 * ((lane & 7) ^ (lane >> 3))) * 2) : kRowOut;
    }
    char *ring = lds + wave * D * S::kTile;
    u32x4 cq[D][NW];
    uint32_t cs[D][NW], cb[D][NW];
    auto issue = [&](int slot, int t) {
        const int g = ga + t * KW + wave;
        const bool live = g < gb;
        const uint32_t agrp = live ? (uint32_t)g * 128u : kGroupOut;
        const uint32_t off = live ? (rec0 + (uint32_t)g * 128u) * 32u + 16u * h : 0xFFFFFFF0u;
        const uint32_t soff = live ? (rec0 + (uint32_t)g * 128u) * 2u : 0xFFFFFFF0u;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            cq[slot][w] = buffer_load16_cp<2>(q_rsrc[w], off, 0);
            cs[slot][w] = buffer_load_u16(s_rsrc[w], soff, 0);
            cb[slot][w] = buffer_load_u16(b_rsrc[w], soff, 0);
        }
#pragma unroll
        for (int j = 0; j < NA; ++j) buffer_load_lds16(a_rsrc, ring + slot * S::kTile + j * 1024, src[j] + agrp);
        __builtin_amdgcn_sched_barrier(0);
    };
    const int steps = (gb - ga + KW - 1) / KW;
#pragma unroll
    for (int k = 0; k < D; ++k) issue(k, k);

    const uint32_t kMask = kNear ? 0x00780078u : 0x000F000Fu;
    uint32_t magic;  // the bf16 exponent of 16 (q in bits 3 .. 6 adds q) or 128 (bits 0 .. 3) in both halves
    if constexpr (kNear) asm volatile("v_mov_b32 %0, 0x41804180" : "=v"(magic));
    else asm volatile("v_mov_b32 %0, 0x43004300" : "=v"(magic));
    const u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
    f32x16 zero;
#pragma unroll
    for (int e = 0; e < 16; ++e) zero[e] = 0.0f;
    float acc[NW][E];
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int e = 0; e < E; ++e) acc[w][e] = 0.0f;
    const uint32_t arow = (uint32_t)(r & (RM - 1)) * 128u;

    for (int t0 = 0; t0 < steps; t0 += D) {
#pragma unroll
        for (int k = 0; k < D; ++k) {
            wait_vmcnt<(D - 1) * kLoads>();  // this group has landed; the D - 1 younger may not have
            asm volatile("" ::: "memory");
            bf16x8 x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const u32x4 v = *(const u32x4 *)(ring + k * S::kTile + arow + (((4 * h + i) ^ (r & 7)) << 4));
                const u32x4 p = {perm_bytes(v.z, v.x, 0x05040100u), perm_bytes(v.z, v.x, 0x07060302u),
                                 perm_bytes(v.w, v.y, 0x05040100u), perm_bytes(v.w, v.y, 0x07060302u)};
                x[i] = as_bf16x8(p);
            }
            f32x16 sum = zero, prod[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w) prod[w] = zero;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[i], as_bf16x8(ones), sum, 0, 0, 0);
#pragma unroll
                for (int w = 0; w < NW; ++w) {
                    const uint32_t q = cq[k][w][i];
                    constexpr int kUp = kNear ? 3 : 0;
                    const u32x4 b = {sk_and_or(q << kUp, kMask, magic), sk_and_or(q >> (4 - kUp), kMask, magic),
                                     sk_and_or(q >> (8 - kUp), kMask, magic), sk_and_or(q >> (12 - kUp), kMask, magic)};
                    prod[w] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[i], as_bf16x8(b), prod[w], 0, 0, 0);
                }
                // (Keeps the second half's operands from being built early: 28 bytes a lane spilled at 8 rows.)
                if (NW == 2 && i == 1) __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const float s = bf16_bits_to_f32(cs[k][w]);
                const float bp = __builtin_fmaf(-kOffset, s, bf16_bits_to_f32(cb[k][w]));
#pragma unroll
                for (int e = 0; e < E; ++e)
                    acc[w][e] = __builtin_fmaf(s, prod[w][e], __builtin_fmaf(bp, sum[e], acc[w][e]));
            }
            // The operands are read before the refill overwrites their slot.
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue(k, t0 + k + D);
        }
    }
    wait_vmcnt<0>();
    float probe = 0.0f;  // NaN if a sum of this lane is infinite or NaN
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int e = 0; e < E; ++e) probe = __builtin_fmaf(acc[w][e], 0.0f, probe);
    __syncthreads();  // every load into LDS has landed: the sums take its place
    float *red = (float *)lds;
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int e = 0; e < E; ++e) red[((wave * NW + w) * E + e) * 64 + lane] = acc[w][e];
    // An infinite activation or scale leaves inf - inf in s P + (b - 128 s) S, and one above 2^120 can overflow
    // it where x w does not: a wave with such a sum goes over its groups again with the dequantized weights (as
    // mma.hip) and takes the new sums in the place of those. No finite sum changes. (Here, with the sums in LDS,
    // it costs a call without such values less than 1%; before they leave the registers 1 to 5%.)
    if (__builtin_expect(__ballot(probe != probe) != 0, 0)) {
        const uint32_t row = r < args.rows ? (uint32_t)(r * args.lda * 2) : kRowOut;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            f32x16 again = zero;
#pragma unroll 1
            for (int g = ga + wave; g < gb; g += KW) {
                const uint32_t rec = rec0 + (uint32_t)g * 128u;
                const u32x4 q = buffer_load16(q_rsrc[w], rec * 32u + 16u * h, 0);
                const float s = bf16_bits_to_f32(buffer_load_u16(s_rsrc[w], rec * 2u, 0));
                const float b = bf16_bits_to_f32(buffer_load_u16(b_rsrc[w], rec * 2u, 0));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const u32x4 x = buffer_load16(a_rsrc, row + (uint32_t)g * 128u + 16u * (4 * h + i), 0);
                    again = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(x), dequant_word_fp8(q[i], s, b), again, 0, 0, 0);
                }
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                float *sum = red + ((wave * NW + w) * E + e) * 64 + lane;
                const float none = *sum * 0.0f;
                if (none != none) *sum = again[e];
            }
        }
    }
    __syncthreads();
    // Thread t takes outputs t, t + kThreads, ... of the block's E x 64 in the MFMA's layout.
    constexpr int V = S::kVals;
    float v[NW * V];
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const int o = tid + j * S::kThreads;
            float x = 0.0f;
            if (o < E * 64) {
#pragma unroll
                for (int s = 0; s < KW; ++s) x += red[(s * NW + w) * E * 64 + o];
            }
            v[w * V + j] = x;
        }
    if (tb >= 0 && !balance_merge<NW * V>(v, tid, S::kActive, tb, sl, args.slices, args.partial, args.partial_bytes,
                                          args.counters))
        return;  // a slice whose block another slice finishes
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int o = tid + j * S::kThreads;
        const int e = o >> 6, l = o & 63;
        const int m = 8 * (e >> 2) + 4 * (l >> 5) + (e & 3);
        if (o >= E * 64 || m >= args.rows) continue;
        auto store = [&](int64_t index, float value) {
            if (args.out_dtype == SPLOSH_F32) {
                if (args.residual) value += ((const float *)args.residual)[index];
                ((float *)out)[index] = value;
            } else {
                if (args.residual) value += bf16_bits_to_f32(((const uint16_t *)args.residual)[index]);
                ((uint16_t *)out)[index] = f32_to_bf16(value);
            }
        };
        const int64_t index = m * ldc + n0 + (l & 31);
        store(index, MODE == kSkinnyMlp ? silu(v[j]) * v[NW * V - V + j] : v[j]);
        if constexpr (MODE == kSkinnySplit) store(index + args.half, v[V + j]);
    }
}

static int skinny_rows(int64_t rows) { return rows <= 8 ? 8 : rows <= 16 ? 16 : 32; }

// How a call is cut: KW waves a workgroup, and K slices of its blocks of 32 columns (NW weights
// each). Four waves where every CU gets at least two workgroups, else eight (K5120 -> N5120, 160
// blocks, 8 rows: 9.8 us at four waves, 7.8 at eight; gate+up, 544 blocks: 22 and 24.7). K is sliced
//  * for the last round of many blocks (plan_balance);
//  * for at most half a block a CU, one workgroup a CU, from K4096 (where a block gets fewer than four slices from
//    K4608, or K5120 at one weight of up to four rows): four rows of K5120 -> N1024 6.8 -> 6.0 us in 5 slices, K4096
//    -> N1024 6.0 -> 5.75 in 4, but K4096 -> N2560 6.2 -> 7.0 in 3, K3072 -> N1024 5.2 -> 5.5 in 3, K2048 4.4 -> 5.2
//    in 2; 16 rows of the pair of K4608 -> 2 x N2560 10.7 -> 9.95 in 3;
//  * for fewer blocks than CUs and long K (24 groups a wave), two workgroups a CU (K17408 -> N5120:
//    18.9 -> 17.3 us): the merge costs about 3 us, which shorter K does not win back (K5120 -> N5120
//    8.2 -> 9.8).
// The registers of two weights and 32 rows leave a CU one workgroup of eight waves or three of four. So the pair
// takes four waves from a block a CU (a second round of eight-wave workgroups would find most CUs empty: 24 rows of
// K4096 -> 2 x N12288 21.6 -> 19.6 us, of K1536 13.9 -> 10.4; 16 rows of K5120 21.3 -> 20.0, at 8 rows level), and its
// slices of 17 to 32 rows are planned for one workgroup a CU (K17408 -> 2 x N4096, 24 rows 33.8 -> 26.5 us; the
// stream-K kernel 27.8). At 32 rows that kernel is still up to 17% faster where its bands come out whole (K5120 -> 2 x
// N12288 26.0 here, 23.6), on weights rounded to bf16.
constexpr int kSkinnyLong = 24;
struct SkinnyPlan {
    int kw;
    BalanceSplit split;
};
static SkinnyPlan plan_skinny(int64_t blocks, int groups, int64_t rows, int nw) {
    SkinnyPlan p;
    const int cus = device_cus();
    p.kw = blocks >= 2 * cus || (nw == 2 && rows > 8 && blocks > cus) ? 4 : 8;
    p.split = plan_balance(blocks, cus, groups);
    const int per_cu = groups < kSkinnyLong * p.kw || (nw == 2 && rows > 16) ? 1 : 2;
    int s = 1;
    const int least = 4 * blocks <= cus ? 64 : nw == 1 && rows <= 4 ? 80 : 72;
    if (2 * blocks <= cus) s = groups < least ? 1 : (int)(cus / blocks) * per_cu;
    else if (blocks < cus && per_cu == 2) s = (int)(2 * cus / blocks);
    s = s < kBalanceMaxSlices ? s : kBalanceMaxSlices;
    while (s >= 2 && (groups < 2 * s * p.kw || blocks * s % 8 != 0)) --s;
    if (s >= 2) p.split = BalanceSplit{0, (int)blocks, s};
    return p;
}

// One weight as the pair of its column halves (half the activation traffic, row sums and operand
// permutes a weight), where the pairs still fill the chip: two a CU (lm_head, 16 rows 181 -> 153 us;
// 32 rows 242 -> 183), one a CU in place of an uneven two (K5120 -> N12288, 8 rows 12.6 -> 10.8), or
// K slices that make up for them (K17408 -> N5120, 16 rows 19.9 -> 17.5). Not between one and two a
// CU (N17408, 272 pairs: 15.6 -> 19).
static bool skinny_split(int64_t columns, int groups) {
    const int64_t cus = device_cus(), blocks = columns / kSkinnyCols, pairs = blocks / 2;
    if (columns % 256 != 0) return false;  // the halves start on a 128-row tile
    return pairs >= 2 * cus || (blocks > cus && pairs <= cus) ||
           (blocks <= cus && 2 * blocks > cus && groups >= kSkinnyLong * 8);
}

// Shapes the kernel takes: tiled weights, 32-bit offsets, activations under 1 GiB, up to 16 rows.
// Above (17 to 32 rows: the scaling doubles with the accumulators) only where it still wins over the
// stream-K kernel: the fused pair (31 against 32.5 us), split weights of two pairs a CU (the
// lm_head: 183 against 191), and at most a block a CU of short K (K5120 -> N5120 10.1-11 against
// 11.6, q/k/v 11.5 against 14).
bool skinny_fits(int64_t rows, int64_t columns, int64_t inner, int64_t lda, bool pair) {
    if (rows < 1 || rows > 32 || columns % 128 != 0 || inner % kGroup != 0 ||
        (rows * lda + inner) * 2 >= ((int64_t)1 << 30) || columns * (inner / kGroup) * 32 >= ((int64_t)1 << 32) - 4096)
        return false;
    const int64_t cus = device_cus(), blocks = columns / kSkinnyCols;
    return rows <= 16 || pair || (columns % 256 == 0 && blocks / 2 >= 2 * cus) ||
           (blocks <= cus && inner / kGroup < kSkinnyLong * 8);
}

// The calls of up to four rows that stay on the decode kernel where it takes them: one and two rows, and one
// weight of at most half a block a CU with K1280 or K1536 (us, decode / here: three rows of K1536 -> N2048 4.0 /
// 4.4, N512 3.8 / 3.9; but K1024 -> N2048 4.0 / 3.45, K1792 5.0 / 4.4, and K1536 -> N4608 5.1 / 4.55; the pair of
// K1536 -> 2 x N2048 is level).
bool decode_before_skinny(int64_t rows, int64_t columns, int64_t inner, bool pair) {
    const int64_t groups = inner / kGroup;
    return rows <= 2 || (rows <= 4 && !pair && 2 * (columns / kSkinnyCols) <= device_cus() && groups > 16 && groups <= 24);
}

static size_t skinny_need(const SkinnyPlan &p, int64_t rows, int nw) {
    if (p.split.slices < 2) return 0;
    const int rm = skinny_rows(rows), e = rm / 2;
    const int vals = (e + p.kw - 1) / p.kw, active = e * 64 < p.kw * 64 ? e * 64 : p.kw * 64;
    return kBalanceCounterBytes + (size_t)p.split.tail * p.split.slices * nw * vals * active * sizeof(float);
}

size_t skinny_workspace_bytes(int64_t rows, int64_t columns, int64_t inner, int nw) {
    if (!skinny_fits(rows, columns, inner, inner, nw == 2)) return 0;
    const int groups = (int)(inner / kGroup);
    size_t need = skinny_need(plan_skinny(columns / kSkinnyCols, groups, rows, 1), rows, 1);
    const size_t pair = nw == 2 ? skinny_need(plan_skinny(columns / kSkinnyCols, groups, rows, 2), rows, 2) : 0;
    need = need > pair ? need : pair;
    if (!skinny_split(columns, groups)) return need;
    const size_t split = skinny_need(plan_skinny(columns / (2 * kSkinnyCols), groups, rows, 2), rows, 2);
    return need > split ? need : split;
}

// Groups in flight a wave. Two leave the registers for more waves and measured as fast as three to
// five or faster (K5120 -> N5120, 8 rows: 7.3, 7.9, 8.2, 7.9 us at 2, 3, 4, 5; 32 rows 11.0 and 12.2
// at 2 and 3).
constexpr int kSkinnyDepth = 2;

template <SkinnyMode MODE, int RM, int KW>
static hipError_t launch_skinny_v(const SkinnyArgs &args, int64_t blocks, hipStream_t stream) {
    using S = SkinnyShape<RM, KW, kSkinnyDepth>;
    auto kernel = q4_skinny_kernel<MODE, RM, KW, kSkinnyDepth>;
    constexpr size_t lds = S::lds(skinny_nw(MODE));
    if constexpr (lds > 64 * 1024) {
        static const bool once = [&] {
            (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            return true;
        }();
        (void)once;
    }
    const int64_t grid = args.slices > 1 ? args.nwhole + (int64_t)args.tail * args.slices : blocks;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(KW * 64), lds, stream, args);
    return hipGetLastError();
}

template <SkinnyMode MODE, int RM>
static hipError_t launch_skinny_rm(const SkinnyArgs &args, int kw, int64_t blocks, hipStream_t stream) {
    return kw == 4 ? launch_skinny_v<MODE, RM, 4>(args, blocks, stream) : launch_skinny_v<MODE, RM, 8>(args, blocks, stream);
}

template <SkinnyMode MODE>
static hipError_t launch_skinny(SkinnyArgs &args, int64_t blocks, int64_t rows, void *workspace, size_t workspace_bytes,
                                hipStream_t stream) {
    const int rm = skinny_rows(rows);
    const SkinnyPlan p = plan_skinny(blocks, args.groups, rows, skinny_nw(MODE));
    const size_t need = skinny_need(p, rows, skinny_nw(MODE));
    args.slices = 1;
    if (need > 0 && workspace && workspace_bytes >= need) {
        args.nwhole = p.split.nwhole;
        args.tail = p.split.tail;
        args.slices = p.split.slices;
        args.counters = (int *)workspace;
        args.partial = (float *)((char *)workspace + kBalanceCounterBytes);
        args.partial_bytes = (uint32_t)(need - kBalanceCounterBytes);
    }
    if (rm == 8) return launch_skinny_rm<MODE, 8>(args, p.kw, blocks, stream);
    if (rm == 16) return launch_skinny_rm<MODE, 16>(args, p.kw, blocks, stream);
    return launch_skinny_rm<MODE, 32>(args, p.kw, blocks, stream);
}

static void skinny_io(SkinnyArgs &args, int64_t inner, const uint16_t *a, int64_t lda, void *out, int64_t ldc,
                      int out_dtype, const void *residual, int64_t rows) {
    args.groups = (int)(inner / kGroup);
    args.a = a;
    args.lda = lda;
    args.out = out;
    args.ldc = ldc;
    args.residual = residual;
    args.rows = (int)rows;
    args.out_dtype = out_dtype;
    args.a_bytes = (uint32_t)(((rows - 1) * lda + inner) * 2);
}

hipError_t launch_q4_skinny(const splosh_q4_weight &w, const splosh_q4_weight *up, const uint16_t *a, int64_t lda,
                            void *out, int64_t ldc, int out_dtype, const void *residual, int64_t rows, void *workspace,
                            size_t workspace_bytes, hipStream_t stream) {
    SkinnyArgs args = {};
    skinny_io(args, w.inner, a, lda, out, ldc, out_dtype, residual, rows);
    const bool split = !up && skinny_split(w.rows, args.groups);
    const int64_t columns = split ? w.rows / 2 : w.rows;
    // Row `columns`'s first record (the second half of a split weight): whole 128-row tiles.
    const int64_t rec = columns * args.groups;
    args.half = columns;
    args.packed[0] = w.packed;
    args.scales[0] = w.scales;
    args.biases[0] = w.biases;
    args.packed[1] = up ? up->packed : split ? w.packed + rec * 8 : w.packed;
    args.scales[1] = up ? up->scales : split ? w.scales + rec : w.scales;
    args.biases[1] = up ? up->biases : split ? w.biases + rec : w.biases;
    args.code_bytes = (uint32_t)(rec * 32);
    args.sidecar_bytes = (uint32_t)(rec * 2);
    const int64_t blocks = columns / kSkinnyCols;
    if (up) return launch_skinny<kSkinnyMlp>(args, blocks, rows, workspace, workspace_bytes, stream);
    return split ? launch_skinny<kSkinnySplit>(args, blocks, rows, workspace, workspace_bytes, stream)
                 : launch_skinny<kSkinnyOne>(args, blocks, rows, workspace, workspace_bytes, stream);
}

hipError_t launch_q4_skinny_group(const splosh_q4_weight *w, int count, void *const *outs, const int64_t *ldcs,
                                  const uint16_t *a, int64_t lda, int out_dtype, int64_t rows, void *workspace,
                                  size_t workspace_bytes, hipStream_t stream) {
    SkinnyArgs args = {};
    skinny_io(args, w[0].inner, a, lda, outs[0], ldcs[0], out_dtype, nullptr, rows);
    args.ngroup = count;
    int blk = 0;
    for (int i = 0; i < count; ++i) {
        args.gblk[i] = blk;
        args.gpacked[i] = w[i].packed;
        args.gscales[i] = w[i].scales;
        args.gbiases[i] = w[i].biases;
        args.gout[i] = outs[i];
        args.gldc[i] = ldcs[i];
        blk += (int)(w[i].rows / kSkinnyCols);
    }
    args.gblk[count] = blk;
    return launch_skinny<kSkinnyGroup>(args, blk, rows, workspace, workspace_bytes, stream);
}

}  // namespace splosh
