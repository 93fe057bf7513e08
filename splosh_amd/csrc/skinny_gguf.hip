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
#include "gguf_half.hpp"
#include "launch.hpp"

namespace splosh {

struct SkinnyGgufArgs : GgufSource {
    int64_t n;
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
        Half<TYPE>::build(lds + S::kTblAt, tid, S::kThreads);
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

// And the calls it is the fastest for (native blocks: of those past the streaming kernels' rows, whose
// weights are not rounded; us, K17408 -> N5120, file order, this kernel against the kernel
// before it): 5 to 16 rows of every type (8 rows: Q8_0 30.3 / 33.1, Q6_K 27.9 / 43.0, Q3_K 21.6 /
// 46.1, IQ3_S 26.2 / 42.4, IQ4_NL 23.3 / 27.2, IQ4_XS 23.0 / 30.0, Q4_K 18.7 / 21.8, Q5_K 21.4 /
// 23.8); two to four rows of the planes (K5120 -> N3328: Q4_K 8.4 / 11.6, Q5_K 9.9 / 12.3; N2560, below
// the line, on mma.hip 11.0 and 11.9) and four of IQ4_NL, from 2048 blocks x units; 17 to 32 rows, where
// the activations' traffic grows, of the types whose loads weigh most in mma.hip (32 rows: Q6_K 39.2 /
// 43.2, Q3_K 31.8 / 46.3, IQ3_S 35.4 / 42.8, IQ4_XS in the file's order 32.3 / 34.1; not Q8_0 41.0 / 38.6).
// Not between one and two blocks a CU, where a last round of workgroups leaves CUs idle, of the types that cost
// mma.hip the least, from the rows at which it is the faster: where its bands come out whole (us, here / there: Q5_K 16
// rows of K4096 -> N14336 15.4 / 14.7, of K1536 -> N12288 8.9 / 7.8 and at 7 rows 8.0 / 7.7; Q8_0 in the ROWS32 order 9 rows
// of K4096 -> N12288 16.3 / 15.0, in the file's 19.3 / 21.6 but of K1536 10.5 / 9.1; IQ4_XS in the file's order 24 rows of
// K1536 10.4 / 9.1), and at long K (K8192 -> N9216, 16 rows: Q5_K 25.2 / 22.2, Q8_0 43 / 34).
static bool sg_uneven(int type, bool rows32, int64_t rows, int64_t columns, int64_t inner) {
    const int64_t cus = device_cus(), blocks = (columns + kSgCols - 1) / kSgCols, units = inner / 256;
    if (blocks <= cus || blocks >= 2 * cus) return false;
    const bool shortk = units < 8, longk = units >= kSgLong;
    int64_t from = 33;
    if (type == 12 || type == 13) from = shortk ? 1 : longk ? 9 : 13;
    else if (type == 8) from = shortk || longk ? 1 : rows32 ? 9 : 33;
    else if ((type == 20 || type == 23) && shortk) from = type == 23 && !rows32 ? 17 : 9;
    return rows >= from && (longk || mma_whole_bands(rows, columns, units, 256));
}
bool gguf_skinny_fits(int type, int64_t rows, int64_t columns, int64_t inner, int64_t lda, int64_t weight_bytes) {
    if (!sg_shape(rows, columns, inner, lda) || weight_bytes >= (int64_t)kSgOut - 65536) return false;
    const bool rows32 = gguf_layout(type);
    if (sg_uneven(type, rows32, rows, columns, inner)) return false;
    if (rows <= 4) return rows > 1 && (columns + kSgCols - 1) / kSgCols * (inner / 256) >= 2048;
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
