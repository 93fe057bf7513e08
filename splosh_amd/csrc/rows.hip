// rows.hip -- q4 projections with few outputs (row-major weights, such as the 48-row gated-delta a
// and b projections the engine keeps untiled) for any number of activation rows, VALU only.
//
// Such a weight is 140 KB: nothing bounds the call but latency, so the work is spread until every
// load can be in flight at once. A workgroup computes C outputs of MR activation rows over the
// whole of K: thread e takes the half groups (32 k) e, e + 256, ... of each of its C weight rows,
// so for K <= 8192 every load of the call is issued before the first is waited for, and the only
// reduction is one shuffle tree and one pass through LDS. There is no reduction across workgroups.
//
// Arithmetic as the decode kernel's: a code word becomes four bf16 pairs (128 + q_j, 128 + q_{j+4}),
// which meet the activation pairs (x_j, x_{j+4}) in v_dot2_f32_bf16; per half group, with P = sum x
// (128 + q) and S = sum x, acc += s P + (b - 128 s) S. The weights are exact and the sums fp32.
#include "common.hpp"
#include "launch.hpp"
#include "mix.hpp"

namespace splosh {

typedef __bf16 bf16x2_r __attribute__((ext_vector_type(2)));

struct RowsArgs {
    const uint32_t *packed;
    const uint16_t *scales, *biases;
    int64_t stride_words;
    int64_t n;
    int groups;
    const uint16_t *a;
    int64_t lda;
    void *out;
    int64_t ldc;
    const void *residual;
    int64_t rows;
    int out_dtype;
    uint32_t a_bytes;
};

constexpr int kRowsWg = 256;

__device__ __forceinline__ float rdot2(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_r, a), __builtin_bit_cast(bf16x2_r, b), c, false);
}
__device__ __forceinline__ uint32_t rand_or(uint32_t a, uint32_t mask, uint32_t c) {
    uint32_t d;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "s"(mask), "v"(c));
    return d;
}

// The sums of V values (a power of two, at most 64) over the lanes of a wave, as a reduce-scatter:
// with lane l ^ xm each lane exchanges half of the values it still holds, then the lanes left
// over are summed plainly. Returns the sum of value `slot`, valid in every lane; `lead` marks one
// lane a value.
template <int V>
__device__ __forceinline__ float scatter_sum(float (&x)[V], int lane, int &slot, bool &lead) {
    slot = 0;
    int xm = 32;
#pragma unroll
    for (int half = V / 2; half >= 1; half >>= 1, xm >>= 1) {
        const bool upper = (lane & xm) != 0;
#pragma unroll
        for (int j = 0; j < half; ++j) {
            const float keep = upper ? x[half + j] : x[j], give = upper ? x[j] : x[half + j];
            x[j] = keep + __shfl_xor(give, xm, 64);
        }
        slot += upper ? half : 0;
    }
    lead = (lane & (2 * xm - 1)) == 0;
#pragma unroll
    for (int m = 64 / V / 2; m >= 1; m >>= 1) x[0] += __shfl_xor(x[0], m, 64);
    return x[0];
}

// Half group e of output n and activation row m, each weight dequantized in fp32.
__device__ __forceinline__ float rows_half_dot(const RowsArgs &args, int64_t n, int64_t m, int e) {
    const float s = bf16_bits_to_f32(args.scales[n * args.groups + (e >> 1)]);
    const float b = bf16_bits_to_f32(args.biases[n * args.groups + (e >> 1)]);
    float sum = 0.0f;
#pragma unroll 1
    for (int j = 0; j < 4; ++j) {
        const uint32_t code = args.packed[n * args.stride_words + (int64_t)e * 4 + j];
        const u32x4 x = *(const u32x4 *)(args.a + m * args.lda + (int64_t)e * 32 + 8 * j);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const float w = __builtin_fmaf((float)((code >> (4 * t)) & 15u), s, b);
            sum = __builtin_fmaf(bf16_bits_to_f32(t & 1 ? x[t / 2] >> 16 : x[t / 2] & 0xFFFFu), w, sum);
        }
    }
    return sum;
}

template <int C, int MR>
__global__ void __launch_bounds__(kRowsWg)
q4_rows_kernel(RowsArgs args) {
    constexpr int V = C * MR;
    __shared__ float red[kRowsWg / 64][V];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t n0 = (int64_t)blockIdx.x * C;
    const int64_t m0 = (int64_t)blockIdx.y * MR;
    const int items = 2 * args.groups;  // half groups
    const uint32_t kMask = 0x000F000Fu;
    uint32_t magic;  // the bf16 exponent of 128 in both halves
    asm("v_mov_b32 %0, 0x43004300" : "=v"(magic));

    float acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = 0.0f;
    for (int e = threadIdx.x; e < items; e += kRowsWg) {
        u32x4 code[C];
        uint32_t sb[C], bb[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int64_t n = n0 + c < args.n ? n0 + c : args.n - 1;
            code[c] = *(const u32x4 *)(args.packed + n * args.stride_words + (int64_t)e * 4);
            sb[c] = args.scales[n * args.groups + (e >> 1)];
            bb[c] = args.biases[n * args.groups + (e >> 1)];
        }
        u32x4 x[MR][4];
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            const int64_t row = m0 + m < args.rows ? m0 + m : args.rows - 1;
            const u32x4 *src = (const u32x4 *)(args.a + row * args.lda + (int64_t)e * 32);
#pragma unroll
            for (int j = 0; j < 4; ++j) x[m][j] = src[j];
        }
        uint32_t pair[C][4][4];
        float s[C], bp[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t w = code[c][j];
#pragma unroll
                for (int p = 0; p < 4; ++p) pair[c][j][p] = rand_or(p ? w >> (4 * p) : w, kMask, magic);
            }
            s[c] = bf16_bits_to_f32(sb[c]);
            bp[c] = __builtin_fmaf(-128.0f, s[c], bf16_bits_to_f32(bb[c]));
        }
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            float s0 = 0.0f, s1 = 0.0f;
            float p0[C], p1[C];
#pragma unroll
            for (int c = 0; c < C; ++c) p0[c] = p1[c] = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const u32x4 v = x[m][j];
                s0 = rdot2(v.x, 0x3F803F80u, s0);
                s1 = rdot2(v.y, 0x3F803F80u, s1);
                s0 = rdot2(v.z, 0x3F803F80u, s0);
                s1 = rdot2(v.w, 0x3F803F80u, s1);
                const uint32_t q[4] = {perm_bytes(v.z, v.x, 0x05040100u), perm_bytes(v.z, v.x, 0x07060302u),
                                       perm_bytes(v.w, v.y, 0x05040100u), perm_bytes(v.w, v.y, 0x07060302u)};
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    p0[c] = rdot2(pair[c][j][0], q[0], p0[c]);
                    p1[c] = rdot2(pair[c][j][1], q[1], p1[c]);
                    p0[c] = rdot2(pair[c][j][2], q[2], p0[c]);
                    p1[c] = rdot2(pair[c][j][3], q[3], p1[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < C; ++c)
                acc[c * MR + m] = __builtin_fmaf(s[c], p0[c] + p1[c], __builtin_fmaf(bp[c], s0 + s1, acc[c * MR + m]));
        }
    }
    int slot;
    bool lead;
    float part = scatter_sum<V>(acc, lane, slot, lead);
    // An infinite activation or scale leaves inf - inf in s P + (b - 128 s) S, and one above 2^120 can overflow
    // it where x w does not: a wave with such a sum takes it again with the dequantized weights. (Looking for one
    // here costs 0.05 us a call; before the reduction it cost the loop its registers, 10 to 28% at 2 x 4 outputs.)
    const float none = part * 0.0f;
    if (__builtin_expect(__ballot(none != none) != 0, 0)) {
        float again[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const int64_t n = n0 + v / MR < args.n ? n0 + v / MR : args.n - 1;
            const int64_t m = m0 + v % MR < args.rows ? m0 + v % MR : args.rows - 1;
            again[v] = 0.0f;
#pragma unroll 1
            for (int e = threadIdx.x; e < items; e += kRowsWg) again[v] += rows_half_dot(args, n, m, e);
        }
        const float sum = scatter_sum<V>(again, lane, slot, lead);
        part = none != none ? sum : part;
    }
    if (lead) red[wave][slot] = part;
    __syncthreads();
    if (threadIdx.x >= V) return;
    float value = 0.0f;
#pragma unroll
    for (int w = 0; w < kRowsWg / 64; ++w) value += red[w][threadIdx.x];
    const int64_t n = n0 + threadIdx.x / MR, m = m0 + threadIdx.x % MR;
    if (n >= args.n || m >= args.rows) return;
    const int64_t index = m * args.ldc + n;
    if (args.out_dtype == SPLOSH_F32) {
        if (args.residual) value += ((const float *)args.residual)[index];
        ((float *)args.out)[index] = value;
    } else {
        if (args.residual) value += bf16_bits_to_f32(((const uint16_t *)args.residual)[index]);
        ((uint16_t *)args.out)[index] = f32_to_bf16(value);
    }
}

// More activation rows: 32 x 32 output tiles on v_mfma_f32_32x32x16_bf16. A workgroup of 16 waves
// owns one tile; wave w takes the groups w, w + 16, ... of K, lane (r, h) feeding row / column r
// with k = 32 h + 8 i .. + 7 of the group in step i. The wave's activations of a group (32 rows of
// 128 bytes) go straight into LDS of its own, eight rows a load (read in the operand's own layout,
// every load would touch 32 cache lines: 2048 rows of K5120 -> N48 19.3 us against 16.6), one group ahead of their use; the weight is dequantized in registers (dequant_word_fp8).
// No barrier until the waves' sums meet in LDS, in wave order.
constexpr int kRowsMmaWaves = 16;
constexpr int kRowsTile = 32 * 128;                              // a group's activations of a wave
constexpr size_t kRowsMmaLds = (size_t)kRowsMmaWaves * 2 * kRowsTile;

__global__ void __launch_bounds__(kRowsMmaWaves * 64)
q4_rows_mma_kernel(RowsArgs args) {
    extern __shared__ __align__(16) char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, h = lane >> 5;
    const int64_t n0 = (int64_t)blockIdx.x * 32, m0 = (int64_t)blockIdx.y * 32;
    const int64_t n = n0 + r < args.n ? n0 + r : args.n - 1;
    const uint32_t *code = args.packed + n * args.stride_words + 4 * h;
    const uint16_t *scale = args.scales + n * args.groups, *bias = args.biases + n * args.groups;
    const rsrc_t a_rsrc = make_rsrc(args.a, args.a_bytes);
    // Load j writes rows 8 j .. 8 j + 7 of the tile: lane l row 8 j + l / 8, slot l % 8, holding the
    // row's 16-byte piece (l % 8) ^ (l / 8) (the operand reads of 8 consecutive rows then hit eight
    // different slots). Rows past the last are clamped (their outputs are not stored).
    uint32_t src[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t m = m0 + 8 * j + (lane >> 3);
        src[j] = (uint32_t)(((m < args.rows ? m : args.rows - 1) * args.lda + 8 * ((lane & 7) ^ (lane >> 3))) * 2);
    }
    char *mine = lds + wave * 2 * kRowsTile;
    u32x4 q[2];
    uint32_t s[2], b[2];
    auto load = [&](int buf, int g) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            buffer_load_lds16(a_rsrc, mine + buf * kRowsTile + j * 1024, src[j] + (uint32_t)g * 128u);
        q[buf] = *(const u32x4 *)(code + (int64_t)g * 8);
        s[buf] = scale[g];
        b[buf] = bias[g];
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int kLoads = 7;  // loads a group issues
    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
    const int G = args.groups;
    // Group g of the wave in buffer `buf`, the next one (past the last: clamped, and not multiplied) on its way
    // into the other.
    auto clamp = [&](int g) { return g < G ? g : G - 1; };
    auto step = [&](int g, int buf) {
        load(buf ^ 1, clamp(g + kRowsMmaWaves));
        wait_vmcnt<kLoads>();  // this group has landed; the next may be in flight
        asm volatile("" ::: "memory");
        const float sc = bf16_bits_to_f32(s[buf]), bi = bf16_bits_to_f32(b[buf]);
        const char *a = mine + buf * kRowsTile + r * 128;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(*(const u32x4 *)(a + (((4 * h + i) ^ (r & 7)) << 4))),
                                                         dequant_word_fp8(q[buf][i], sc, bi), acc, 0, 0, 0);
        // The fragments are read before the next step's loads overwrite this buffer.
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    if (wave < G) {
        load(0, wave);
        for (int g = wave; g < G; g += 2 * kRowsMmaWaves) {
            step(g, 0);
            if (g + kRowsMmaWaves >= G) break;
            step(g + kRowsMmaWaves, 1);
        }
    }
    wait_vmcnt<0>();
    __syncthreads();  // every load into LDS has landed: the sums take its place
    float *red = (float *)lds;
#pragma unroll
    for (int e = 0; e < 16; ++e) red[(wave * 16 + e) * 64 + lane] = acc[e];
    __syncthreads();
    // Thread (wave, lane) sums element `wave` of the tile's MFMA layout.
    float value = 0.0f;
#pragma unroll
    for (int w = 0; w < kRowsMmaWaves; ++w) value += red[(w * 16 + wave) * 64 + lane];
    const int64_t m = m0 + 8 * (wave >> 2) + 4 * h + (wave & 3);
    if (n0 + r >= args.n || m >= args.rows) return;
    const int64_t index = m * args.ldc + n0 + r;
    if (args.out_dtype == SPLOSH_F32) {
        if (args.residual) value += ((const float *)args.residual)[index];
        ((float *)args.out)[index] = value;
    } else {
        if (args.residual) value += bf16_bits_to_f32(((const uint16_t *)args.residual)[index]);
        ((uint16_t *)args.out)[index] = f32_to_bf16(value);
    }
}

// Which calls come here: any width at one or two rows (K5120, one row: N=512 17.1 us on the
// lane-per-row kernel, 2.7 here; N=5120 17.7 -> 6.7; N=17408 27.9 -> 17.7; two rows of N=17408 41 ->
// 26); up to kRowsDotOutputs outputs of at most kRowsDotColumns columns on the same kernel
// (N=48: 16 rows 10.0 -> 3.0 us, 64 rows 12 -> 4.7, 333 rows 19 -> 12; N=512, 16 rows 12.2 -> 7.5;
// at 16384 outputs and 64 rows or fewer the M <= 64 kernel is level with it); above 66 rows (65 and 66 are 64
// and a call of one or two, whose weights enter the sums exactly; this kernel rounds them to bf16), while
// there is at most one 32 x 32 tile a CU, the MFMA kernel (N=48: 2048 rows 32.6 -> 14.9 us; N=512,
// 333 rows 22.3 -> 15.1; with two tiles a CU level with the tile kernel, behind it from there).
constexpr int64_t kRowsDotOutputs = 16384, kRowsDotColumns = 1024;

static bool rows_dot(int64_t rows, int64_t columns) {
    return rows <= 2 || (columns <= kRowsDotColumns && rows * columns <= kRowsDotOutputs);
}

bool rows_fit(int64_t rows, int64_t columns, int64_t inner, int64_t lda) {
    if (rows < 1 || inner % kGroup != 0 || columns > (1 << 30) || inner > (1 << 30)) return false;
    if (rows_dot(rows, columns)) return true;
    // (The activations are read through a buffer resource: 32-bit byte offsets.)
    return rows > 66 && (rows + 31) / 32 * ((columns + 31) / 32) <= device_cus() &&
           (rows * lda + inner) * 2 < ((int64_t)1 << 32) - 256;
}

template <int C, int MR>
static hipError_t launch_rows_v(const RowsArgs &args, hipStream_t stream) {
    const dim3 grid((unsigned)((args.n + C - 1) / C), (unsigned)((args.rows + MR - 1) / MR));
    hipLaunchKernelGGL((q4_rows_kernel<C, MR>), grid, dim3(kRowsWg), 0, stream, args);
    return hipGetLastError();
}

hipError_t launch_q4_rows(const splosh_q4_weight &w, const uint16_t *a, int64_t lda, void *out, int64_t ldc,
                          int out_dtype, const void *residual, int64_t rows, hipStream_t stream) {
    RowsArgs args = {};
    args.packed = w.packed;
    args.scales = w.scales;
    args.biases = w.biases;
    args.stride_words = w.row_stride_words;
    args.n = w.rows;
    args.groups = (int)(w.inner / kGroup);
    args.a = a;
    args.lda = lda;
    args.out = out;
    args.ldc = ldc;
    args.residual = residual;
    args.rows = rows;
    args.out_dtype = out_dtype;
    if (!rows_dot(rows, w.rows)) {
        args.a_bytes = (uint32_t)(((rows - 1) * lda + w.inner) * 2);
        static const bool once = [] {
            (void)hipFuncSetAttribute((const void *)q4_rows_mma_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)kRowsMmaLds);
            return true;
        }();
        (void)once;
        const dim3 grid((unsigned)((w.rows + 31) / 32), (unsigned)((rows + 31) / 32));
        hipLaunchKernelGGL(q4_rows_mma_kernel, grid, dim3(kRowsMmaWaves * 64), kRowsMmaLds, stream, args);
        return hipGetLastError();
    }
    // Outputs a workgroup: one while latency is all there is, then activations shared by weight
    // rows and weights by activation rows (N=48, K5120: 33 rows 3.7 / 3.8 / 4.1 us, 64 rows 4.9 / 4.7 /
    // 5.2, 128 rows 7.8 / 7.1 / 6.8 with 1 x 1, 1 x 2 and 2 x 4).
    const int64_t outputs = rows * w.rows;
    if (rows == 1 || outputs <= 2048) return launch_rows_v<1, 1>(args, stream);
    if (rows == 2 || outputs <= 4096) return launch_rows_v<1, 2>(args, stream);
    return launch_rows_v<2, 4>(args, stream);
}

}  // namespace splosh
