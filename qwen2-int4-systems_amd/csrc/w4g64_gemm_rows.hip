// W4G64 GEMM for few products (17 rows up to short prompts; plan_rows draws the
// line): batched decode, draft verification, prompts of a few hundred tokens.  The arithmetic is
// the prefill GEMM's (w4g64_gemm.hip): staged fp16 rows times a power of two,
// exact integer (code - zero) on the matrix cores, the group scale in fp32,
// the row factor last.  What differs is the shape: a 128 x 256 tile is mostly
// padding there, and its few tiles need a K split and a reduction launch to
// fill the chip.
//
//   rows_stage_kernel, rows_stage_swiglu_kernel
//       fp16 values (hi and lo planes for the fp32-class kinds) in MFMA
//       operand order [row tile][group][plane][half][lane][8], so that an
//       operand load is a contiguous kilobyte.
//   rows_gemm_kernel
//       one workgroup of W waves per 16 CT output features, row block of MT
//       row tiles and K range.  Each wave takes a contiguous part of the
//       range's groups over all of the block's rows;
//       the waves' sums meet in LDS at the end.  Two planes meet the same
//       decoded weights, in one sum per group.
//
// Bound by vector memory instructions: one that reads a few bytes of 16 rows
// costs a cache line per lane where one over contiguous lanes costs four.
// With weights, scales and zero points loaded straight into operands gate|up
// 17920x1536 at 24 rows spent 15 us here, 63 cycles per load; with the weights
// by 64-byte runs through the wave's own LDS and the scales staged once per
// workgroup, 8.  Per call with the staging and any reduction, bf16,
// graph-replayed over rotated weights, against the 128 x 256 tiles: 24 x
// 17920x1536 29.0 -> 11.6 us, 24 x 1536x1536 16.0 -> 6.8, 40 x 8960x1536 23.1
// -> 11.1, 128 x 8960x1536 27.9 -> 16.1, 512 x 1536x1536 24.7 -> 14.3, 24 x
// 1536x8960 of the SwiGLU product (fp32) 33.2 -> 17.1, 64 x 1536x8960 fp32 32.7
// -> 22.4.
#include "w4g64_gemm.h"
#include "w4g64_internal.h"

namespace w4g64 {
namespace {

struct RowsArgs {
    const uint16_t* x;      // staged rows, operand order
    const float* rowscale;  // power-of-two row factors
    const uint8_t* qweight;
    const uint16_t* scales;
    const uint8_t* zeros;
    const void* bias;
    int bias_kind;
    void* y;
    int out_kind;
    float* partials;  // [splits][M][N], or null
    int M;
    int N;
    int G;    // groups
    int gps;  // groups per K range, even
    int const_bytes;
    int vec_out;  // y is 16-byte aligned and N % 4 == 0
};

// Operand slot (16-byte unit) of row m, chunk c (8 values, K = 8 c .. 8 c + 7)
// of a plane: [row tile][group][plane][half][lane].
template <int PL>
__device__ __forceinline__ int64_t operand_slot(int m, int c, int plane, int G) {
    return (((((int64_t)(m >> 4) * G + (c >> 3)) * PL + plane) * 2 + (c & 1)) * 64) + ((c >> 1) & 3) * 16 + (m & 15);
}

// Workgroup barrier that covers LDS alone: global loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Order of a wave's own LDS accesses, lane to lane: the hardware keeps it, this
// tells the compiler.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

template <int XK, int THREADS>
__global__ __launch_bounds__(THREADS) void rows_stage_kernel(const void* x, u32x4* out, float* rowscale, int K) {
    constexpr int kPlanes = XK == kF32 ? 2 : 1;
    constexpr int kHeld = 2;
    __shared__ float wmax[THREADS / 64];
    const int m = blockIdx.x;
    const int chunks = K / 8;
    const int G = K / 64;
    float v[kHeld][8];
    float mx = 0.0f;
    auto largest = [&](const float (&t)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (__builtin_isfinite(t[i])) mx = fmaxf(mx, fabsf(t[i]));
    };
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
        const int c = threadIdx.x + THREADS * u;
        if (c < chunks) {
            stage_load8<XK>(x, m, K, c, v[u]);
            largest(v[u]);
        }
    }
    for (int c = threadIdx.x + THREADS * kHeld; c < chunks; c += THREADS) {  // (read again below)
        float t[8];
        stage_load8<XK>(x, m, K, c, t);
        largest(t);
    }
    float inv = 1.0f, rs = 1.0f;
    if constexpr (XK != kF16) {
        mx = wave_max64(mx);
        if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < THREADS / 64; ++w) mx = fmaxf(mx, wmax[w]);
        row_factors(mx, inv, rs);
    }
    if (threadIdx.x == 0) rowscale[m] = rs;
    auto store = [&](int c, const float (&t)[8]) {
        u32x4 hi, lo;
        stage_split8(t, inv, hi, lo);
        out[operand_slot<kPlanes>(m, c, 0, G)] = hi;
        if constexpr (kPlanes == 2) out[operand_slot<kPlanes>(m, c, 1, G)] = lo;
    };
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
        const int c = threadIdx.x + THREADS * u;
        if (c < chunks) store(c, v[u]);
    }
    for (int c = threadIdx.x + THREADS * kHeld; c < chunks; c += THREADS) {
        float t[8];
        stage_load8<XK>(x, m, K, c, t);
        store(c, t);
    }
}

// The SwiGLU product, one workgroup per row and 4096 values: its exponentials
// and divisions, on one CU per row, took 7.0 us at 24 x 8960.  Every
// workgroup of a row scans all of it for the largest finite product, so they
// agree on the row's factor.  The scan's products come of the exponential and
// reciprocal instructions: within 2^-16 of the staged ones, which moves the
// factor of a row whose maximum lies that close to a power of two, and the
// largest staged value from [2^14, 2^15) to at most 2^15 (1 + 2^-16).
// (max|gate| times max|up| in its place loses the row where they lie in
// different columns or the gate is negative.)  Threads per workgroup, us per
// call of 24, 64 and 160 x 1536x8960: 256 17.05, 25.0, 31.4; 512 17.1, 24.0,
// 30.5; 1024 18.3, 25.5, 31.3 (16.7, 24.4, 30.1 were those of the lost rows).
constexpr int kSwigluThreads = 512;
__global__ __launch_bounds__(kSwigluThreads) void rows_stage_swiglu_kernel(const void* x, u32x4* out, float* rowscale,
                                                                          int K) {
    __shared__ float wmax[kSwigluThreads / 64];
    const int m = blockIdx.x;
    const int chunks = K / 8;
    const uint16_t* gu = (const uint16_t*)x + (int64_t)m * 2 * K;
    const int own = blockIdx.y * kSwigluThreads + threadIdx.x;
    float v[8];
    if (own < chunks) stage_load8<kSwiGLU>(x, m, K, own, v);
    float mx = 0.0f;
    auto largest = [&](uint32_t gate, uint32_t up) {
        // |g| / (1 + e^-g) |u|; 2^-8 on both sides of the quotient keeps the
        // reciprocal (of at most 2^128) a normal number
        const float g = bf16_bits_to_float(gate), u = bf16_bits_to_float(up);
        const float e = __builtin_amdgcn_exp2f(g * -1.4426950408889634f);
        const float p = (fabsf(g) * 0x1p-8f) * __builtin_amdgcn_rcpf(__builtin_fmaf(e, 0x1p-8f, 0x1p-8f)) * fabsf(u);
        mx = p < INFINITY ? fmaxf(mx, p) : mx;  // (neither infinite nor NaN)
    };
    for (int c = threadIdx.x; c < chunks; c += kSwigluThreads) {
        const u32x4 g = *(const u32x4*)(gu + 8 * c), u = *(const u32x4*)(gu + K + 8 * c);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            largest(g[i] & 0xFFFFu, u[i] & 0xFFFFu);
            largest(g[i] >> 16, u[i] >> 16);
        }
    }
    mx = wave_max64(mx);
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kSwigluThreads / 64; ++w) mx = fmaxf(mx, wmax[w]);
    float inv, rs;
    row_factors(mx, inv, rs);
    if (threadIdx.x == 0 && blockIdx.y == 0) rowscale[m] = rs;
    if (own < chunks) {
        u32x4 hi, lo;
        stage_split8(v, inv, hi, lo);
        out[operand_slot<2>(m, own, 0, K / 64)] = hi;
        out[operand_slot<2>(m, own, 1, K / 64)] = lo;
    }
}

template <int PL, int MT, int CT, int W>
__global__ __launch_bounds__(64 * W) void rows_gemm_kernel(RowsArgs a) {
    constexpr int kRows = 16 * MT, kCols = 16 * CT;
    constexpr int kStride = kCols + 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15;
    const int q = lane >> 4;
    const int n0 = blockIdx.x * kCols;
    const int t0 = blockIdx.z * MT;        // first row tile
    const int first = blockIdx.y * a.gps;  // (gps is even)
    const int count = min(a.gps, a.G - first);
    const int pairs = (count + 1) / 2;
    const int beg = first + 2 * (pairs * wave / W);  // this wave's groups: whole pairs
    const int end = min(first + 2 * (pairs * (wave + 1) / W), first + count);
    // LDS: per group of the range and column the scale and the zero point's
    // constants; per wave CT kilobytes of packed weights
    u32x2* consts = (u32x2*)smem;
    unsigned char* mine = smem + a.const_bytes + 1024 * CT * wave;

    const __amdgpu_buffer_rsrc_t x_rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)(a.x + (int64_t)t0 * a.G * (1024 * PL)), 0,
                                          (int)((uint32_t)(MT * a.G) * (2048u * PL)), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t w_rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)a.qweight, 0, (int)((uint32_t)a.N * (uint32_t)a.G * 32u), kRsrcWord3);

    // ---- scales and zero points: a column's groups by consecutive lanes ----
    constexpr int kOwn = (kCols + W - 1) / W;
    for (int g0 = 0; g0 < count; g0 += 64) {
        const int g = min(g0 + lane, count - 1);
        uint32_t sv[kOwn], zv[kOwn];
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            const uint32_t e = (uint32_t)min(n0 + wave + W * i, a.N - 1) * (uint32_t)a.G + (uint32_t)(first + g);
            sv[i] = a.scales[e];
            zv[i] = (uint32_t)a.zeros[e >> 1] >> (4 * (e & 1));
        }
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            const int zn = __builtin_amdgcn_sbfe((int)zv[i], 0, 4);
            // fp16 bits of 1032 + z (mantissa unit 1) and of 72 + z (mantissa unit 1/16)
            if (g0 + lane < count && wave + W * i < kCols)
                consts[(g0 + lane) * kCols + wave + W * i] =
                    u32x2{__builtin_bit_cast(uint32_t, half_bits_to_float((uint16_t)sv[i])),
                          (uint32_t)(0x6408 + zn) | ((uint32_t)(0x5480 + 16 * zn) << 16)};
        }
    }

    // Packed weights of a pair of groups, 64 bytes of a column: four
    // consecutive lanes load it (operand form straight from memory would be 8
    // bytes of 16 rows per 16 lanes, a cache line each), and it goes through
    // the wave's own LDS.  Piece c of column r in slot c ^ (r / 4 % 4): the
    // 8-byte operand reads of 16 columns meet different banks.
    uint32_t w_at[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
        w_at[c] = (uint32_t)min(n0 + 16 * c + (lane >> 2), a.N - 1) * (uint32_t)a.G * 32u + 16u * (lane & 3);
    unsigned char* w_put = mine + 64 * (lane >> 2) + 16 * ((lane & 3) ^ ((lane >> 4) & 3));
    const unsigned char* w_get[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) w_get[u] = mine + 64 * j + 16 * ((2 * u + (q >> 1)) ^ (j >> 2)) + 8 * (q & 1);

    struct Rows {
        u32x4 x[MT][PL][2];
    };
    auto load_w = [&](u32x4 (&w)[CT], int g) {
#pragma unroll
        for (int c = 0; c < CT; ++c)
            w[c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, w_at[c], 32 * g, 0));
    };
    auto load_x = [&](Rows& t, int g) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int p = 0; p < PL; ++p)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    t.x[m][p][h] = __builtin_bit_cast(
                        u32x4, __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, 16 * lane + 1024 * (2 * p + h),
                                                                     2048 * PL * (m * a.G + g), 0));
    };
    float4v acc[MT][CT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[m][c] = float4v{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const Rows& t, int g, int u) {  // u: the group's half of its pair
        u32x4 f[CT][2];
        float sc[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const u32x2 w = *(const u32x2*)(w_get[u] + 1024 * c);
            const u32x2 k = consts[(g - first) * kCols + 16 * c + j];
            const uint32_t scale = k[0], zero = k[1];  // (a bit cast of a vector's element reads element 0)
            sc[c] = __builtin_bit_cast(float, scale);
            const half2v z = __builtin_bit_cast(half2v, zero);
#pragma unroll
            for (int h = 0; h < 2; ++h) f[c][h] = decode_codes(w[h], half2v{z[0], z[0]}, half2v{z[1], z[1]});
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                float4v d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int p = PL - 1; p >= 0; --p)  // lo before hi: the sum is of hi's size for two products only
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, t.x[m][p][h]),
                                                                   __builtin_bit_cast(half8, f[c][h]), d, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[m][c][r] = __builtin_fmaf(sc[c], d[r], acc[m][c][r]);
            }
    };
    auto put_w = [&](const u32x4 (&w)[CT]) {  // after the last pair's reads, before this one's
        wave_lds_order();
#pragma unroll
        for (int c = 0; c < CT; ++c) *(u32x4*)(w_put + 1024 * c) = w[c];
        wave_lds_order();
    };
    Rows x0, x1;
    u32x4 w[CT];
    if (beg < end) {
        load_w(w, beg);
        load_x(x0, beg);
        load_x(x1, min(beg + 1, end - 1));
    }
    lds_barrier();  // the constants are in place (loads stay in flight)
    if (beg < end) {
        int g = beg;
        for (; g + 2 < end; g += 2) {
            put_w(w);
            load_w(w, g + 2);
            compute(x0, g, 0);
            load_x(x0, g + 2);
            compute(x1, g + 1, 1);
            load_x(x1, min(g + 3, end - 1));
        }
        put_w(w);
        compute(x0, g, 0);
        if (g + 1 < end) compute(x1, g + 1, 1);
    }

    // ---- the waves' sums meet in LDS, added in wave order ----
    lds_barrier();
    float(*so)[kRows][kStride] = (float(*)[kRows][kStride])smem;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) so[wave][16 * m + 4 * q + r][16 * c + j] = acc[m][c][r];
    __syncthreads();
    for (int e = tid; e < kRows * kCols / 4; e += 64 * W) {
        const int local = e / (kCols / 4);
        const int row = 16 * t0 + local;
        const int col = 4 * (e % (kCols / 4));
        const int n = n0 + col;
        if (row >= a.M || n >= a.N) continue;
        float4v sum = *(const float4v*)&so[0][local][col];
#pragma unroll
        for (int w = 1; w < W; ++w) sum += *(const float4v*)&so[w][local][col];
        sum *= a.rowscale[row];
        const int64_t at = (int64_t)row * a.N + n;
        if (a.partials) {
            float* to = a.partials + (int64_t)blockIdx.y * a.M * a.N + at;
            for (int i = 0; i < 4 && n + i < a.N; ++i) to[i] = sum[i];
            continue;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] += load_bias(a.bias, a.bias_kind, n + i < a.N ? n + i : a.N - 1);
        if (PL == 2 || a.out_kind == kF32) {
            float* to = (float*)a.y + at;
            if (a.vec_out) *(float4v*)to = sum;
            else
                for (int i = 0; i < 4 && n + i < a.N; ++i) to[i] = sum[i];
            continue;
        }
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = a.out_kind == kF16 ? float_to_half_bits(sum[i]) : float_to_bf16_bits(sum[i]);
        uint16_t* to = (uint16_t*)a.y + at;
        if (a.vec_out) *(u32x2*)to = u32x2{v[0] | (v[1] << 16), v[2] | (v[3] << 16)};
        else
            for (int i = 0; i < 4 && n + i < a.N; ++i) to[i] = (uint16_t)v[i];
    }
}

bool two_planes(int x_kind) { return x_kind == kF32 || x_kind == kSwiGLU; }

}  // namespace

// Row blocks, waves and columns per workgroup, K ranges.  Measured per call.
// Up to four row tiles (two of two planes with K to 4096), one block (24, 40
// and 64 rows; CT x W with one range, or with the ranges given):
//   up to 256 column tiles, K up to 4096: 1 x 8 (2048x1536 at 24 rows 7.0 us
//     against 7.2 for 1 x 4 and 7.6 for 2 x 8; 4096x4096 at 40 11.0, 11.7, 12.3);
//   more column tiles: 1 x 4 while they are few enough to be one round of
//     workgroups (8960x1536 at 40 rows 11.1, 2 x 4 11.6; 17920x1536 at 24 12.0,
//     2 x 4 11.6);
//   longer K: 2 x 8 and as many ranges as keep one workgroup per CU
//     (1536x8960 at 40 rows: one range 17.0, two of 1 x 8 15.0, four of 2 x 8
//     14.7).
// More rows: blocks of two row tiles, 2 x 8, while those are at most one
// workgroup per CU (128 x 1536x1536 8.0 us, blocks of four 9.4, one of eight
// 10.1), else of up to four, with four waves past one workgroup per CU (256 x
// 8960x1536 22.8, blocks of eight 27.0; 512 x 1536x1536 14.3, eight waves 16.9);
// 64 x 8960x1536 of two planes 19.3 in one block, 14.0 in two.
// The line to the 128 x 256 tiles (that kernel | this one):
//   one round of workgroups, or K of 1024 to 4096 up to 6e9 products: 160 x
//     1536x1536 18.9 | 9.5, 2048 x 256x1536 26.6 | 19.1, 512 x 2048x1536 27.0 |
//     15.1, 333 x 8960x1536 35.9 | 28.7, 2048 x 1536x1536 40.6 | 33.3; past
//     that they meet: 512 x 8960x1536 37.5 | 36.1, 200 x 16384x2560 44.1 | 43.9;
//   shorter K is the join of the waves' sums alone: 2048 x 1536x256 14.4 | 16.5;
//   longer K: 256 x 1536x8960 32.8 | 27.0, but 512 x 1536x8960 39.5 | 40.9 and
//     200 x 10000x6400 63.0 | 67.9;
//   many rows of few features, where the staging decides: 4096 x 256x1536
//     28.3 | 30.5;
//   two planes: 512 x 4096x1536 35.1 | 30.8, 333 x 8960x1536 43.5 | 41.8, 160 x
//     1536x8960 36.2 | 27.5, but 256 x 1536x8960 36.7 | 42.0, 512 x 512x9216
//     35.0 | 43.8 and 2048 x 256x1536 25.7 | 30.4.
// A range holds at most 160 groups (40 KB of scales and zero points in LDS).
RowsPlan plan_rows(int64_t rows, int64_t out_features, int64_t in_features, int x_kind) {
    RowsPlan pl{};
    const bool two = two_planes(x_kind);
    const int64_t tiles = (rows + 15) / 16;
    if (tiles < 2) return pl;
    const int G = (int)(in_features / 64);
    const int64_t columns = (out_features + 15) / 16;
    pl.blocks = 1;
    pl.cols = 1;
    pl.waves = 8;
    int64_t splits = 1;
    const int64_t pairs = (columns + 1) / 2;
    if (tiles > 4 || (two && tiles > 2 && G <= 64)) {
        const int64_t most = pairs * ((tiles + 1) / 2) <= 256 ? 2 : 4;  // tiles per block
        const int64_t blocks = (tiles + most - 1) / most;
        pl.tiles = (int)((tiles + blocks - 1) / blocks);
        pl.blocks = (int)blocks;
        pl.cols = 2;
        pl.waves = pairs * blocks <= 256 ? 8 : 4;
        const double products = (double)rows * (double)out_features * (double)in_features;
        if (tiles > (two ? 4 : 8)) {
            if (rows > (two ? 1024 : 2048)) return pl;
            if (G > 64 && (two ? most > 2 || products > 2.3e9 : pairs * blocks > 256 && products > 4e9)) return pl;
            if (G <= 64 && pairs * blocks > 256 && (G < 16 || products > (two ? 4e9 : 6e9))) return pl;
        }
    } else {
        pl.tiles = (int)tiles;
        if (G > 64) {
            pl.cols = 2;
            splits = 224 / pairs;
            splits = splits < G / 16 ? splits : G / 16;
        } else if (columns > 256) {
            pl.cols = columns <= 640 ? 1 : 2;
            pl.waves = 4;
        }
    }
    const int64_t staged = (int64_t)pl.blocks * pl.tiles * 16 * in_features * (two ? 4 : 2);
    if (staged >= (int64_t(1) << 31)) return pl;  // 32-bit operand offsets
    const int64_t least = (G + 159) / 160;
    splits = splits < least ? least : splits;
    pl.gps = (int)((G + splits - 1) / splits + 1) / 2 * 2;
    pl.splits = (G + pl.gps - 1) / pl.gps;
    auto up256 = [](int64_t v) { return (v + 255) / 256 * 256; };
    pl.staged_offset = up256(pl.splits > 1 ? (int64_t)pl.splits * rows * out_features * 4 : 0);
    pl.rowscale_offset = pl.staged_offset + up256(staged);
    pl.workspace_bytes = pl.rowscale_offset + rows * 4;
    pl.taken = true;
    return pl;
}

namespace {
template <int PL, int MT, int CT, int W>
hipError_t launch_shape(RowsArgs args, const RowsPlan& pl, hipStream_t stream, hipEvent_t stop) {
    args.const_bytes = args.gps * 16 * CT * 8;
    const dim3 grid((unsigned)((args.N + 16 * CT - 1) / (16 * CT)), (unsigned)pl.splits, (unsigned)pl.blocks);
    const size_t sums = (size_t)W * (16 * MT) * (16 * CT + 4) * 4, work = (size_t)args.const_bytes + 1024 * CT * W;
    return launch_kernel(rows_gemm_kernel<PL, MT, CT, W>, grid, dim3(64 * W), sums > work ? sums : work, stream,
                         nullptr, stop, args);
}
template <int PL, int MT>
hipError_t launch_tiles(const RowsArgs& args, const RowsPlan& pl, hipStream_t stream, hipEvent_t stop) {
    if (pl.waves == 4)
        return pl.cols == 1 ? launch_shape<PL, MT, 1, 4>(args, pl, stream, stop)
                            : launch_shape<PL, MT, 2, 4>(args, pl, stream, stop);
    return pl.cols == 1 ? launch_shape<PL, MT, 1, 8>(args, pl, stream, stop)
                        : launch_shape<PL, MT, 2, 8>(args, pl, stream, stop);
}
template <int PL>
hipError_t launch_planes(const RowsArgs& args, const RowsPlan& pl, hipStream_t stream, hipEvent_t stop) {
    switch (pl.tiles) {
        case 2: return launch_tiles<PL, 2>(args, pl, stream, stop);
        case 3: return launch_tiles<PL, 3>(args, pl, stream, stop);
        case 4: return launch_tiles<PL, 4>(args, pl, stream, stop);
        default: break;
    }
    return hipErrorInvalidValue;
}
template <int XK>
hipError_t launch_stage(const LinearProblem& p, u32x4* staged, float* rowscale, hipStream_t stream, hipEvent_t start) {
    const int k = (int)p.in_features;
    const dim3 grid((unsigned)p.rows);
    return k <= 4096 ? launch_kernel(rows_stage_kernel<XK, 256>, grid, dim3(256), 0, stream, start, nullptr, p.x, staged, rowscale, k)
                     : launch_kernel(rows_stage_kernel<XK, 1024>, grid, dim3(1024), 0, stream, start, nullptr, p.x, staged, rowscale, k);
}
}  // namespace

hipError_t launch_rows(const LinearProblem& p, const RowsPlan& pl, void* workspace, hipStream_t stream,
                       hipEvent_t start, hipEvent_t stop) {
    u32x4* staged = (u32x4*)((char*)workspace + pl.staged_offset);
    float* rowscale = (float*)((char*)workspace + pl.rowscale_offset);
    const bool two = two_planes(p.x_kind);
    RowsArgs args{};
    args.x = (const uint16_t*)staged;
    args.rowscale = rowscale;
    args.qweight = p.qweight;
    args.scales = p.scales;
    args.zeros = p.zeros;
    args.bias = p.bias;
    args.bias_kind = p.bias_kind;
    args.y = p.y;
    args.out_kind = two ? (int)kF32 : p.x_kind;
    args.partials = pl.splits > 1 ? (float*)workspace : nullptr;
    args.M = (int)p.rows;
    args.N = (int)p.out_features;
    args.G = (int)(p.in_features / 64);
    args.gps = pl.gps;
    args.vec_out = (((uintptr_t)p.y & 15) == 0) && p.out_features % 4 == 0;
    hipError_t err;
    switch (p.x_kind) {
        case kF16: err = launch_stage<kF16>(p, staged, rowscale, stream, start); break;
        case kBF16: err = launch_stage<kBF16>(p, staged, rowscale, stream, start); break;
        case kSwiGLU:
            err = launch_kernel(rows_stage_swiglu_kernel,
                                dim3((unsigned)p.rows, (unsigned)((p.in_features / 8 + kSwigluThreads - 1) / kSwigluThreads)),
                                dim3(kSwigluThreads), 0, stream, start, nullptr, p.x, staged, rowscale, (int)p.in_features);
            break;
        default: err = launch_stage<kF32>(p, staged, rowscale, stream, start); break;
    }
    if (err != hipSuccess) return err;
    const bool reduce = pl.splits > 1;
    hipEvent_t gstop = reduce ? nullptr : stop;
    err = two ? launch_planes<2>(args, pl, stream, gstop) : launch_planes<1>(args, pl, stream, gstop);
    if (err != hipSuccess || !reduce) return err;
    return launch_split_reduce(args.partials, p.bias, p.bias_kind, p.y, args.M, args.N, pl.splits, false, args.out_kind, stream, stop);
}

}  // namespace w4g64
