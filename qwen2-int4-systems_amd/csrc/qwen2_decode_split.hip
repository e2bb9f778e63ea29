// Decode attention with the context split over workgroups (the launch side of
// qwen2_decode_attention, include/qwen2_decode.h, for batches and contexts
// past what one 64-position workgroup per chunk serves well).
//
//   decode_split_kernel  one workgroup of 4 independent waves per (sequence,
//                        key/value head, split).  The context's 32-position
//                        blocks are dealt round robin to the splits, then to
//                        their waves.  A wave works on its blocks alone, in
//                        registers: no LDS and no barrier until the end.
//   decode_merge_kernel  one workgroup per (sequence, query head): adds the
//                        splits' partial results.
//
// MFMA layout (v_mfma_f32_16x16x32_bf16; lane l = 16 q + j supplies A row j
// and B column j with the values of K slots [8 q, 8 q + 8), and receives
// D[4 q + r][j], r < 4):
//   scores  A = 16 keys, loaded from the cache in this form (16 bytes of key
//           row j per lane), B = the rotated query heads: lane (j, q) gets
//           head j's scores of keys 4 q + r of each 16-key tile.
//   values  a key's place among the K slots is free as long as both operands
//           agree, so the lane's own 8 scores (2 tiles x 4) are its 8 slots
//           of B as they are.  The A operand is the values transposed: lane
//           (j, q) loads dimensions 8 j .. 8 j + 7 of its 8 keys (256
//           contiguous bytes per key and 16 lanes) and pairs them up by
//           v_perm, 4 dwords per dimension; dimension 8 j + dd is row j of
//           the dd-th product.  Lane (j, q) then holds dimensions 32 q + 8 r
//           + dd of head j, so the softmax rescaling is a multiplication by
//           the lane's own factor.
//
// Bound by the cache's read for long contexts, by its chain of round trips
// (position, keys, launch of the merge) for short ones.  Two blocks (32 KB) in
// flight per wave, at most two waves per SIMD (217 registers, no spills; with
// the last block's code in both halves of the loop 42 registers spilled and
// 24 x 1024 positions took 10.5-12.6 us).  Graph-replayed, per call, against
// the one-workgroup-per-chunk kernel with its arrival counters: 8 sequences at
// position 3900 of 4096, 12/2 heads, 51.1 -> 12.7 us (2.5 TB/s); 4 at 2000
// of 2048, 16/16 heads, 93 -> 20.5 (6.4 of a 4.9 TB/s copy's reads, part of
// them in the Infinity Cache); 24 at 700 of 1024 28.0 -> 11.7; 32 at 40 of 64
// 8.4 -> 5.3 (one split: no merge launch).
#include <math.h>

#include <type_traits>

#include "qwen2_attention.h"

namespace w4g64 {
namespace {

constexpr int kSplitWaves = 4;
constexpr int kSplitThreads = 64 * kSplitWaves;
constexpr int kSplitBlock = 32;  // positions per block
constexpr int kOutStride = kAttnHeadDim + 4;

struct Kv {
    u32x4 k[2][4];  // key tile t, dimensions 32 sl + 8 q ..: 16-byte pieces
    u32x4 v[8];     // value of key 16 (e / 4) + 4 q + e % 4, dimensions 8 j ..
};

__global__ __launch_bounds__(kSplitThreads, 2) void decode_split_kernel(DecodeSplitArgs a) {
    __shared__ __attribute__((aligned(16))) float so[kSplitWaves][kAttnMaxGroup][kOutStride];
    __shared__ float sm[kSplitWaves][kAttnMaxGroup];
    __shared__ float sl[kSplitWaves][kAttnMaxGroup];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: the block loop branches on it
    const int j = lane & 15;
    const int q = lane >> 4;
    const int split = blockIdx.x % a.splits;
    const int slot = blockIdx.x / a.splits;  // b * kv_heads + kvh
    const int kvh = slot % a.kv_heads;
    const int b = slot / a.kv_heads;
    const int group = a.heads / a.kv_heads;

    int64_t p64 = *a.position;
    p64 = p64 < 0 ? 0 : (p64 >= a.max_len ? a.max_len - 1 : p64);
    const int pos = (int)p64;
    const int blocks = pos / kSplitBlock + 1;
    if (split >= blocks) return;  // the merge does not read this split

    const uint16_t* qkv = a.qkv + (int64_t)b * (a.heads + 2 * a.kv_heads) * kAttnHeadDim;
    const uint16_t* cs = a.cos + (int64_t)b * kAttnHeadDim;
    const uint16_t* sn = a.sin + (int64_t)b * kAttnHeadDim;
    uint16_t* kc = a.k_cache + (int64_t)slot * a.max_len * kAttnHeadDim;
    uint16_t* vc = a.v_cache + (int64_t)slot * a.max_len * kAttnHeadDim;

    // block of wave w, step i: split + splits (w + 4 i)
    int blk = split + a.splits * wave;
    const int stride = a.splits * kSplitWaves;
    // (byte offsets from the uniform bases: at most 17408 rows of 256 bytes;
    // only the last block can reach past the cache's end, its rows are clamped)
    constexpr uint32_t kRowBytes = 2 * kAttnHeadDim;
    auto load = [&](Kv& t, int block) {
        const int t0 = block * kSplitBlock;
        if (block == blocks - 1) {
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const uint32_t at = (uint32_t)min(t0 + 16 * m + j, a.max_len - 1) * kRowBytes + 16 * q;
#pragma unroll
                for (int s = 0; s < 4; ++s) t.k[m][s] = *(const u32x4*)((const char*)kc + (at + 64 * s));
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t at = (uint32_t)min(t0 + 16 * (e / 4) + 4 * q + e % 4, a.max_len - 1) * kRowBytes + 16 * j;
                t.v[e] = *(const u32x4*)((const char*)vc + at);
            }
            return;
        }
        const uint32_t ak = (uint32_t)(t0 + j) * kRowBytes + 16 * q;
        const uint32_t av = (uint32_t)(t0 + 4 * q) * kRowBytes + 16 * j;
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                t.k[m][s] = *(const u32x4*)((const char*)kc + (ak + 16 * kRowBytes * m) + 64 * s);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            t.v[e] = *(const u32x4*)((const char*)vc + (av + 16 * kRowBytes * (e / 4)) + kRowBytes * (e % 4));
    };
    Kv buf[2];
    if (blk < blocks) load(buf[0], blk);

    u32x4 qf[4];  // columns past the group repeat its last head and are not stored
    rope_pieces(qkv + (kvh * group + min(j, group - 1)) * kAttnHeadDim, cs, sn, q, qf);

    float m_run = kScoreFloor, l_run = 0.0f;
    float4v o[8];
#pragma unroll
    for (int dd = 0; dd < 8; ++dd) o[dd] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    // ends: the context's last block, which holds the new position
    auto compute = [&](Kv& t, int block, auto ends) {
        constexpr bool kLast = decltype(ends)::value;
        const int t0 = block * kSplitBlock;
        if constexpr (kLast) {
            const u32x4 vnew = *(const u32x4*)(qkv + (a.heads + a.kv_heads + kvh) * kAttnHeadDim + 8 * j);
            const u32x4 zero = {0u, 0u, 0u, 0u};
            u32x4 kf[4];
            rope_pieces(qkv + (a.heads + kvh) * kAttnHeadDim, cs, sn, q, kf);
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const bool here = t0 + 16 * m + j == pos;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    if (here) {
                        t.k[m][s] = kf[s];
                        *(u32x4*)(kc + (int64_t)pos * kAttnHeadDim + 32 * s + 8 * q) = kf[s];
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int key = t0 + 16 * (e / 4) + 4 * q + e % 4;
                if (key == pos) *(u32x4*)(vc + (int64_t)pos * kAttnHeadDim + 8 * j) = vnew;
                t.v[e] = key < pos ? t.v[e] : (key == pos ? vnew : zero);
            }
        }
        float s[8];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            float4v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int u = 0; u < 4; ++u)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, t.k[m][u]),
                                                              __builtin_bit_cast(bf16x8, qf[u]), acc, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) s[4 * m + r] = acc[r] * a.scale2;
        }
        if constexpr (kLast) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (t0 + 16 * (e / 4) + 4 * q + e % 4 > pos) s[e] = -INFINITY;
        }
        float bm = s[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) bm = fmaxf(bm, s[e]);
        const float mn = fmaxf(m_run, quarters_max(bm));
        if (__any(mn != m_run)) {
            const float alpha = __builtin_amdgcn_exp2f(m_run - mn);
            l_run *= alpha;
#pragma unroll
            for (int dd = 0; dd < 8; ++dd) o[dd] *= alpha;
            m_run = mn;
        }
        // probabilities, split into bf16 hi + lo
        u32x4 ph, pl;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float p0 = __builtin_amdgcn_exp2f(s[2 * e] - mn), p1 = __builtin_amdgcn_exp2f(s[2 * e + 1] - mn);
            l_run += p0 + p1;
            ph[e] = pack_bf16x2(p0, p1);
            pl[e] = pack_bf16x2(p0 - bf16_lo(ph[e]), p1 - bf16_hi(ph[e]));
        }
#pragma unroll
        for (int dd = 0; dd < 8; ++dd) {
            const uint32_t sel = (dd & 1) ? 0x07060302u : 0x05040100u;  // high or low halves
            u32x4 vt;
#pragma unroll
            for (int e = 0; e < 4; ++e) vt[e] = __builtin_amdgcn_perm(t.v[2 * e + 1][dd / 2], t.v[2 * e][dd / 2], sel);
            o[dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vt),
                                                            __builtin_bit_cast(bf16x8, ph), o[dd], 0, 0, 0);
            o[dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vt),
                                                            __builtin_bit_cast(bf16x8, pl), o[dd], 0, 0, 0);
        }
    };
    // two blocks in flight: the next one's loads are issued before this one's products
    const int full = blocks - 1;
    while (blk < full) {
        if (blk + stride < blocks) load(buf[1], blk + stride);
        compute(buf[0], blk, std::false_type{});
        blk += stride;
        if (blk >= full) {
            buf[0] = buf[1];
            break;
        }
        if (blk + stride < blocks) load(buf[0], blk + stride);
        compute(buf[1], blk, std::false_type{});
        blk += stride;
    }
    if (blk == full) compute(buf[0], blk, std::true_type{});

    // ---- the waves' results meet in LDS ----
    const float l_all = quarters_sum(l_run);
    if (j < group) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            *(float4v*)&so[wave][j][32 * q + 8 * r] = float4v{o[0][r], o[1][r], o[2][r], o[3][r]};
            *(float4v*)&so[wave][j][32 * q + 8 * r + 4] = float4v{o[4][r], o[5][r], o[6][r], o[7][r]};
        }
        if (q == 0) {
            sm[wave][j] = m_run;
            sl[wave][j] = l_all;
        }
    }
    __syncthreads();
    // thread t: head t / 32, dimensions 4 (t % 32) .. + 3.  A wave without a
    // block, or a finite score, adds its sums of zero.
    const int g = tid / 32;
    const int d4 = 4 * (tid % 32);
    if (g >= group) return;
    float m = sm[0][g];
#pragma unroll
    for (int w = 1; w < kSplitWaves; ++w) m = fmaxf(m, sm[w][g]);
    float4v sum = {0.0f, 0.0f, 0.0f, 0.0f};
    float l = 0.0f;
#pragma unroll
    for (int w = 0; w < kSplitWaves; ++w) {
        const float f = __builtin_amdgcn_exp2f(sm[w][g] - m);
        l = fmaf(sl[w][g], f, l);
        const float4v ow = *(const float4v*)&so[w][g][d4];
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] = fmaf(ow[i], f, sum[i]);
    }
    if (a.splits == 1) {
        const float inv = 1.0f / l;
        *(u32x2*)(a.out + (int64_t)b * a.heads * kAttnHeadDim + (kvh * group + g) * kAttnHeadDim + d4) =
            u32x2{pack_bf16x2(sum[0] * inv, sum[1] * inv), pack_bf16x2(sum[2] * inv, sum[3] * inv)};
        return;
    }
    float* part = a.partials + ((int64_t)slot * a.splits + split) * kAttnPartFloats;
    *(float4v*)(part + 2 * kAttnMaxGroup + g * kAttnHeadDim + d4) = sum;
    if (d4 == 0) {
        part[g] = m;
        part[kAttnMaxGroup + g] = l;
    }
}

// One workgroup per (sequence, query head): thread t adds dimensions 4 (t %
// 32) .. + 3 of the splits t / 32, t / 32 + 8, ...; the eight sums meet in
// LDS.  Every load is issued before the position arrives; splits without a
// block (never written) are masked out.
__global__ __launch_bounds__(256) void decode_merge_kernel(DecodeSplitArgs a) {
    __shared__ __attribute__((aligned(16))) float so[8][kAttnHeadDim];
    constexpr int kPer = kDecodeMaxSplits / 8;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int u = tid / 32;
    const int d4 = 4 * (tid % 32);
    const int head = blockIdx.x % a.heads;
    const int b = blockIdx.x / a.heads;
    const int group = a.heads / a.kv_heads;
    const int g = head % group;
    const float* base = a.partials + (int64_t)(b * a.kv_heads + head / group) * a.splits * kAttnPartFloats;
    const float* own = base + (int64_t)min(lane, a.splits - 1) * kAttnPartFloats;
    float mc = own[g], lc = own[kAttnMaxGroup + g];
    float4v v[kPer];
    float mv[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        if (8 * i >= a.splits) break;
        const float* part = base + (int64_t)min(u + 8 * i, a.splits - 1) * kAttnPartFloats;
        v[i] = *(const float4v*)(part + 2 * kAttnMaxGroup + g * kAttnHeadDim + d4);
        mv[i] = part[g];
    }
    int64_t p64 = *a.position;
    p64 = p64 < 0 ? 0 : (p64 >= a.max_len ? a.max_len - 1 : p64);
    const int used = min(a.splits, (int)p64 / kSplitBlock + 1);
    mc = lane < used ? mc : -INFINITY;
    const float m = wave_max64(mc);
    const float l = wave_sum64(lane < used ? lc * __builtin_amdgcn_exp2f(mc - m) : 0.0f);
    float4v sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        if (8 * i >= a.splits) break;
        if (u + 8 * i >= used) continue;
        const float f = __builtin_amdgcn_exp2f(mv[i] - m);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] = fmaf(v[i][e], f, sum[e]);
    }
    *(float4v*)&so[u][d4] = sum;
    __syncthreads();
    if (tid >= 32) return;
    float4v t = *(const float4v*)&so[0][d4];
#pragma unroll
    for (int w = 1; w < 8; ++w) t += *(const float4v*)&so[w][d4];
    const float inv = 1.0f / l;
    *(u32x2*)(a.out + (int64_t)b * a.heads * kAttnHeadDim + head * kAttnHeadDim + d4) =
        u32x2{pack_bf16x2(t[0] * inv, t[1] * inv), pack_bf16x2(t[2] * inv, t[3] * inv)};
}

}  // namespace

// Splits per (sequence, key/value head): enough for one workgroup per CU,
// but no more than one 32-position block per wave of a full cache (128
// positions a workgroup).  With 512 workgroups and 128 / 256 / 384 positions,
// 24 x 1024 measured 11.2 / 10.9 / 10.9 us, 8 x 4096 13.5 / 12.7 / 13.2 and 4
// x 2048 of 16 heads 20.0 / 20.0 / 20.2; with 256 workgroups 11.7 / 10.8 /
// 10.9, 12.7 / 12.7 / 13.2 and 20.5 each; 8 x 640 9.2 / 9.8 / 10.6 and one
// sequence of 4096 8.1 / 8.6 / 9.6 with either.
int decode_splits(int64_t batch, int64_t kv_heads, int64_t max_length) {
    const int64_t slots = batch * kv_heads;
    const int64_t most = (max_length + 127) / 128;  // (the workspace holds twice as many partial results)
    int64_t splits = (256 + slots - 1) / slots;
    splits = splits < most ? splits : most;
    return (int)(splits < kDecodeMaxSplits ? splits : kDecodeMaxSplits);
}

hipError_t launch_decode_split(const DecodeSplitArgs& args, int64_t batch, hipStream_t stream) {
    hipLaunchKernelGGL(decode_split_kernel, dim3((unsigned)(batch * args.kv_heads * args.splits)), dim3(kSplitThreads),
                       0, stream, args);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess || args.splits == 1) return err;
    hipLaunchKernelGGL(decode_merge_kernel, dim3((unsigned)(batch * args.heads)), dim3(256), 0, stream, args);
    return hipGetLastError();
}

}  // namespace w4g64
