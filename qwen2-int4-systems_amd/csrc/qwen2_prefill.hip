// Attention over a prompt (the launch side of qwen2_prefill_attention,
// include/qwen2_decode.h; model.py:17-31, :61-122).
//
//   prefill_cache_kernel      rotated keys and values into the caches
//   prefill_attention_kernel  causal grouped-query attention, one workgroup of
//                             4 waves per (sequence, head, 32 query rows)
//
// A wave works on all 32 rows over every fourth 32-key block, alone (no
// barrier between the queries' staging and the end, where the four waves'
// results meet in LDS).  MFMA layout as in qwen2_decode_split.hip, with two
// column tiles of 16 query rows: scores A = 16 keys, B = the rotated queries,
// both read from LDS; values A = the block's values transposed by v_perm, B
// = the lane's own probabilities, so that a probability never moves between
// lanes and the row statistics and the rescaling are the lane's own.
//
// Bound by the vector unit (per 32 x 32 block 48 MFMAs of 16 cycles and about
// 165 vector instructions, 16 of them exponentials) and, a quarter of the
// time at 2048 positions, by the keys' and values' reads from L2 (16 KB per
// wave and block).  Three waves per SIMD (168 registers: the queries stay in
// LDS).  Measured on the way, 12/2 heads at 2048 positions, both launches,
// graph-replayed: 101 us for the previous kernel (64 rows, probabilities
// through LDS, four barriers a block, rotated queries through memory); 51 with
// the keys loaded straight into operands (16 bytes of 16 rows per 16 lanes),
// 42.7 with them through LDS, 41.5 with the lazy rescaling, 36.7 with the
// queries rotated once per workgroup and three waves per SIMD.  At 512
// positions 23.5 -> 13.9 us, 3000 140 -> 65, 4 x 750 55 -> 31, 16 8.6 -> 8.4;
// with the queries in an LDS object of their own (one object shared with the
// keys made every query read wait for the keys in flight) 2048 positions 35.3,
// 512 12.9, 3000 60.9; without the joins of waves that had no block 16
// positions 8.5 -> 7.0, 64 9.0 -> 8.1.
//
// The masked form serves the cached-generation layer (a growing cache, left
// padding): a block's mask is one byte per lane, made a 32-bit word by a
// ballot; blocks without an excluded key or a causal edge take no masking
// instructions.  With the rotary step and the cache's concatenation in the
// first launch it replaced some 30 torch launches: a layer over four prompts
// of up to 300 tokens 401 -> 119 us, of which its four linears took 90 then.
// It replaced fp32 probabilities, so it splits them into three bf16 terms, all
// of their bits (the prompt's form keeps the two of the kernel before it):
// 1.2e-4 of the outputs are then not the exact value's rounding, 1.5e-3 with
// two terms, 1.7e-4 with torch in fp32; the layer 93.0 -> 93.6 us.
#include <math.h>

#include <type_traits>

#include "qwen2_attention.h"

namespace w4g64 {
namespace {

constexpr int kTile = 32;   // query rows per workgroup and keys per block
constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kOutStride = kAttnHeadDim + 4;

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// s_waitcnt with one counter constrained (gfx9 encoding: vmcnt in bits 3:0
// and 15:14, expcnt 6:4, lgkmcnt 11:8); the fences keep the compiler from
// moving LDS accesses across.
__device__ __forceinline__ void wait_vmcnt8() {
    __builtin_amdgcn_s_waitcnt(8 | (0x7 << 4) | (0xF << 8));
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void wait_lgkmcnt0() {
    __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4));
    asm volatile("" ::: "memory");
}

// One thread per 8 dimensions of a key or value head of a position: the cache's
// earlier positions copied (kPast), the new keys rotated, the new values as they are.
template <bool kPast>
__global__ __launch_bounds__(256) void prefill_cache_kernel(PrefillArgs a, int64_t pieces) {
    const int64_t at = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (at >= pieces) return;
    constexpr int kPer = kAttnHeadDim / 8;
    const int d = 8 * (int)(threadIdx.x % kPer);
    const int64_t line = at / kPer;
    const int total = (kPast ? a.past : 0) + a.length;
    const int64_t spot = line / (2 * a.kv_heads);                  // b * total + position
    const int head = (int)(line - spot * 2 * a.kv_heads);          // key heads, then value heads
    const int b = (int)(spot / total);
    const int position = (int)(spot - (int64_t)b * total);
    const bool key = head < a.kv_heads;
    const int64_t slot = (int64_t)b * a.kv_heads + (key ? head : head - a.kv_heads);
    const int64_t to = (slot * a.max_len + position) * kAttnHeadDim + d;
    uint16_t* cache = key ? a.k_cache : a.v_cache;
    if (kPast && position < a.past) {
        const uint16_t* from = key ? a.past_k : a.past_v;
        *(u32x4*)(cache + to) = *(const u32x4*)(from + (slot * a.past + position) * kAttnHeadDim + d);
        return;
    }
    const int64_t row = (int64_t)b * a.length + position - (kPast ? a.past : 0);
    const uint16_t* vec = (key ? a.k : a.v) + row * a.kv_row + (slot - (int64_t)b * a.kv_heads) * kAttnHeadDim;
    if (key)
        *(u32x4*)(cache + to) = rope_piece(vec, a.cos + row * kAttnHeadDim, a.sin + row * kAttnHeadDim, d);
    else
        *(u32x4*)(cache + to) = *(const u32x4*)(vec + d);
}

// The queries of rows q_row apart into rows of their own, 16 bytes per thread.
__global__ __launch_bounds__(256) void prefill_queries_kernel(PrefillArgs a, int64_t pieces) {
    const int64_t at = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (at >= pieces) return;
    const int per = a.heads * (kAttnHeadDim / 8);
    const int64_t row = at / per;
    *(u32x4*)(a.q_copy + 8 * at) = *(const u32x4*)(a.q + row * a.q_row + 8 * (at - row * per));
}

// kMasked: the queries follow `past` cached positions, and a key may be excluded
// for a whole sequence (mask); a row without an allowed key gives zeros.
template <bool kMasked>
__global__ __launch_bounds__(kThreads, 3) void prefill_attention_kernel(PrefillArgs a) {
    // the rotated queries; one block's keys per wave and at the end, in their
    // place, the results of two waves (two objects: a read of the queries then
    // does not wait for the next keys on their way to the other)
    __shared__ __attribute__((aligned(16))) unsigned char queries[kTile * 2 * kAttnHeadDim];
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * kTile * kOutStride * 4];
    static_assert(sizeof(smem) >= kWaves * kTile * 2 * kAttnHeadDim, "a block's keys per wave");
    __shared__ float sm[2][kTile];
    __shared__ float sl[2][kTile];
    __shared__ int sn[2][kTile];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: the block loop branches on it
    const int j = lane & 15;
    const int q = lane >> 4;
    const int tiles = (a.length - 1) / kTile + 1;
    const int heads = a.batch * a.heads;
    const int qt = tiles - 1 - (int)blockIdx.x / heads;  // the longest rows first
    const int head = blockIdx.x % heads % a.heads;
    const int b = blockIdx.x % heads / a.heads;
    const int kvh = head / (a.heads / a.kv_heads);
    const int q0 = qt * kTile;
    const int total = kMasked ? a.past + a.length : a.length;  // keys
    // last block that a row of the tile attends to, and its first position
    const int last = kMasked ? min(a.past + q0 + kTile - 1, total - 1) / kTile : qt;
    const int base = kMasked ? a.past + q0 : q0;
    const int64_t cache = ((int64_t)b * a.kv_heads + kvh) * a.max_len * kAttnHeadDim;
    const uint16_t* kc = a.k_cache + cache;
    const uint16_t* vc = a.v_cache + cache;
    constexpr int kRowBytes = 2 * kAttnHeadDim;

    unsigned char* stage = smem + wave * kTile * kRowBytes;
    u32x4 vf[8];
    // keys and values of a block through a buffer over the rest of the keys (a
    // raw gfx9 buffer: rows past it read zeros, and are masked: key > query)
    auto rest = [&](const uint16_t* rows, int block) {
        const int t0 = block * kTile;
        return __builtin_amdgcn_make_buffer_rsrc((void*)(rows + (int64_t)t0 * kAttnHeadDim), 0,
                                                 min(kTile, total - t0) * kRowBytes, 0x00020000);
    };
    // Keys go to LDS directly, a row's 16 pieces by 16 lanes (operand pieces
    // straight from memory would be 16 bytes of 16 rows per 16 lanes).  Piece
    // c of row r lands in slot c ^ (r % 16): the operand reads, one slot
    // column of 16 rows, meet 16 different bank groups.
    int k_at[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) k_at[s] = (4 * s + q) * kRowBytes + 16 * (j ^ (4 * s + q));
    const int v_at = 4 * q * kRowBytes + 16 * j;
    auto load_k = [&](int block) {
        const __amdgpu_buffer_rsrc_t r = rest(kc, block);
#pragma unroll
        for (int u = 0; u < 8; ++u)  // rows 4 u .. 4 u + 3
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)(stage + 1024 * u), 16, k_at[u % 4],
                                                     16 * kRowBytes * (u / 4), 0, 0);
    };
    auto load_v = [&](int block) {
        const __amdgpu_buffer_rsrc_t r = rest(vc, block);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            vf[e] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, v_at + kRowBytes * (e % 4), 16 * kRowBytes * (e / 4), 0));
    };
    // the block's mask, one key per lane (twice), loaded with its keys
    const uint8_t* mask = kMasked && a.mask ? a.mask + (int64_t)b * total : nullptr;
    auto load_mask = [&](int block) -> int {
        const int t = block * kTile + (lane & 31);
        return t < total ? (mask ? mask[t] : 1) : 0;
    };
    int blk = wave;
    int mv = 0;
    if (blk <= last) {
        if constexpr (kMasked) mv = load_mask(blk);
        load_k(blk);
        load_v(blk);
    }
    // Rotated queries into LDS, slots as the keys': thread t takes piece t % 16
    // of rows t / 16 and t / 16 + 16.  (A negative scale goes into their
    // signs: the largest product is then the largest score.)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int r = tid / 16 + 16 * u;
        const int64_t row = (int64_t)b * a.length + min(q0 + r, a.length - 1);
        const u32x4 x = rope_piece(a.q + row * a.q_row + head * kAttnHeadDim,
                                   a.cos + row * kAttnHeadDim, a.sin + row * kAttnHeadDim, 8 * (tid % 16));
        *(u32x4*)(queries + r * kRowBytes + 16 * ((tid % 16) ^ (r % 16))) = x ^ a.query_sign;
    }
    __syncthreads();
    float m_run[2] = {kScoreFloor, kScoreFloor}, l_run[2] = {0.0f, 0.0f};
    bool seen[2] = {false, false};  // kMasked: the row had an allowed key
    float4v o[8][2];
#pragma unroll
    for (int dd = 0; dd < 8; ++dd)
#pragma unroll
        for (int u = 0; u < 2; ++u) o[dd][u] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    // more: the wave has a block after this one, whose keys and values are
    // loaded as this one's leave their registers
    auto step = [&](auto more) {
        constexpr bool kMore = decltype(more)::value;
        float s[2][8];
        uint32_t word = 0;
        {
            // this block's keys have landed: the 8 value loads came after
            // (the mask before the keys: its arrival is theirs too)
            wait_vmcnt8();
            if constexpr (kMasked) word = (uint32_t)__ballot(mv != 0);
            u32x4 kf[2][4];
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    kf[m][p] = *(const u32x4*)(stage + (16 * m + j) * kRowBytes + 16 * ((4 * p + q) ^ j));
            wait_lgkmcnt0();
            if constexpr (kMore) {
                if constexpr (kMasked) mv = load_mask(blk + kWaves);
                load_k(blk + kWaves);
            }
            float4v acc[2][2];
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int u = 0; u < 2; ++u) acc[m][u] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int p = 0; p < 4; ++p) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const u32x4 qv = *(const u32x4*)(queries + (16 * u + j) * kRowBytes + 16 * ((4 * p + q) ^ j));
#pragma unroll
                    for (int m = 0; m < 2; ++m)
                        acc[m][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8, kf[m][p]), __builtin_bit_cast(bf16x8, qv), acc[m][u], 0, 0, 0);
                }
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int e = 0; e < 8; ++e) s[u][e] = acc[e / 4][u][e % 4];
        }
        if constexpr (kMasked) {
            const int t0 = blk * kTile;
            if (word != 0xFFFFFFFFu || t0 + kTile - 1 > base) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int most = base + 16 * u + j - t0;  // last key the row may attend to
                    const uint32_t causal = most >= 31 ? 0xFFFFFFFFu : (most < 0 ? 0u : (2u << most) - 1u);
                    const uint32_t own = (word & causal) >> (4 * q);  // bits 0..3 and 16..19: the lane's keys
                    seen[u] = seen[u] || (word & causal) != 0;
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (!((own >> (16 * (e / 4) + e % 4)) & 1)) s[u][e] = -INFINITY;
                }
            } else {
                seen[0] = seen[1] = true;
            }
        } else if (!kMore && blk == qt) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (16 * (e / 4) + 4 * q + e % 4 > 16 * u + j) s[u][e] = -INFINITY;
        }
        // online softmax (base 2) of the lane's two query rows
        u32x4 ph[2], pl[2], pt[2];  // probabilities: bf16 hi + lo, kMasked a third term (all 24 bits)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            float bm = s[u][0];
#pragma unroll
            for (int e = 1; e < 8; ++e) bm = fmaxf(bm, s[u][e]);
            // the sums are rescaled only once a score passes their reference
            // by 8 units of the base-2 exponent (from the floor on the first
            // block); until then probabilities reach 2^8, which changes no
            // relative rounding
            const float mn = quarters_max(bm) * a.scale2;
            if (__any(mn - m_run[u] > 8.0f)) {
                const float to = fmaxf(m_run[u], mn);
                const float alpha = __builtin_amdgcn_exp2f(m_run[u] - to);  // (1 where it is another row's turn)
                l_run[u] *= alpha;
#pragma unroll
                for (int dd = 0; dd < 8; ++dd) o[dd][u] *= alpha;
                m_run[u] = to;
            }
            const float ref = -m_run[u];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float p0 = __builtin_amdgcn_exp2f(fmaf(s[u][2 * e], a.scale2, ref));
                const float p1 = __builtin_amdgcn_exp2f(fmaf(s[u][2 * e + 1], a.scale2, ref));
                l_run[u] += p0 + p1;
                ph[u][e] = pack_bf16x2(p0, p1);
                const float r0 = p0 - bf16_lo(ph[u][e]), r1 = p1 - bf16_hi(ph[u][e]);
                pl[u][e] = pack_bf16x2(r0, r1);
                if constexpr (kMasked) pt[u][e] = pack_bf16x2(r0 - bf16_lo(pl[u][e]), r1 - bf16_hi(pl[u][e]));
            }
        }
#pragma unroll
        for (int dd = 0; dd < 8; ++dd) {
            const uint32_t sel = (dd & 1) ? 0x07060302u : 0x05040100u;  // high or low halves
            u32x4 vt;
#pragma unroll
            for (int e = 0; e < 4; ++e) vt[e] = __builtin_amdgcn_perm(vf[2 * e + 1][dd / 2], vf[2 * e][dd / 2], sel);
#pragma unroll
            for (int u = 0; u < 2; ++u)
                o[dd][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vt),
                                                                   __builtin_bit_cast(bf16x8, ph[u]), o[dd][u], 0, 0, 0);
#pragma unroll
            for (int u = 0; u < 2; ++u)
                o[dd][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vt),
                                                                   __builtin_bit_cast(bf16x8, pl[u]), o[dd][u], 0, 0, 0);
            if constexpr (kMasked) {
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    o[dd][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, vt), __builtin_bit_cast(bf16x8, pt[u]), o[dd][u], 0, 0, 0);
            }
        }
        if constexpr (kMore) load_v(blk + kWaves);
    };
    for (; blk + kWaves <= last; blk += kWaves) step(std::true_type{});
    if (blk <= last) step(std::false_type{});

    // ---- the waves' results meet in LDS: waves 2 and 3 give theirs to 0 and
    // 1, then wave 1 to wave 0, which stores the rows; a wave without a block
    // (or an allowed key) adds its sums of zero ----
    float l_all[2] = {quarters_sum(l_run[0]), quarters_sum(l_run[1])};
    float(*so)[kTile][kOutStride] = (float(*)[kTile][kOutStride])smem;
#pragma unroll
    for (int half = 2; half > 0; half /= 2) {
        // No block reached those waves (last is the workgroup's): nothing to
        // add.  Both joins cost a prompt of 16 positions 1.5 of 8.5 us.
        if (last < half) continue;
        __syncthreads();
        if (wave >= half && wave < 2 * half) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float* to = &so[wave - half][16 * u + j][32 * q + 8 * r];
                    *(float4v*)to = float4v{o[0][u][r], o[1][u][r], o[2][u][r], o[3][u][r]};
                    *(float4v*)(to + 4) = float4v{o[4][u][r], o[5][u][r], o[6][u][r], o[7][u][r]};
                }
                if (q == 0) {
                    sm[wave - half][16 * u + j] = m_run[u];
                    sl[wave - half][16 * u + j] = l_all[u];
                    sn[wave - half][16 * u + j] = seen[u];
                }
            }
        }
        __syncthreads();
        if (wave < half) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const float mo = sm[wave][16 * u + j];
                const float to = fmaxf(m_run[u], mo);
                const float f = __builtin_amdgcn_exp2f(m_run[u] - to);
                const float fo = __builtin_amdgcn_exp2f(mo - to);
                m_run[u] = to;
                seen[u] = seen[u] || sn[wave][16 * u + j] != 0;
                l_all[u] = fmaf(sl[wave][16 * u + j], fo, l_all[u] * f);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float* from = &so[wave][16 * u + j][32 * q + 8 * r];
                    const float4v lo = *(const float4v*)from, hi = *(const float4v*)(from + 4);
#pragma unroll
                    for (int dd = 0; dd < 4; ++dd) {
                        o[dd][u][r] = fmaf(lo[dd], fo, o[dd][u][r] * f);
                        o[4 + dd][u][r] = fmaf(hi[dd], fo, o[4 + dd][u][r] * f);
                    }
                }
            }
        }
    }
    if (wave != 0) return;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int i = q0 + 16 * u + j;
        if (i >= a.length) continue;
        const float inv = kMasked && !seen[u] ? 0.0f : 1.0f / l_all[u];
        uint16_t* out = a.out + (((int64_t)b * a.length + i) * a.heads + head) * kAttnHeadDim + 32 * q;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            u32x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = pack_bf16x2(o[2 * e][u][r] * inv, o[2 * e + 1][u][r] * inv);
            *(u32x4_any*)(out + 8 * r) = w;
        }
    }
}

}  // namespace

hipError_t launch_prefill_attention(PrefillArgs args, hipStream_t stream) {
    if (args.q_copy) {
        const int64_t copied = (int64_t)args.batch * args.length * args.heads * (kAttnHeadDim / 8);
        hipLaunchKernelGGL(prefill_queries_kernel, dim3((unsigned)((copied + 255) / 256)), dim3(256), 0, stream, args,
                           copied);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
        args.q = args.q_copy;
        args.q_row = (int64_t)args.heads * kAttnHeadDim;
    }
    const bool masked = args.mask || args.past > 0;
    const int64_t pieces = (int64_t)args.batch * (args.past + args.length) * 2 * args.kv_heads * (kAttnHeadDim / 8);
    const dim3 cgrid((unsigned)((pieces + 255) / 256));
    if (args.past > 0)
        hipLaunchKernelGGL(prefill_cache_kernel<true>, cgrid, dim3(256), 0, stream, args, pieces);
    else
        hipLaunchKernelGGL(prefill_cache_kernel<false>, cgrid, dim3(256), 0, stream, args, pieces);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    const int64_t tiles = ((int64_t)args.length + kTile - 1) / kTile;
    const dim3 grid((unsigned)(tiles * args.batch * args.heads));
    if (masked)
        hipLaunchKernelGGL(prefill_attention_kernel<true>, grid, dim3(kThreads), 0, stream, args);
    else
        hipLaunchKernelGGL(prefill_attention_kernel<false>, grid, dim3(kThreads), 0, stream, args);
    return hipGetLastError();
}

}  // namespace w4g64
