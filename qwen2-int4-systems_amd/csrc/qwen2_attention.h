// Device-side helpers of the register-resident attention kernels (decode
// split, prompt): lane l = 16 q + j of a wave holds column j (a query) of the
// score products and, with lanes j + 16, j + 32 and j + 48, its keys.
#pragma once

#include "w4g64_device.h"
#include "w4g64_internal.h"

namespace w4g64 {

// Where a softmax's running maximum starts: finite, so that a row whose keys so
// far all scored -inf (masked, or their products overflowed) adds exp2(-inf) =
// 0 to its sums, not exp2(-inf + inf), and below every finite score.
constexpr float kScoreFloor = -3.402823466e+38f;

// Maximum / sum over the four lanes j, j + 16, j + 32, j + 48.  (The swapped
// pair is bit cast as a whole: a bit cast of one element of the builtin's
// integer pair compiles to element 0 with this compiler.)
__device__ __forceinline__ float2v swap16(float v) {
    const uint32_t a = __builtin_bit_cast(uint32_t, v);
    return __builtin_bit_cast(float2v, __builtin_amdgcn_permlane16_swap(a, a, false, false));
}
__device__ __forceinline__ float2v swap32(float v) {
    const uint32_t a = __builtin_bit_cast(uint32_t, v);
    return __builtin_bit_cast(float2v, __builtin_amdgcn_permlane32_swap(a, a, false, false));
}
__device__ __forceinline__ float quarters_max(float v) {
    const float2v r = swap16(v);
    const float2v s = swap32(fmaxf(r[0], r[1]));
    return fmaxf(s[0], s[1]);
}
__device__ __forceinline__ float quarters_sum(float v) {
    const float2v r = swap16(v);
    const float2v s = swap32(r[0] + r[1]);
    return s[0] + s[1];
}

// 16 bytes at an address that need only be a bf16's (the rotary factors and
// prompt outputs of a caller): one access, the target takes unaligned ones.
typedef u32x4 u32x4_any __attribute__((aligned(2)));

// Dimensions d .. d + 7 (d % 8 == 0) of a head vector rotated by its
// position's factors: x * cos + rotate_half(x) * sin, each product and the sum
// rounded to bf16 (model.py:17-19, :76-77).
__device__ __forceinline__ u32x4 rope8(const u32x4& x, const u32x4& partner, const u32x4& c, const u32x4& n,
                                       float sign) {
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t pa = pack_bf16x2(bf16_lo(x[e]) * bf16_lo(c[e]), bf16_hi(x[e]) * bf16_hi(c[e]));
        const uint32_t pb = pack_bf16x2((sign * bf16_lo(partner[e])) * bf16_lo(n[e]),
                                        (sign * bf16_hi(partner[e])) * bf16_hi(n[e]));
        r[e] = pack_bf16x2(bf16_lo(pa) + bf16_lo(pb), bf16_hi(pa) + bf16_hi(pb));
    }
    return r;
}
__device__ __forceinline__ u32x4 rope_piece(const uint16_t* vec, const uint16_t* cs, const uint16_t* sn, int d) {
    const u32x4 c = *(const u32x4_any*)(cs + d), n = *(const u32x4_any*)(sn + d);
    return rope8(*(const u32x4*)(vec + d), *(const u32x4*)(vec + (d ^ (kAttnHeadDim / 2))), c, n,
                 d < kAttnHeadDim / 2 ? -1.0f : 1.0f);
}

// The whole vector as MFMA operand pieces: dimensions 32 s + 8 q .. + 7, whose
// rotate_half partners are piece s ^ 2 of the same lane.
__device__ __forceinline__ void rope_pieces(const uint16_t* vec, const uint16_t* cs, const uint16_t* sn, int q,
                                            u32x4 (&r)[4]) {
    u32x4 x[4], c[4], n[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        x[s] = *(const u32x4*)(vec + 32 * s + 8 * q);
        c[s] = *(const u32x4_any*)(cs + 32 * s + 8 * q);
        n[s] = *(const u32x4_any*)(sn + 32 * s + 8 * q);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) r[s] = rope8(x[s], x[s ^ 2], c[s], n[s], s < 2 ? -1.0f : 1.0f);
}

}  // namespace w4g64
