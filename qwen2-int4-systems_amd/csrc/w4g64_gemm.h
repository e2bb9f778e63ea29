// Shared by the GEMM kernels (rows > 16): the staging of activation rows as fp16
// times a power of two, in MFMA slot order, and the decode of packed weights
// into exact fp16 integers.
#pragma once

#include "w4g64_device.h"

namespace w4g64 {

// Word 3 of a raw gfx9 buffer resource (32-bit data format; no swizzle, no stride).
constexpr int kRsrcWord3 = 0x00020000;

// Bitwise select (x ^ C) & M | (C & ~M), one v_bitop3: inside the mask the
// nibble n XOR 8 = n' = code + 8, outside it the magic exponent bits of C.
template <uint32_t C, uint32_t M>
__device__ __forceinline__ uint32_t nib_select(uint32_t x) {
    return ((x ^ C) & M) | (C & ~M);
}
// fp16 pairs (1024 + n', 1024 + n'') from bits 0-3 / 16-19 and (64 + n', 64 +
// n'') from bits 4-7 / 20-23 (n' XOR-ed in by the 8s of C).
constexpr uint32_t kMaskLo = 0x000F000Fu, kSelLo = 0x64086408u;
constexpr uint32_t kMaskHi = 0x00F000F0u, kSelHi = 0x54805480u;

// (code - zero) of one packed dword (8 consecutive K values of a column), as
// 4 fp16 pairs in slot order [k0 k4 | k1 k5 | k2 k6 | k3 k7].  zlo = fp16
// pair (1032 + z, 1032 + z), zhi = (72 + z, 72 + z): (1024 + n') - (1032 + z)
// = (64 + n') - (72 + z) = code - z, exact.
__device__ __forceinline__ u32x4 decode_codes(uint32_t w, half2v zlo, half2v zhi) {
    const uint32_t w8 = w >> 8;
    u32x4 r;
    r[0] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, nib_select<kSelLo, kMaskLo>(w)) - zlo);
    r[1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, nib_select<kSelHi, kMaskHi>(w)) - zhi);
    r[2] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, nib_select<kSelLo, kMaskLo>(w8)) - zlo);
    r[3] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, nib_select<kSelHi, kMaskHi>(w8)) - zhi);
    return r;
}

template <int XK>
__device__ __forceinline__ void stage_load8(const void* x, int64_t m, int K, int c, float (&v)[8]) {
    if constexpr (XK == kF16 || XK == kBF16) {
        const u32x4 d = *(const u32x4*)((const uint16_t*)x + m * K + 8 * c);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t bits = (d[i / 2] >> (16 * (i & 1))) & 0xFFFFu;
            v[i] = XK == kF16 ? half_bits_to_float((uint16_t)bits) : bf16_bits_to_float(bits);
        }
    } else if constexpr (XK == kF32) {
        const float4v f0 = *(const float4v*)((const float*)x + m * K + 8 * c);
        const float4v f1 = *(const float4v*)((const float*)x + m * K + 8 * c + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = f0[i];
            v[4 + i] = f1[i];
        }
    } else {
        const uint16_t* gu = (const uint16_t*)x + m * 2 * K + 8 * c;
        const u32x4 gv = *(const u32x4*)gu;
        const u32x4 uv = *(const u32x4*)(gu + K);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float gf = bf16_bits_to_float((gv[i / 2] >> (16 * (i & 1))) & 0xFFFFu);
            const float uf = bf16_bits_to_float((uv[i / 2] >> (16 * (i & 1))) & 0xFFFFu);
            v[i] = (gf / (1.0f + expf(-gf))) * uf;
        }
    }
}

// Scale 2^-e for a row whose largest finite magnitude is mx (e = 0 for 0).
__device__ __forceinline__ void row_factors(float mx, float& inv, float& rs) {
    inv = 1.0f;
    rs = 1.0f;
    if (mx > 0.0f) {
        int ex;
        (void)frexpf(mx, &ex);  // mx = f 2^ex, f in [0.5, 1)
        int sh = 15 - ex;       // mx 2^sh in [2^14, 2^15)
        sh = sh > 126 ? 126 : sh;
        inv = ldexpf(1.0f, sh);
        rs = ldexpf(1.0f, -sh);
    }
}

// 8 values times inv as fp16 hi and lo (lo = RNE of the rest), in slot order.
__device__ __forceinline__ void stage_split8(const float (&v)[8], float inv, u32x4& hi, u32x4& lo) {
    constexpr int kSlot[8] = {0, 4, 1, 5, 2, 6, 3, 7};
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        uint32_t hb[2], lb[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float t = v[kSlot[2 * p + h]] * inv;
            const _Float16 th = (_Float16)t;
            hb[h] = __builtin_bit_cast(uint16_t, th);
            // (an infinite hi keeps a zero lo: inf - inf would turn the row's results into NaN)
            lb[h] = __builtin_isfinite((float)th) ? __builtin_bit_cast(uint16_t, (_Float16)(t - (float)th)) : 0;
        }
        hi[p] = hb[0] | (hb[1] << 16);
        lo[p] = lb[0] | (lb[1] << 16);
    }
}

}  // namespace w4g64
