// A word of the prepacked MatMulNBits weight as an operand of the f16 matrix cores: what the kernels for more than one row
// share.
#pragma once

#include <hip/hip_fp16.h>

#include "internal.h"

namespace hipc {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// two f16 values as one word, the first in the low half
__device__ __forceinline__ uint32_t two_halves(__half lo, __half hi) {
    return (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
}

// An f32 row enters as f16 terms of the row times 2^-e, with the e that brings its largest magnitude (given as bits) into
// [2^14, 2^15). 2^-e has to be a normal number: rows whose largest value is below 2^-113, subnormal and zero ones among them,
// are all scaled by 2^127, which their terms hold as well (a subnormal's last bit becomes 2^-22); a row with an infinity is
// scaled like one of the largest finite value.
__device__ __forceinline__ int row_exponent(uint32_t largest) { return min(max((int)(largest >> 23), 14), 254) - 127 - 14; }
__device__ __forceinline__ float two_to_minus(int e) { return __uint_as_float((uint32_t)(127 - e) << 23); }
// Each term is the nearest f16 of what the ones before leave (exactly formed). Of two terms, which hold 22 bits, the second is
// as it comes: of a small value up to 2^-25 is lost where that is more, 2^-39 of a largest value of 2^14. Three stand for every
// bit of the row's values, so the second and third are 2^11 and 2^22 times what they stand for: 2^-47 is lost at most, and 24
// bits are held of values down to 2^-23 -- of 2^-1 were the terms as they come.
constexpr float kTermStep = 0x1p11f;
template <int NT>
__device__ __forceinline__ void split_terms(float x, _Float16 (&t)[NT]) {
    constexpr float step = NT == 3 ? kTermStep : 1.f;
    t[0] = (_Float16)x;
    if constexpr (NT >= 2) {
        // (an infinity leaves infinity minus itself: the maximum makes a number of that, which the infinite first term outweighs.
        // Any other remainder is 8 at most, half a step of f16 below 2^15.)
        const float r = fmaxf(x - (float)t[0], -8.f) * step;
        t[1] = (_Float16)r;
        if constexpr (NT == 3) t[2] = (_Float16)((r - (float)t[1]) * step);
    }
}
__device__ __forceinline__ float join_terms(float d0, float d1, float d2) { return fmaf(fmaf(d2, 1.f / kTermStep, d1), 1.f / kTermStep, d0); }

// 1024 + zp and 64 + zp as f16 in both halves of a word (zb carries 128 + zp)
struct ZeroPair {
    f16x2 unit, sixteenth;
};
// (two multiply-adds of 24-bit numbers: both halves at once)
__device__ __forceinline__ ZeroPair zero_pair(uint32_t zb) {
    const uint32_t a = (uint32_t)__umul24(zb, 0x00010001u) + (0x64006400u - 128u * 0x00010001u), b = (uint32_t)__umul24(zb, 0x00100010u) + (0x54005400u - 128u * 0x00100010u);
    return {__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b)};
}
// eight nibbles (k0 k2 k4 k6 in the low half, k1 k3 k5 k7 in the high half) -> the f16 values q - zp in k order.
// Nibbles 0 and 2 of each half sit where the low mantissa bits are: or-ed with the exponent of 1024 that is
// 1024 + q. Nibbles 1 and 3 sit four bits higher: 1024 + 16 q, and one fused multiply-add by 1/16 makes q - zp
// of it ((1024 + 16 q) / 16 = 64 + q is exact). One shift instead of three.
// (x & mask) | 0x64006400 as one instruction: v_and_or_b32 can take one scalar operand only, so the exponent pattern is handed
// over in a vector register the compiler knows nothing about (HIPC_PIN_VGPR). Not as inline assembly: the wait states a
// matrix product needs before one of its registers is written again are the compiler's to count, and it does not count them
// for an instruction it cannot see.
__device__ __forceinline__ uint32_t and_or_1024(uint32_t x, uint32_t mask, uint32_t ones) { return (x & mask) | ones; }
__device__ __forceinline__ f16x8 dequant_operand(uint32_t w, const ZeroPair &z, uint32_t ones) {
    const f16x2 sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
    const uint32_t w8 = w >> 8;
    const f16x2 p0 = __builtin_bit_cast(f16x2, and_or_1024(w, 0x000f000fu, ones)) - z.unit;
    const f16x2 p1 = __builtin_bit_cast(f16x2, and_or_1024(w, 0x00f000f0u, ones)) * sixteenth - z.sixteenth;
    const f16x2 p2 = __builtin_bit_cast(f16x2, and_or_1024(w8, 0x000f000fu, ones)) - z.unit;
    const f16x2 p3 = __builtin_bit_cast(f16x2, and_or_1024(w8, 0x00f000f0u, ones)) * sixteenth - z.sixteenth;
    return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}
__device__ __forceinline__ uint32_t word_of(const uint4 &v, int j) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; }

}  // namespace hipc
