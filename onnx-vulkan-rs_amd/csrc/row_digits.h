// A row of a product as whole numbers: the values of a chunk (32 of the row) in steps of 2^-29 to 2^-30 of the largest, each as
// four signed bytes ("digits", the lowest first in a word) that int8 matrix instructions multiply exactly.
//
// What that loses: a value of the chunk is off by half a step at most, 2^-30 of the largest, so a product whose weights are codes
// q of 0 .. 15 about a zero point z by at most 32 * 15 * 2^-30 = 2^-21 of the largest times the scale, whatever the weights. The
// form before this one, two bf16 terms a value, keeps every value to 2^-17 of itself, but multiplies by codes of 128 + q and adds in f32:
// a value is rounded with its chunk's sum, 2^-24 of 128 times the largest, even where its own weight is zero.
// Logits against 64 bits where one value of a product's row is 2^16 times the others and its weights are zero (two layers of 448 / 1088;
// q|k|v, o, gate|up, down): two bf16 terms 2.4e-4 6.0e-5 2.5e-4 4.1e-3, three bytes (23 bits, sums of unrounded values) 8.5e-5 3.0e-5 5.8e-5
// 8.7e-4, four bytes 2.8e-6 each, what the unembedding leaves; of even rows 2.5 to 3.3e-6 with all of them.
#pragma once
#include <cstdint>

#include <hip/hip_runtime.h>

namespace hipc {

constexpr uint32_t kDigitsMin = 29;   // a smaller exponent counts as this one: the scale stays finite, steps of 2^-127

// the chunk's exponent, from the largest of its values' bits without the sign (a NaN's are above an infinity's)
__host__ __device__ __forceinline__ uint32_t digits_exponent(uint32_t bits) {
    const uint32_t ex = bits >> 23;
    return ex > kDigitsMin ? ex : kDigitsMin;
}
// what values are multiplied by: the largest comes to 2^29 .. 2^30, so its highest byte does not overflow
__host__ __device__ __forceinline__ float digits_scale(uint32_t ex) { return __builtin_bit_cast(float, (283u - ex) << 23); }
// what digits_join()'s 1 stands for; NaN where an infinity or a NaN, which has no digits, is among the values
__host__ __device__ __forceinline__ float digits_unit(uint32_t ex) { return __builtin_bit_cast(float, ex == 255u ? 0x7fc00000u : (ex - 13u) << 23); }

// the digits of a scaled value: 0x80 added to each byte and taken away without borrowing
__host__ __device__ __forceinline__ uint32_t digits_of(float scaled) {
    return ((uint32_t)(int32_t)__builtin_rintf(scaled) + 0x80808080u) ^ 0x80808080u;
}
// sums over a chunk of (q - z) times the upper and times the lower two digits, as one number in units of 2^16 steps. (Each is below
// 2^24 and exact, and so is the result where the upper one is zero.)
__host__ __device__ __forceinline__ float digits_join(int upper, int lower) { return __builtin_fmaf((float)lower, 1.52587890625e-5f, (float)upper); }

}  // namespace hipc
