// What the one-row kernel (gemv_lean.hip) and the resident decode kernel (decode_resident.hip) share: buffer loads with
// scalar offsets, the scales of a weight tile, activations as bf16 terms. AUX: the cache policy bits of a load (0 ordinary).
#pragma once

#include "internal.h"

namespace hipc {

typedef __attribute__((ext_vector_type(4))) float lf32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 lbf16x8;

// scales and (128 + zero point) bytes of one 16-column x 128-k tile column: SG groups, by buffer load
// (v_sc / v_zb: the lane's byte offsets inside a tile's scale and zero-point blocks; tl: the tile, scalar)
template <int SG>
struct ScaleVecLean;
template <>
struct ScaleVecLean<4> {
    float s[4];
    uint32_t z;
    template <int AUX = 0>
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t sc, __amdgpu_buffer_rsrc_t zb, uint32_t v_sc, uint32_t v_zb, uint32_t tl) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(sc, (int)v_sc, (int)(tl * 256u), AUX);
        s[0] = __uint_as_float(v[0]), s[1] = __uint_as_float(v[1]), s[2] = __uint_as_float(v[2]), s[3] = __uint_as_float(v[3]);
        z = __builtin_amdgcn_raw_buffer_load_b32(zb, (int)v_zb, (int)(tl * 64u), AUX);
    }
};
template <>
struct ScaleVecLean<2> {
    float s[2];
    uint32_t z;
    template <int AUX = 0>
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t sc, __amdgpu_buffer_rsrc_t zb, uint32_t v_sc, uint32_t v_zb, uint32_t tl) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(sc, (int)v_sc, (int)(tl * 128u), AUX);
        s[0] = __uint_as_float(v[0]), s[1] = __uint_as_float(v[1]);
        z = __builtin_amdgcn_raw_buffer_load_b16(zb, (int)v_zb, (int)(tl * 32u), AUX);
    }
};
template <>
struct ScaleVecLean<1> {
    float s[1];
    uint32_t z;
    template <int AUX = 0>
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t sc, __amdgpu_buffer_rsrc_t zb, uint32_t v_sc, uint32_t v_zb, uint32_t tl) {
        s[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(sc, (int)v_sc, (int)(tl * 64u), AUX));
        z = __builtin_amdgcn_raw_buffer_load_b8(zb, (int)v_zb, (int)(tl * 16u), AUX);
    }
};

__device__ __forceinline__ float lean_gelu_tanh(float v) {
    return 0.5f * v * (1.f + tanhf(0.79788456080286536f * fmaf(0.044715f, v * v * v, v)));
}

// ---- buffer loads: a uniform descriptor, a per-lane byte offset computed once and a SCALAR offset per
// load, so that asking for a tile, a partial row or a context chunk costs the vector unit nothing;
// a load whose per-lane offset lies past the end of the descriptor's range returns zeros (no clamping,
// no zero filling); the scalar offset is NOT part of that check and must stay inside the buffer
typedef unsigned int lu32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t lean_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}
template <int AUX = 0>
__device__ __forceinline__ uint4 lean_ld16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, AUX));
}
__device__ __forceinline__ void lean_ld8f(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, float (&o)[8]) {
    const uint4 a = lean_ld16(r, voff, soff), b = lean_ld16(r, voff + 16u, soff);
    o[0] = __uint_as_float(a.x), o[1] = __uint_as_float(a.y), o[2] = __uint_as_float(a.z), o[3] = __uint_as_float(a.w);
    o[4] = __uint_as_float(b.x), o[5] = __uint_as_float(b.y), o[6] = __uint_as_float(b.z), o[7] = __uint_as_float(b.w);
}

// eight consecutive values -> NT operands of eight bf16 each: the nearest bf16 of the value, of the
// remainder, of the second remainder (every remainder is exact in f32)
typedef __attribute__((ext_vector_type(2))) __bf16 lbf16x2;
typedef __attribute__((ext_vector_type(2))) float lf32x2;
// The sum of the two bf16 halves of every word of NT operands (f32): what a product of the operands with ones
// would give, on the vector unit (one v_dot2c_f32_bf16 per word).
typedef __attribute__((ext_vector_type(2))) __bf16 lbf16pair;
template <int NT>
__device__ __forceinline__ float lean_term_sum(const uint4 (&op)[3]) {
    const lbf16pair ones = __builtin_bit_cast(lbf16pair, 0x3f803f80u);
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        s0 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(lbf16pair, op[t].x), ones, s0, false);
        s1 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(lbf16pair, op[t].y), ones, s1, false);
        s0 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(lbf16pair, op[t].z), ones, s0, false);
        s1 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(lbf16pair, op[t].w), ones, s1, false);
    }
    return s0 + s1;
}
template <int NT>
__device__ __forceinline__ void lean_split8(const float (&av)[8], uint4 (&op)[3]) {
    uint32_t w[3][4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        float r0 = av[2 * q], r1 = av[2 * q + 1];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const uint32_t pk = __builtin_bit_cast(uint32_t, __builtin_convertvector(lf32x2{r0, r1}, lbf16x2));
            w[t][q] = pk;
            if (t + 1 < NT) r0 -= __uint_as_float(pk << 16), r1 -= __uint_as_float(pk & 0xffff0000u);
        }
    }
#pragma unroll
    for (int t = 0; t < NT; t++) op[t] = make_uint4(w[t][0], w[t][1], w[t][2], w[t][3]);
}
// one value -> its NT bf16 terms (16 bits each)
template <int NT>
__device__ __forceinline__ void lean_split1(float v, uint16_t (&t)[3]) {
    float r = v;
#pragma unroll
    for (int e = 0; e < NT; e++) {
        const uint32_t pk = __builtin_bit_cast(uint32_t, __builtin_convertvector(lf32x2{r, 0.f}, lbf16x2));
        t[e] = (uint16_t)pk;
        if (e + 1 < NT) r -= __uint_as_float(pk << 16);
    }
}

}  // namespace hipc
