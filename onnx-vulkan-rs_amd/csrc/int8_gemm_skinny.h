// The int8 matrix product for a few rows of A (MatMulInteger / QLinearMatMul, 16-byte aligned rows, up to 64 of them): a
// stream's chunk, a decoded token, a classifier's head.
//
// What such a product has to move is the weight, and what it waited for on the 64x64 tiles was being few: 1024 columns
// are 16 tiles, sixteen CUs reading a whole column range each, with their prologues, stages and barriers in a row. Here a
// workgroup owns 16 or 32 columns -- 64 to 256 workgroups for the usual widths -- and its 4 to 16 wavefronts share out k:
// each asks for everything it will multiply at once (up to four 64-k steps in flight), both operands straight into the
// operand registers of v_mfma_i32_16x16x64_i8 -- the fragment-major weight in 256-byte runs, A's rows in 64-byte pieces
// -- and the partial sums meet in LDS. No stages, one barrier. Rows are taken 16 at a time (RB blocks to a workgroup, and
// as many workgroups along the rows as it takes), so one row costs a quarter of what the 64x64 tile's A costs in load instructions.
//
// Measured (whole call, before -> after): see launch_mm_skinny.
#pragma once

#include "int8_gemm.h"

namespace hipc {

constexpr int kSkinnyRows = 64;    // rows of A it takes
constexpr int kSkinnyAhead = 4;    // 64-k steps a wavefront has in flight
constexpr size_t skinny_lds(int waves, int rb, int cb) { return (size_t)waves * (rb * cb * 256 + rb * 16) * sizeof(int); }

// RB: blocks of 16 rows, CB: blocks of 16 columns. blockDim.x / 64 wavefronts, a multiple of CB.
template <int EPI, bool DYN, int RB, int CB>
__global__ void __launch_bounds__(1024) int8_gemm_skinny_kernel(const GemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
    const int i16 = lane & 15, kg = lane >> 4;
    i32x4 *red = reinterpret_cast<i32x4 *>(lds_raw);   // [wavefronts][RB][CB][64]: a lane's four rows of its column
    int *lds_sum = reinterpret_cast<int *>(red + waves * (RB * CB * 64));   // [wavefronts][16 RB]
    const int j0 = blockIdx.x * 16 * CB, i0 = blockIdx.y * 16 * RB;
    const int steps = p.K_pad / 64;

    const __amdgpu_buffer_rsrc_t rsrc_p = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(p.P), 0, (int)((uint32_t)p.I * (uint32_t)p.lda), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_q = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(p.Q), 0, (int)((uint32_t)((p.J + kBN - 1) / kBN * kBN) * (uint32_t)p.K_pad), 0x00020000);
    uint32_t a_row[RB], q_off[CB];
#pragma unroll
    for (int i = 0; i < RB; i++) a_row[i] = (uint32_t)min(i0 + i * 16 + i16, p.I - 1) * (uint32_t)p.lda;   // rows past I: clamped, never stored
#pragma unroll
    for (int j = 0; j < CB; j++) q_off[j] = qfrag_offset(j0 + j * 16 + i16, kg * 16, p.K_pad);         // B is packed in whole 128-column tiles

    u32x4 ra[kSkinnyAhead][RB], rb[kSkinnyAhead][CB];
    // steps go to the wavefronts in pairs, the 128 bytes of k that are a line of A's rows; a step past the end is read
    // again and its A is zeroed
    auto step_of = [&](int first, int d) { return 2 * (first + (d >> 1) * waves) + (d & 1); };
    auto load = [&](int first) {
#pragma unroll
        for (int d = 0; d < kSkinnyAhead; d++) {
            const int s = min(step_of(first, d), steps - 1);
#pragma unroll
            for (int j = 0; j < CB; j++) rb[d][j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_q, q_off[j], s * 2048, 0);
        }
        // both halves of a line one after the other: 64 rows of it are more than the L1 keeps
#pragma unroll
        for (int h = 0; h < kSkinnyAhead; h += 2)
#pragma unroll
            for (int i = 0; i < RB; i++)
#pragma unroll
                for (int d = h; d < h + 2; d++) {
                    const int s = min(step_of(first, d), steps - 1);
                    const uint32_t k = (uint32_t)min(s * 64 + kg * 16, p.lda - 16);   // past the row: its last 16 bytes, against zeros of B
                    ra[d][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_p, a_row[i] + k, 0, 0);
                }
    };
    load(wave);

    const int zd = (p.host_zp ? p.dyn_zp_value : zp_byte(p.dyn_zp, p.dyn_signed)) - p.dyn_shift;
    const int zc = (p.host_zp ? p.const_zp_value : zp_byte(p.const_zp, p.const_signed)) - p.const_shift;
    const uint32_t flip = p.dyn_shift ? 0x80808080u : 0u;
    // at the end wavefront f finishes fragment f (column block f % CB): what its column needs is asked for now
    const int cb = wave % CB, gj = j0 + cb * 16 + i16, col = min(gj, p.J - 1);
    const int csum = p.const_sum[col];
    const EmitColumn ecol = gemm_emit_column<EPI>(p, col);

    i32x4 acc[RB][CB];
    int dsum[RB] = {};
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < CB; j++) acc[i][j] = i32x4{0, 0, 0, 0};
    for (int first = wave; 2 * first < steps; first += kSkinnyAhead / 2 * waves) {
        if (first != wave) load(first);
#pragma unroll
        for (int d = 0; d < kSkinnyAhead; d++) {
            const int s = step_of(first, d);
            const uint32_t keep = s < steps && !(DYN && s * 64 + kg * 16 > p.lda - 16) ? 0xffffffffu : 0u;
#pragma unroll
            for (int i = 0; i < RB; i++) {
                const u32x4 a = (ra[d][i] ^ flip) & keep;
                if (DYN) dsum[i] += dot_ones(__builtin_bit_cast(uint4, a));
#pragma unroll
                for (int j = 0; j < CB; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, rb[d][j]), acc[i][j], 0, 0, 0);
            }
        }
    }

#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < CB; j++) red[(wave * (RB * CB) + i * CB + j) * 64 + lane] = acc[i][j];
    if (DYN) {
#pragma unroll
        for (int i = 0; i < RB; i++) {
            dsum[i] += __shfl_xor(dsum[i], 16, 64);
            dsum[i] += __shfl_xor(dsum[i], 32, 64);
            if (kg == 0) lds_sum[wave * (RB * 16) + i * 16 + i16] = dsum[i];
        }
    }
    __syncthreads();

    const int fixed = p.K * zd * zc - zd * csum;
    float fmn = 0.f, fmx = 0.f;
    const bool words = EPI == EPI_REQUANT && ((p.J | (int)(reinterpret_cast<uintptr_t>(p.Y) & 3)) & 3) == 0;   // bytes leave four columns at a time
    const RequantBytes bytes{ecol.s, (float)p.y_zp + (p.out_signed ? 128.f : 0.f), p.out_signed ? 0x80808080u : 0u};
    for (int f = wave; f < RB * CB; f += waves) {   // (waves is a multiple of CB: the column block stays)
        const int own = (f / CB) * 16 + kg * 4, row = i0 + own;   // (own: of this workgroup's rows)
        if (row - kg * 4 >= p.I) break;
        i32x4 v = {fixed, fixed, fixed, fixed}, sum = {0, 0, 0, 0};
        for (int w = 0; w < waves; w += 4) {        // (and of 4)
            i32x4 part[4];
#pragma unroll
            for (int e = 0; e < 4; e++) part[e] = red[((w + e) * (RB * CB) + f) * 64 + lane];
            v += (part[0] + part[1]) + (part[2] + part[3]);
            if (DYN) {
#pragma unroll
                for (int e = 0; e < 4; e++) sum += *reinterpret_cast<const i32x4 *>(lds_sum + (w + e) * (RB * 16) + own);
            }
        }
        if (DYN) v -= zc * sum;
        if (EPI == EPI_REQUANT && words) {
            const int q[4] = {v[0] + ecol.qb, v[1] + ecol.qb, v[2] + ecol.qb, v[3] + ecol.qb};
            const uint32_t word = gemm_quad_row(gemm_requant4(bytes, q));
            const int gi = row + (lane & 3);
            if (gi < p.I && gj < p.J) *reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(p.Y) + (size_t)gi * p.J + (gj & ~3)) = word;
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (row + r < p.I && gj < p.J) gemm_emit_mm<EPI>(p, ecol, row + r, gj, v[r], fmn, fmx);
        }
    }
    if (EPI == EPI_SCALE_BIAS) gemm_emit_range(p, lane, wave, waves, fmn, fmx);
}

}  // namespace hipc
