// MatMulNBits for a few activation rows: 2 to 64 of f16 or f32 (one of f16), on the prepacked weight. A handful of
// sequences decoded together, a short prompt, the chunk of a stream.
//
// Reference: crates/onnx-vulkan-core/src/shaders/matmul_nbits.rs:316-374, interp.rs:6429-6561.
//
// The weight is a few MB and so are the rows once every workgroup has read them, which makes the rows the thing to design
// for: on the streaming kernel (mmnb_gemv_kernel) each 16-column workgroup read and split all of them again, item after
// item, each a trip to memory of its own -- 10 of the 11.5 us of 8 x 1152 x 13824. Here
//   * a workgroup owns up to 64 columns, its wavefronts share out k (and columns), and the rows pass through LDS once: a
//     thread asks for all of its pieces at once, whole 128-byte lines, and they are written in operand order;
//   * products run on v_mfma_f32_16x16x32_f16. A nibble becomes the exact integer q - zp (nbits_f16.h), so no sums of the
//     activations are needed to take a bias out; an f16 row is one operand, exact;
//   * an f32 row is two f16 terms of the row times a power of two that brings its largest value (in the workgroup's range
//     of k) into [2^14, 2^15), or to 2^7 at least, or three terms where every bit counts (split_terms).
//     No row goes unscaled: beside values near 1, f16's smallest step (2^-24) would cost the small values of a row most of
//     their bits, in columns where the large ones meet a zero all that counts. Up to 16 rows are split by the workgroup itself (SRC_F32);
//     more are split once by a launch in front (nbits_prefill's), and travel as f16 rows;
//   * the wavefronts' partial sums meet in LDS, in a fixed order. With few columns and a long k the range of k is also
//     split over workgroups, and a second launch adds their partial rows (rows_plan weighs that launch against the bytes).
#include <algorithm>

#include "lanes.h"
#include "nbits_f16.h"

namespace hipc {

typedef __attribute__((ext_vector_type(4))) float f32x4;

enum { SRC_F16 = 0, SRC_F32 = 1 };   // the rows as they arrive: f16 (already split or exact), or f32 to be split here
constexpr int kRowsWaves = 8;        // wavefronts of a workgroup, at most (ten leave 168 registers: the kernels for more than 16 rows spill)
constexpr int kRowsPieces = 8;       // pieces of eight f32 values a thread holds while it splits them (SRC_F32)
constexpr int kRowsPieces16 = 16;    // pieces of eight f16 values on their way to LDS (SRC_F16)

struct RowsArgs {
    const void *A;
    const uint4 *Wq;
    const float *Sc;
    const uint8_t *Zb;
    void *Y;
    float *Ypart;      // with k split over workgroups: [gridDim.y][M][N]
    const int *exps;   // SRC_F16: row m of the result is multiplied by 2^exps[m] (null: not)
    int M, K, N, n_tiles, n_cg;
    int WK, WN;        // wavefronts along k, along n
    int split_tiles;   // 128-k tiles per workgroup
    int stage_tiles;   // of them in LDS at a time (all of them when the rows are split here)
    int y_f16;
    int loops;         // workgroups take one column group after another (gridDim.x of them at a time)
};

// LDS of a workgroup: 32 words of flags and magnitudes, operands [chunk][term][4 k groups][rows, made odd], partial sums --
// behind the operands where the workgroup takes several column groups, over them where it takes one
constexpr size_t kRowsHead = 128;
constexpr int kUsualExponent = -9;   // see the splitting of SRC_F32 rows
__host__ __device__ inline int rows_pitch(int M) { return M | 1; }
__host__ __device__ inline size_t rows_operands(int M, int terms, int stage_tiles) { return (size_t)stage_tiles * 4 * terms * 4 * rows_pitch(M) * 16; }

// SG: scale groups per 128-k tile (8, 4, 2, 1 for blocks of 16, 32, 64, 128 and more). NT: f16 terms per row. RB: blocks of 16 rows; NR: result registers per block in use (M <=
// 4 NR with one block: then register r of lane group g is row g + 4 r, else row 4 g + r). T: 16-column tiles per wavefront.
// P: pieces of the rows a thread holds at most (kRowsPieces of f32, kRowsPieces16 of f16, or a quarter: a launch starts with
// its instruction cache empty, and code for pieces that do not exist is 0.3 us a kilobyte).
// Two column tiles of blocks of 16 are told to keep within 128 registers (four wavefronts on a SIMD), which rows_plan counts
// on and they would miss by a few (one row, 1152 -> 13824 in two terms: 8.6 us, so 7.0).
template <int SG, int SRC, int NT, int RB, int NR, int T, int P>
__global__ void __launch_bounds__(64 * kRowsWaves, SG == 8 && RB == 1 && T == 2 && P <= 4 ? 4 : 1) mmnb_rows_kernel(const RowsArgs p) {
    extern __shared__ uint4 smem[];
    const int tid = threadIdx.x, nthreads = blockDim.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % p.WK, wn = wave / p.WK;
    const int i16 = lane & 15, g4 = lane >> 4;
    const int M = p.M, MP = rows_pitch(M);
    const int tile0 = blockIdx.y * p.split_tiles, tile1 = min(p.n_cg, tile0 + p.split_tiles);
    const int group_tiles = p.WN * T, groups = (p.n_tiles + group_tiles - 1) / group_tiles;
    // SRC_F32: [0..15] row m has a value of 1/4 or more, [16] some value is 64 or more; where not every row is a usual one,
    // the largest magnitude of row m in this workgroup's range of k, as bits
    int *head = reinterpret_cast<int *>(smem);
    bool usual = true;
    uint4 *As = smem + kRowsHead / 16;
    float *red = reinterpret_cast<float *>(reinterpret_cast<char *>(As) + (p.loops ? rows_operands(M, NT, p.stage_tiles) : 0));

    // ---- the weight: tile `tl` of T columns of tiles, as it arrives
    struct Stage {
        uint4 wq[T];
        float s[T][SG > 1 ? SG : 1];
        uint32_t z[T][SG == 8 ? 2 : 1];
    };
    // (buffer loads: what a lane adds is computed once, the tile's place is a scalar -- three instructions a tile instead of
    // a dozen. Every scalar offset is a tile's of the weight, the lane's part stays inside the tile.)
    const uint32_t n_all = (uint32_t)p.n_tiles * (uint32_t)p.n_cg;
    const auto r_wq = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4 *>(p.Wq), 0, (int)(n_all * 1024u), 0x00020000);
    const auto r_sc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.Sc), 0, (int)(n_all * 64u * SG), 0x00020000);
    const auto r_zb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(p.Zb), 0, (int)(n_all * 16u * SG), 0x00020000);
    const uint32_t v_wq = (uint32_t)lane * 16u, v_sc = (uint32_t)i16 * (4u * SG), v_zb = (uint32_t)i16 * SG;
    auto load_stage = [&](int group, int tile, Stage &st) {
        const int nt0 = group * group_tiles + wn * T;
#pragma unroll
        for (int t = 0; t < T; t++) {
            const uint32_t tl = (uint32_t)min(nt0 + t, p.n_tiles - 1) * (uint32_t)p.n_cg + (uint32_t)tile;
            st.wq[t] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r_wq, v_wq, tl * 1024u, 0));
            if constexpr (SG == 8) {
                const float4 v = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r_sc, v_sc, tl * 512u, 0));
                const float4 u = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r_sc, v_sc + 16u, tl * 512u, 0));
                const uint2 z = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r_zb, v_zb, tl * 128u, 0));
                st.s[t][0] = v.x, st.s[t][1] = v.y, st.s[t][2] = v.z, st.s[t][3] = v.w;
                st.s[t][4 % SG] = u.x, st.s[t][5 % SG] = u.y, st.s[t][6 % SG] = u.z, st.s[t][7 % SG] = u.w;
                st.z[t][0] = z.x, st.z[t][SG == 8] = z.y;
            } else if constexpr (SG == 4) {
                const float4 v = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r_sc, v_sc, tl * 256u, 0));
                st.s[t][0] = v.x, st.s[t][1] = v.y, st.s[t][2] = v.z, st.s[t][3] = v.w;
                st.z[t][0] = __builtin_amdgcn_raw_buffer_load_b32(r_zb, v_zb, tl * 64u, 0);
            } else if constexpr (SG == 2) {
                const float2 v = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r_sc, v_sc, tl * 128u, 0));
                st.s[t][0] = v.x, st.s[t][1] = v.y;
                st.z[t][0] = __builtin_amdgcn_raw_buffer_load_b16(r_zb, v_zb, tl * 32u, 0);
            } else {
                st.s[t][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r_sc, v_sc, tl * 64u, 0));
                st.z[t][0] = __builtin_amdgcn_raw_buffer_load_b8(r_zb, v_zb, tl * 16u, 0);
            }
        }
    };

    // ---- the rows: a piece is eight consecutive k of one row (of one term: term e of row m is row e M + m of A)
    auto slot = [&](int chunk, int kg, int term, int m) { return ((chunk * NT + term) * 4 + kg) * MP + m; };

    f32x4 acc[RB][T];
#pragma unroll
    for (int b = 0; b < RB; b++)
#pragma unroll
        for (int t = 0; t < T; t++) acc[b][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int a_row = NR == 4 ? i16 : (i16 >> 2) + 4 * (i16 & 3);   // the row this lane feeds (of a block); past M: row 0, never stored
    int row_at[RB];
#pragma unroll
    for (int b = 0; b < RB; b++) row_at[b] = b * 16 + a_row < M ? b * 16 + a_row : 0;
    uint32_t ones = 0x64006400u;   // kept in a vector register (see and_or_1024)
    HIPC_PIN_VGPR(ones);

    // blocks of 16: a product step of 32 k covers two of them, k groups 0 and 1 the first, 2 and 3 the second. Each is a
    // product of its own with the other half of one operand zeroed (the matrix cores have the time): of a row's first term,
    // which may hold an infinity that a weight of zero would make NaN of, and of the weight for the others, which are finite
    const uint32_t first16 = SG == 8 && g4 < 2 ? ~0u : 0u;
    const auto masked = [](const f16x8 &o, uint32_t keep) {
        const uint4 v = __builtin_bit_cast(uint4, o);
        return __builtin_bit_cast(f16x8, make_uint4(v.x & keep, v.y & keep, v.z & keep, v.w & keep));
    };
    // Where the registers allow it (128 hold twice the wavefronts of 129) the first terms' products have a sum of their own --
    // an f16 by a four-bit integer 32 times over leaves next to no rounding to do -- that the others' joins once per scale
    // group. The step between the second and third of three terms, and before it where all share a sum, is in the weight:
    // times 2^-11 and 2^-22, exact for small integers.
    constexpr bool APART = RB == 1 && NT > 1 && (T == 1 || (T == 2 && (NT == 3 || SG < 8)));
    constexpr int ND = APART ? 2 : 1;
    const auto joined = [](const f32x4 (&v)[ND], int r) {
        if constexpr (APART) return fmaf(v[1][r], NT == 3 ? 1.f / kTermStep : 1.f, v[0][r]);
        else return v[0][r];
    };
    const auto weight_for = [](const f16x8 &w, int e) {
        const int steps = NT < 3 ? 0 : APART ? e - 1 : e;
        return steps <= 0 ? w : w * (_Float16)(steps == 1 ? 1.f / kTermStep : 1.f / (kTermStep * kTermStep));
    };
    auto compute = [&](const Stage &st, int first_chunk) {
        f32x4 d[RB][T][ND];
        // three terms, and registers left: a tile's scale groups are added up among themselves first, one rounding at the size of
        // the whole sum a tile instead of one a group
        constexpr bool BY_TILE = APART && NT == 3 && T == 1 && SG < 8;
        f32x4 tile_sum[RB][T];
        const auto add = [&](int b, int t, int r, bool opens, float s, float v) {
            if (!BY_TILE) acc[b][t][r] = fmaf(s, v, acc[b][t][r]);
            else tile_sum[b][t][r] = opens ? s * v : fmaf(s, v, tile_sum[b][t][r]);
        };
        ZeroPair z[T];
        constexpr int CPG = SG == 8 ? 1 : 4 / SG;   // chunks per scale group
#pragma unroll
        for (int j = 0; j < 4; j++) {
            f16x8 a[RB][NT];
#pragma unroll
            for (int b = 0; b < RB; b++)
#pragma unroll
                for (int e = 0; e < NT; e++) a[b][e] = __builtin_bit_cast(f16x8, As[slot(first_chunk + j, g4, e, row_at[b])]);
            const bool first = j % CPG == 0, last = j % CPG == CPG - 1;
            const int g = j / CPG;
#pragma unroll
            for (int t = 0; t < T; t++) {
                if constexpr (SG == 8) {
                    z[t] = zero_pair((st.z[t][j >> 1] >> (16 * (j & 1) + (first16 ? 0 : 8))) & 0xffu);   // of the lane's own block
                } else {
                    if (first) z[t] = zero_pair((st.z[t][0] >> (8 * g)) & 0xffu);
                }
                const f16x8 w = dequant_operand(word_of(st.wq[t], j), z[t], ones);
                if constexpr (SG == 8) {
                    const f16x8 w0 = masked(w, first16), w1 = masked(w, ~first16);
#pragma unroll
                    for (int b = 0; b < RB; b++) {
                        f32x4 v0[ND], v1[ND];
#pragma unroll
                        for (int e = 0; e < ND; e++) v0[e] = v1[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int e = NT - 1; e >= 0; e--) {
                            const int c = APART && e > 0;
                            v0[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(e ? a[b][e] : masked(a[b][e], first16), e ? weight_for(w0, e) : w, v0[c], 0, 0, 0);
                            v1[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(e ? a[b][e] : masked(a[b][e], ~first16), e ? weight_for(w1, e) : w, v1[c], 0, 0, 0);
                        }
#pragma unroll
                        for (int r = 0; r < NR; r++) add(b, t, r, j == 0, st.s[t][2 * j % SG], joined(v0, r)), add(b, t, r, false, st.s[t][(2 * j + 1) % SG], joined(v1, r));
                    }
                    continue;
                }
#pragma unroll
                for (int b = 0; b < RB; b++) {
                    if (first)
#pragma unroll
                        for (int e = 0; e < ND; e++) d[b][t][e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int e = NT - 1; e >= 0; e--) {
                        const int c = APART && e > 0;
                        d[b][t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[b][e], weight_for(w, e), d[b][t][c], 0, 0, 0);
                    }
                    if (last) {
#pragma unroll
                        for (int r = 0; r < NR; r++) add(b, t, r, g == 0, st.s[t][g], joined(d[b][t], r));
                    }
                }
            }
        }
        if constexpr (BY_TILE)
#pragma unroll
            for (int b = 0; b < RB; b++)
#pragma unroll
                for (int t = 0; t < T; t++)
#pragma unroll
                    for (int r = 0; r < NR; r++) acc[b][t][r] += tile_sum[b][t][r];
    };
    // This wavefront's tiles of a stage [t0, t1) in LDS; `cur` is the first of them, and on leaving the first of the next
    // stage (a stage is a whole number of rounds of the wavefronts) or group, the tile after it always on its way.
    Stage cur;
    auto walk = [&](int group, int t0, int t1) {
        for (int tile = t0 + wk; tile < t1; tile += p.WK) {
            Stage next;
            const bool more = tile + p.WK < tile1;
            load_stage(more ? group : min(group + (int)gridDim.x, groups - 1), more ? tile + p.WK : min(tile0 + wk, tile1 - 1), next);
            __builtin_amdgcn_sched_barrier(0);   // (the compiler moves these loads behind the products: every tile then waits out a trip to memory)
            compute(cur, (tile - t0) * 4);
            cur = next;
        }
    };
    // The wavefronts along k meet: [wn][register][wk][lane], every wavefront finishing its share of the registers.
    auto finish = [&](int group) {
        if (!p.loops) __syncthreads();   // the operands have been read
        constexpr int Q = RB * T * NR;
#pragma unroll
        for (int b = 0; b < RB; b++)
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    red[((wn * Q + (b * T + t) * NR + r) * p.WK + wk) * 64 + lane] = acc[b][t][r];
                    acc[b][t][r] = 0.f;
                }
        __syncthreads();
        for (int q = wk; q < Q; q += p.WK) {
            const float *src = red + (size_t)(wn * Q + q) * p.WK * 64 + lane;
            float part[kRowsWaves], v = 0.f;
#pragma unroll
            for (int k = 0; k < kRowsWaves; k++) part[k] = src[min(k, p.WK - 1) * 64];
#pragma unroll
            for (int k = 0; k < kRowsWaves; k++) v += k < p.WK ? part[k] : 0.f;
            const int b = q / (T * NR), t = q / NR % T, r = q % NR;
            const int m = b * 16 + (NR == 4 ? 4 * g4 + r : g4 + 4 * r), n = (group * group_tiles + wn * T + t) * 16 + i16;
            if (m >= M || n >= p.N) continue;
            if (SRC == SRC_F32) v = ldexpf(v, usual ? kUsualExponent : row_exponent((uint32_t)head[m]));
            const size_t at = (size_t)m * p.N + n;
            if (p.Ypart) {
                p.Ypart[(size_t)blockIdx.y * M * p.N + at] = v;
            } else {
                if (SRC == SRC_F16 && p.exps) v = ldexpf(v, p.exps[m]);
                if (p.y_f16) static_cast<__half *>(p.Y)[at] = __float2half(v);
                else static_cast<float *>(p.Y)[at] = v;
            }
        }
    };

    if constexpr (SRC == SRC_F32) {
        // pieces tid, tid + nthreads, ... of M rows x R pieces; R is a multiple of 16, so the 16 lanes of a DPP row hold
        // pieces of one row
        const int R = (tile1 - tile0) * 16, items = M * R;
        const int step_m = nthreads / R, step_c = nthreads - step_m * R;
        int m = tid / R, c = tid - m * R;
        const float *A = static_cast<const float *>(p.A) + tile0 * 128;
        const int k_left = p.K - tile0 * 128;
        if (tid < 32) head[tid] = 0;
        float4 lo[P], hi[P];
        int at_m[P], at_c[P];
#pragma unroll
        for (int u = 0; u < P; u++) {
            lo[u] = hi[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            at_m[u] = m, at_c[u] = c;
            if (tid + u * nthreads < items && c * 8 < k_left) {   // (K is a multiple of 8)
                const float4 *src = reinterpret_cast<const float4 *>(A + (size_t)m * p.K + c * 8);
                lo[u] = src[0], hi[u] = src[1];
            }
            m += step_m, c += step_c;
            if (c >= R) c -= R, m++;
        }
        load_stage(blockIdx.x, min(tile0 + wk, tile1 - 1), cur);   // the first weight tiles travel meanwhile
        auto largest = [&](int u) {
            const float a = fmaxf(fmaxf(fabsf(lo[u].x), fabsf(lo[u].y)), fmaxf(fabsf(lo[u].z), fabsf(lo[u].w)));
            return fmaxf(a, fmaxf(fmaxf(fabsf(hi[u].x), fabsf(hi[u].y)), fmaxf(fabsf(hi[u].z), fabsf(hi[u].w))));
        };
        auto split = [&](int u, float down) {
            const float v[8] = {lo[u].x, lo[u].y, lo[u].z, lo[u].w, hi[u].x, hi[u].y, hi[u].z, hi[u].w};
            f16x8 t[NT];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                _Float16 terms[NT];
                split_terms<NT>(v[i] * down, terms);
#pragma unroll
                for (int e = 0; e < NT; e++) t[e][i] = terms[e];
            }
#pragma unroll
            for (int e = 0; e < NT; e++) As[slot(at_c[u] >> 2, at_c[u] & 3, e, at_m[u])] = __builtin_bit_cast(uint4, t[e]);
        };
        __syncthreads();   // the flags are cleared
        // Rows as they usually are, every one's largest value in [1/4, 64), are all scaled by 2^9 as their pieces arrive, without
        // waiting for the maxima: that puts the largest value between 2^7 and 2^15, and what two terms lose (2^-25) at 2^-32
        // of it at most. (8 x 1152 x 4096: 4.9 us, 5.3 with a power of two for each row; 16 x 1152 x 13824 9.0 and 10.4)
#pragma unroll
        for (int u = 0; u < P; u++) {
            if (tid + u * nthreads >= items) continue;
            const float mx = largest(u);
            if (mx >= 0.25f) head[at_m[u]] = 1;
            if (!(mx < 64.f)) head[16] = 1;
            split(u, two_to_minus(kUsualExponent));
        }
        __syncthreads();
        if (__any(head[16] != 0 || (lane < M && head[lane & 15] == 0))) {   // (the same in every wavefront)
            usual = false;
            // the largest magnitude of each row, as bits (non-negative floats order like them)
            __syncthreads();
            if (tid < 16) head[tid] = 0;
            __syncthreads();
#pragma unroll
            for (int u = 0; u < P; u++) {
                if ((tid & ~15) + u * nthreads >= items) continue;
                const float mx = lean_row_max(largest(u));
                if (i16 == 0) atomicMax(&head[at_m[u]], (int)__float_as_uint(mx));
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < P; u++)
                if (tid + u * nthreads < items) split(u, two_to_minus(row_exponent((uint32_t)head[at_m[u]])));
            __syncthreads();
        }
        for (int group = blockIdx.x; group < groups; group += gridDim.x) {
            if (group != (int)blockIdx.x) __syncthreads();   // the sums of the group before have been read
            walk(group, tile0, tile1);
            finish(group);
        }
    } else {
        const __half *A = static_cast<const __half *>(p.A);
        const int rows = NT * M;
        uint4 piece[P];
        // pieces of a stage: R to a row
        auto fetch = [&](int t0) {
            const int R = (min(tile1, t0 + p.stage_tiles) - t0) * 16, items = rows * R;
            const int step_m = nthreads / R, step_c = nthreads - step_m * R;
            int m = tid / R, c = tid - m * R;
#pragma unroll
            for (int u = 0; u < P; u++) {
                piece[u] = make_uint4(0u, 0u, 0u, 0u);
                if (tid + u * nthreads < items && t0 * 128 + c * 8 < p.K) piece[u] = *reinterpret_cast<const uint4 *>(A + (size_t)m * p.K + t0 * 128 + c * 8);
                m += step_m, c += step_c;
                if (c >= R) c -= R, m++;
            }
        };
        auto store = [&](int t0) {
            const int R = (min(tile1, t0 + p.stage_tiles) - t0) * 16, items = rows * R;
            const int step_m = nthreads / R, step_c = nthreads - step_m * R;
            int m = tid / R, c = tid - m * R;
#pragma unroll
            for (int u = 0; u < P; u++) {
                if (tid + u * nthreads < items) {
                    const int e = NT > 1 ? (m >= M) + (NT > 2 && m >= 2 * M) : 0;
                    As[slot(c >> 2, c & 3, e, m - e * M)] = piece[u];
                }
                m += step_m, c += step_c;
                if (c >= R) c -= R, m++;
            }
        };
        fetch(tile0);
        load_stage(blockIdx.x, min(tile0 + wk, tile1 - 1), cur);
        if (p.loops) {   // all of this workgroup's k in LDS: any number of column groups
            store(tile0);
            for (int group = blockIdx.x; group < groups; group += gridDim.x) {
                __syncthreads();
                walk(group, tile0, tile1);
                finish(group);
            }
        } else {                                // (the launch then has a workgroup per group)
            for (int t0 = tile0; t0 < tile1; t0 += p.stage_tiles) {
                const int t1 = min(tile1, t0 + p.stage_tiles);
                if (t0 != tile0) __syncthreads();   // the stage before has been read
                store(t0);
                __syncthreads();
                if (t1 < tile1) fetch(t1);
                walk(blockIdx.x, t0, t1);
            }
            finish(blockIdx.x);
        }
    }
}

// Y = sum over the workgroups' partial rows, in order, times 2^exps[row] where given; four results per thread
template <bool VEC>   // VEC: N is a multiple of four and Y's rows take 16-byte (f16: 8-byte) stores
static __global__ void __launch_bounds__(64)
mmnb_rows_join_kernel(const float *__restrict__ part, void *__restrict__ Y, long total, int splits, int N, const int *__restrict__ exps, int y_f16) {
    const long i = ((long)blockIdx.x * 64 + threadIdx.x) * (VEC ? 4 : 1);
    if (i >= total) return;
    constexpr int V = VEC ? 4 : 1;
    float v[V];
    auto read = [&](int s, float (&o)[V]) {
        const float *src = part + (size_t)s * total + i;
        if (VEC) {
            const float4 f = *reinterpret_cast<const float4 *>(src);
            o[0] = f.x;
            if constexpr (VEC) o[1] = f.y, o[2] = f.z, o[3] = f.w;
        } else {
            o[0] = *src;
        }
    };
    read(0, v);
    int s = 1;
    constexpr int kFlight = 8;          // reads in flight: a trip to memory is most of what this launch lasts
    for (; s < splits; s += kFlight) {
        float u[kFlight][V];
#pragma unroll
        for (int d = 0; d < kFlight; d++) read(min(s + d, splits - 1), u[d]);
#pragma unroll
        for (int d = 0; d < kFlight; d++)
#pragma unroll
            for (int j = 0; j < V; j++) v[j] += s + d < splits ? u[d][j] : 0.f;
    }
    if (exps) {
        const int e = exps[i / N];
#pragma unroll
        for (int j = 0; j < V; j++) v[j] = ldexpf(v[j], e);
    }
    if constexpr (VEC) {
        if (y_f16)
            *reinterpret_cast<uint2 *>(static_cast<__half *>(Y) + i) = make_uint2(two_halves(__float2half(v[0]), __float2half(v[1])), two_halves(__float2half(v[2]), __float2half(v[3])));
        else
            *reinterpret_cast<float4 *>(static_cast<float *>(Y) + i) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
        if (y_f16) static_cast<__half *>(Y)[i] = __float2half(v[0]);
        else static_cast<float *>(Y)[i] = v[0];
    }
}

namespace {

struct RowsPlan {
    int T, WN, WK, splits, split_tiles, stage_tiles, grid_x;
    bool loops;
    size_t lds;
};

// How many columns a workgroup takes and how many ways k is split over workgroups. A CU takes in about 32 bytes per clock
// (17.7 TB/s of L2 over 256 CUs), of rows and of weight alike: few columns per workgroup read the rows often, many leave
// CUs without work, the code of a tile's products is fetched by an empty instruction cache (600 clocks per row block and
// column tile: 24 x 2048 x 8320 9.2 us without that term, 7.6 with it), and a split costs a second launch: 3000 clocks with
// its own trip through memory, most of the launch's 2.4 us hiding behind the first one's last workgroups. (Counted as 6000, the
// rule kept 2 x 11008 x 1024 and x 2048 whole: 8.8 and 9.7 us, 6.6 and 7.8 split; counted as 2000, it splits 2 x 8192 x 512 and 20 x 2048 x 1024
// for 8 % more, called one by one. Joining in the workgroup that comes last instead of a launch: 7.6 us for the 6.8 of 8 x 6912 x 1152.)
bool rows_plan(hipc_ctx *ctx, const hipc_nbits_weight *w, int M, int src, int NT, int RB, int NR, bool may_split, RowsPlan *best) {
    const int cus = std::max(1, ctx->cu_count), max_waves = kRowsWaves;
    const int most_splits = may_split ? std::min(w->n_cg, std::max(16, (int)ceil_div(w->n_cg, 8))) : 1;   // (up to eight tiles of k fit any launch)
    double best_cost = 0;
    bool found = false;
    static const int shapes[][2] = {{4, 1}, {2, 1}, {1, 1}, {2, 2}, {1, 2}};   // column tiles per wavefront, wavefronts side by side
    for (const auto &shape : shapes) {
        if ((RB > 2 || w->SG == 8) && shape[0] == 4) continue;   // (registers)
        if ((NT * M > 64) != (shape[1] > 1)) continue;   // a stage is at least a round of the wavefronts along k: eight of them only up to 64 rows
        const int cw = shape[0] * shape[1];
        const int64_t groups = ceil_div(w->n_tiles, cw);
        for (int splits = 1; splits <= most_splits; splits++) {
            const int st = (int)ceil_div(w->n_cg, splits);
            if ((int)ceil_div(w->n_cg, st) != splits) continue;
            RowsPlan pl;
            pl.splits = splits, pl.split_tiles = st, pl.T = shape[0], pl.WN = shape[1];
            pl.WK = (int)ceil_div(st, ceil_div(st, max_waves / pl.WN));
            const int waves = pl.WK * pl.WN, threads = 64 * waves, regs = RB * pl.T * NR;
            if (src == SRC_F32) {
                pl.stage_tiles = st;
                if ((int64_t)M * st * 16 > (int64_t)kRowsPieces * threads) continue;
            } else {
                pl.stage_tiles = (int)std::min<int64_t>(st, (int64_t)kRowsPieces16 * threads / ((int64_t)NT * M * 16));
                if (pl.stage_tiles < st) pl.stage_tiles = pl.stage_tiles / pl.WK * pl.WK;   // whole rounds of the wavefronts
                if (pl.stage_tiles < 1) continue;
            }
            // two wavefronts on a SIMD, four where the kernel keeps within 128 registers
            const int64_t pieces = ceil_div((int64_t)(src == SRC_F32 ? 1 : NT) * M * pl.stage_tiles * 16, threads);
            const int cu_waves = src == SRC_F32 ? (pl.T * pieces <= 8 || pl.T == 1 ? 16 : 8) : RB <= 2 && NT * RB * pl.T * pieces <= 16 ? 16 : 8;
            // several column groups one after another where there are more of them than the chip holds workgroups, and all
            // of the workgroup's k is in LDS
            const int64_t wgs = groups * splits;
            const size_t operands = rows_operands(M, NT, pl.stage_tiles), sums = (size_t)waves * regs * 256;
            const auto resident_of = [&](size_t lds) { return std::max<int64_t>(1, std::min<int64_t>((int64_t)(160 * 1024 / lds), 64 * cu_waves / threads)); };
            pl.lds = kRowsHead + operands + sums;
            pl.loops = pl.stage_tiles >= st && pl.lds <= 150 * 1024 && wgs > cus * resident_of(pl.lds);
            if (!pl.loops) pl.lds = kRowsHead + std::max(operands, sums);
            if (pl.lds > 150 * 1024) continue;
            const int64_t resident = resident_of(pl.lds);
            pl.grid_x = pl.loops ? (int)std::max<int64_t>(1, cus * resident / splits) : (int)groups;
            const double row_bytes = (double)M * st * 128 * (src == SRC_F32 ? 4 : 2 * NT), weight_bytes = (double)cw * st * (1024 + 80 * w->SG);
            const double rounds = (double)ceil_div(wgs, cus * resident), per_cu = (double)std::min<int64_t>(resident, ceil_div(wgs, cus));
            double cost = 600.0 * RB * pl.T + (pl.loops ? per_cu * row_bytes / 32 + 2500 + rounds * (per_cu * weight_bytes / 32 + 800) : rounds * (per_cu * (row_bytes + weight_bytes) / 32 + 2500));
            if (splits > 1) cost += 3000 + (double)splits * M * w->N * 8 / (32.0 * cus);
            if (!found || cost < best_cost) found = true, best_cost = cost, *best = pl;
        }
    }
    return found;
}

// ... for this call: without a split of k where its scratch memory is not to be had
size_t rows_part_bytes(const hipc_nbits_weight *w, int M, const RowsPlan &pl) { return (size_t)pl.splits * M * w->N * sizeof(float); }
bool rows_plan_now(hipc_ctx *ctx, const hipc_nbits_weight *w, int M, int src, int NT, int RB, int NR, RowsPlan *pl) {
    if (!rows_plan(ctx, w, M, src, NT, RB, NR, true, pl)) return false;
    return pl->splits == 1 || scratch_fits(ctx, 0, rows_part_bytes(w, M, *pl)) || rows_plan(ctx, w, M, src, NT, RB, NR, false, pl);
}

template <int SG, int SRC, int NT, int RB, int NR, int T, int P>
int rows_launch_p(hipc_ctx *ctx, const RowsArgs &a, const RowsPlan &pl) {
    static bool lds_allowed[kMaxDevices] = {};
    if (int rc = allow_dynamic_lds(ctx, mmnb_rows_kernel<SG, SRC, NT, RB, NR, T, P>, 150 * 1024, lds_allowed)) return rc;
    const dim3 grid((unsigned)pl.grid_x, (unsigned)pl.splits);
    hipLaunchKernelGGL((mmnb_rows_kernel<SG, SRC, NT, RB, NR, T, P>), grid, dim3(64 * pl.WK * pl.WN), pl.lds, ctx->stream, a);
    HIPC_LAUNCHED(ctx);
    return HIPC_OK;
}
template <int SG, int SRC, int NT, int RB, int NR, int T>
int rows_launch(hipc_ctx *ctx, const RowsArgs &a, const RowsPlan &pl) {
    constexpr int most = SRC == SRC_F32 ? kRowsPieces : kRowsPieces16;
    const int64_t pieces = ceil_div((int64_t)(SRC == SRC_F32 ? 1 : NT) * a.M * pl.stage_tiles * 16, 64 * pl.WK * pl.WN);
    if constexpr (RB <= 2) {
        if (pieces <= most / 4) return rows_launch_p<SG, SRC, NT, RB, NR, T, most / 4>(ctx, a, pl);
        if (pieces <= most / 2) return rows_launch_p<SG, SRC, NT, RB, NR, T, most / 2>(ctx, a, pl);
    }
    return rows_launch_p<SG, SRC, NT, RB, NR, T, most>(ctx, a, pl);
}
template <int SRC, int NT, int RB, int NR, int T>
int rows_launch_sg(hipc_ctx *ctx, const RowsArgs &a, const RowsPlan &pl, int SG) {
    switch (SG) {
        case 8:
            if constexpr (T <= 2) return rows_launch<8, SRC, NT, RB, NR, T>(ctx, a, pl);
            break;   // (rows_plan: never)
        case 4: return rows_launch<4, SRC, NT, RB, NR, T>(ctx, a, pl);
        case 2: return rows_launch<2, SRC, NT, RB, NR, T>(ctx, a, pl);
        case 1: return rows_launch<1, SRC, NT, RB, NR, T>(ctx, a, pl);
    }
    return fail(ctx, HIPC_ERR_INVALID, "MatMulNBits rows: no kernel for %d scale groups and %d column tiles", SG, T);
}
template <int SRC, int NT, int RB, int NR>
int rows_run(hipc_ctx *ctx, RowsArgs a, const hipc_nbits_weight *w) {
    RowsPlan pl;
    HIPC_REFUSE(ctx, !rows_plan_now(ctx, w, a.M, SRC, NT, RB, NR, &pl), "MatMulNBits rows: no launch shape for %d rows", a.M);
    a.Wq = w->Wq, a.Sc = w->Sc, a.Zb = w->Zb;
    a.K = (int)w->K, a.N = (int)w->N, a.n_tiles = w->n_tiles, a.n_cg = w->n_cg;
    a.WK = pl.WK, a.WN = pl.WN, a.split_tiles = pl.split_tiles, a.stage_tiles = pl.stage_tiles;
    a.loops = pl.loops;
    a.Ypart = nullptr;
    if (pl.splits > 1) {
        void *part = nullptr;
        if (int rc = scratch_get(ctx, 0, rows_part_bytes(w, a.M, pl), &part)) return rc;
        a.Ypart = static_cast<float *>(part);
    }
    int rc;
    if constexpr (RB <= 2) {
        rc = pl.T == 4 ? rows_launch_sg<SRC, NT, RB, NR, 4>(ctx, a, pl, w->SG) : pl.T == 2 ? rows_launch_sg<SRC, NT, RB, NR, 2>(ctx, a, pl, w->SG) : rows_launch_sg<SRC, NT, RB, NR, 1>(ctx, a, pl, w->SG);
    } else {
        rc = pl.T == 2 ? rows_launch_sg<SRC, NT, RB, NR, 2>(ctx, a, pl, w->SG) : rows_launch_sg<SRC, NT, RB, NR, 1>(ctx, a, pl, w->SG);
    }
    if (rc != HIPC_OK || pl.splits == 1) return rc;
    const long total = (long)a.M * a.N;
    if (a.N % 4 == 0 && aligned(a.Y, a.y_f16 ? 8 : 16))
        hipLaunchKernelGGL((mmnb_rows_join_kernel<true>), dim3((unsigned)ceil_div(total, 256)), 64, 0, ctx->stream, static_cast<const float *>(a.Ypart), a.Y, total, pl.splits, a.N, a.exps, a.y_f16);
    else
        hipLaunchKernelGGL((mmnb_rows_join_kernel<false>), dim3((unsigned)ceil_div(total, 64)), 64, 0, ctx->stream, static_cast<const float *>(a.Ypart), a.Y, total, pl.splits, a.N, a.exps, a.y_f16);
    HIPC_LAUNCHED(ctx);
    return HIPC_OK;
}

}  // namespace

// (this file is compiled twice: HIPC_ROWS_F16 is the half whose rows arrive as f16)
#ifdef HIPC_ROWS_F16

// rows of f16, `terms` of them per row of the result (term e of row m is row e M + m of A); exps / y_f16 as in RowsArgs
int nbits_rows_f16(hipc_ctx *ctx, const void *A, int terms, const int *exps, const hipc_nbits_weight *w, void *Y, int y_f16, int M) {
    RowsArgs a{};
    a.A = A, a.Y = Y, a.exps = exps, a.M = M, a.y_f16 = y_f16;
    if (terms == 3) return M <= 32 ? rows_run<SRC_F16, 3, 2, 4>(ctx, a, w) : rows_run<SRC_F16, 3, 4, 4>(ctx, a, w);
    if (terms == 2) return M <= 32 ? rows_run<SRC_F16, 2, 2, 4>(ctx, a, w) : rows_run<SRC_F16, 2, 4, 4>(ctx, a, w);
    if (M <= 4) return rows_run<SRC_F16, 1, 1, 1>(ctx, a, w);
    if (M <= 8) return rows_run<SRC_F16, 1, 1, 2>(ctx, a, w);
    if (M <= 16) return rows_run<SRC_F16, 1, 1, 4>(ctx, a, w);
    return M <= 32 ? rows_run<SRC_F16, 1, 2, 4>(ctx, a, w) : rows_run<SRC_F16, 1, 4, 4>(ctx, a, w);
}

#else

// Which row counts come here (kernel time of the call, before -> after; the streaming kernel 16 rows at a time, the tiled
// kernel from 17 rows of f16 and 33 of f32 on): 8 x 1152 x 13824 11.5 -> 7.5 us, 16 rows 23 -> 9.4, 32 rows 46 -> 19; 8 x 6912
// x 1152 10.4 -> 7.1, 16 rows 19 -> 8.2; f16 2048 -> 11008: 1 row 7.3 -> 6.5, 4 rows 11.2 -> 6.5, 16 rows 24 -> 7.8, 17 rows
// 11.3 -> 8.6; 24 x 512 -> 1152 5.4 -> 4.5, but -> 16384 5.5 -> 5.9. From 33 rows on only where the tiled kernel has few tiles: f16 48 x 6912 x 1152 27.4 -> 11.6, but 48 x 4096 x
// 4096 18.1 -> 21.4; f32 (which the tiled kernel takes 64 rows at a time) 48 x 6912 x 1152 41 -> 22.7, 48 x 4096 x 4096 39 ->
// 25, but 64 x 2048 x 8192 32.6 -> 37. A weight of 2048 column tiles or more and up to 16 rows stay on the streaming kernel,
// whose wavefronts each walk all of k and meet nobody: 4 x 1152 x 262144 35.7 us there (5.5 TB/s), 50 here.
// Inside a capture, only where the scratch memory is to be had or not needed.
bool nbits_rows_takes(hipc_ctx *ctx, const void *A, int a_dtype, const hipc_nbits_weight *w, int64_t M, int terms) {
    if (M > kFewRows || terms * M > 128 || w->K % 8 != 0 || !aligned(A, 16)) return false;
    const bool shape = M <= 16 ? w->n_tiles < 2048 || w->SG == 8   // (the streaming kernel has no form for blocks of 16)
                     : M <= 32 ? terms > 1 || w->n_tiles <= 300 || w->n_cg > 4 : w->n_tiles <= (terms > 1 ? 300 : 128);
    if (!shape || !ctx->capturing) return shape;
    const bool split_in_front = a_dtype == HIPC_F32 && M > 16;
    if (split_in_front && !scratch_fits(ctx, 2, nbits_split_bytes(terms * M, M, w->K))) return false;
    const int src = a_dtype == HIPC_F32 && M <= 16 ? SRC_F32 : SRC_F16;
    const int RB = M > 32 ? 4 : M > 16 ? 2 : 1, NR = M <= 4 ? 1 : M <= 8 ? 2 : 4;   // (as nbits_rows_f32 and nbits_rows_f16 dispatch)
    RowsPlan pl;
    return rows_plan_now(ctx, w, (int)M, src, terms, RB, NR, &pl);
}

// up to 16 rows of f32, as two f16 terms or three
int nbits_rows_f32(hipc_ctx *ctx, const void *A, const hipc_nbits_weight *w, void *Y, int M, int terms) {
    RowsArgs a{};
    a.A = A, a.Y = Y, a.M = M;
    if (terms == 3) return M <= 4 ? rows_run<SRC_F32, 3, 1, 1>(ctx, a, w) : M <= 8 ? rows_run<SRC_F32, 3, 1, 2>(ctx, a, w) : rows_run<SRC_F32, 3, 1, 4>(ctx, a, w);
    return M <= 4 ? rows_run<SRC_F32, 2, 1, 1>(ctx, a, w) : M <= 8 ? rows_run<SRC_F32, 2, 1, 2>(ctx, a, w) : rows_run<SRC_F32, 2, 1, 4>(ctx, a, w);
}

#endif

}  // namespace hipc
