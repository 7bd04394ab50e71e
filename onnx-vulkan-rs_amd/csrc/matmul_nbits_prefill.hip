// MatMulNBits for many rows of f16 activations (prefill): Y[M, N] = A[M, K] x dequant(W)[K, N].
//
// The reference has no tiled path for this shape: its kernels re-read the weight once per row
// (crates/onnx-vulkan-core/src/shaders/matmul_nbits.rs:21-25). Here the weight is read once per
// 64- or 128-row tile of A and the products run on the matrix cores. Two kernels: the one further
// down (mmnb_prefill_direct_kernel), which every shape takes by default, keeps the weight out of LDS;
// the first one passes both operands through LDS and stays behind the prefill_direct option as the
// control the other is tested against:
//
//   * a 256-thread workgroup owns a T x T tile of Y (T = 128, or 64 when that would leave CUs
//     idle), four wavefronts as 2 x 2, each T/2 x T/2 as 32x32 accumulators of
//     v_mfma_f32_32x32x16_f16 (f16 x f16 products are exact in the f32 accumulator);
//   * a k stage is 64 values: 128-byte LDS rows (pitch 144, conflict-free 128-bit reads) for
//     both operands. A goes memory -> registers -> LDS as it is. The weight comes from the
//     prepacked tiles as 32-bit words of eight nibbles and becomes f16 on the way into LDS:
//     the prepacked nibble order makes (word >> 4 i) & 0x000f000f the pair (k_2i, k_2i+1); or-ed with
//     0x6400 that is f16 1024 + q (exact), and the f16 value 1024 + zero_point is subtracted, so LDS
//     holds the exact integers q - zp;
//   * scales stay out of the f16 operands (folding them in would round every weight): the
//     accumulators of one quantisation block are multiplied by the block's scale and added to
//     the running total in f32, once per block (per 32, 64 or 128 k).
//
// Two register sets and two LDS buffers keep two stages in flight, as in the int8 kernel.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cstdlib>

#include "internal.h"
#include "nbits_f16.h"

namespace hipc {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kPK = 64;          // k values per stage
constexpr int kPPitch = 144;     // bytes between LDS rows (128 of data)
constexpr size_t prefill_lds(int tile) { return 4 * (size_t)tile * kPPitch; }

struct PrefillArgs {
    const __half *A;
    const uint4 *Wq;
    const float *Sc;
    const uint8_t *Zb;
    __half *Y;
    int M, K, N;
    int n_tiles, n_cg;
    int xcd_rows, xcd_cols;
    // k split over workgroups (gridDim.y): each takes `split_stages` stages (an even number, so that
    // weight tiles are not cut) and writes f32 partials [split][M][N] that a second launch adds up
    int ksplit, split_stages;
    float *Ypart;
    float *Yf32;   // when set, the result is written here as f32 and Y is not used (rows of f32 activations, see nbits_prefill_f32)
    // Rows in terms (set together; only the kernel that keeps the weight out of LDS): A holds the `terms` (2 or 3) f16 terms of
    // `pair_rows` f32 rows, the high terms of 32 rows followed by these rows' lower terms, and a wavefront owns all terms of its
    // rows: they add up in its accumulator. Row r of the result is stored times 2^exps[r] -- into Yf32, or unscaled into the k
    // split's partials [split][pair_rows][N].
    // exps without pair_rows: A holds one f16 term per f32 row and row r of the f32 result is stored times 2^exps[r]
    // (any of the kernels; the k split's partials stay unscaled).
    const int *exps;
    int pair_rows, terms;
};

// eight nibbles (order k0 k2 k4 k6 k1 k3 k5 k7) -> eight f16 values q - zp in k order, as four words of pairs
__device__ __forceinline__ uint4 dequant8(uint32_t w, uint32_t zb) {
    // 1024 + zp in both halves; zb carries 128 + zp
    const uint32_t zh = 0x6400u + (zb - 128u);
    const f16x2 z2 = __builtin_bit_cast(f16x2, zh | (zh << 16));
    uint32_t out[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        // nibbles i and i + 4 into the two halves, then the exponent of 1024: f16 (1024 + q), exact
        const uint32_t pair = ((w >> (4 * i)) & 0x000f000fu) | 0x64006400u;
        out[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, pair) - z2);
    }
    return make_uint4(out[0], out[1], out[2], out[3]);
}

// the wavefront's accumulators (F x F blocks of 32x32, first row i0, first column j0) to Y, to the f32 result or to
// the k split's partials. Which of the three, and whether the wavefront's square lies inside the matrix, is decided
// once (asked per element, the same questions made 3000 instructions of this and 5 of the kernel's 45 us).
template <int FM, int FN, bool CHECKED, typename OUT>
__device__ __forceinline__ void prefill_store_as(OUT *__restrict__ dst, int M, int N, const f32x16 (&total)[FM][FN], int i0, int j0, int r32, int kg,
                                                 const int *__restrict__ exps = nullptr) {   // exps (f32 results only): row r times 2^exps[r]
#pragma unroll
    for (int i = 0; i < FM; i++) {
        int e[16];
        if constexpr (sizeof(OUT) == 4) {
#pragma unroll
            for (int r = 0; r < 16; r++) e[r] = exps ? exps[min(i0 + i * 32 + kg * 4 + (r >> 2) * 8 + (r & 3), M - 1)] : 0;
        }
#pragma unroll
        for (int j = 0; j < FN; j++) {
            const int gj = j0 + j * 32 + r32;
            OUT *at = dst + (size_t)(i0 + i * 32 + kg * 4) * N + gj;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int rf = (r >> 2) * 8 + (r & 3);   // (+ kg * 4, which is in `at`)
                if (!CHECKED || (i0 + i * 32 + kg * 4 + rf < M && gj < N)) {
                    if constexpr (sizeof(OUT) == 2) at[(size_t)rf * N] = __float2half(total[i][j][r]);
                    else at[(size_t)rf * N] = exps ? ldexpf(total[i][j][r], e[r]) : total[i][j][r];
                }
            }
        }
    }
}
template <int FM, int FN>
__device__ __forceinline__ void prefill_store(const PrefillArgs &p, const f32x16 (&total)[FM][FN], int i0, int j0, int r32, int kg) {
    const bool inside = i0 + FM * 32 <= p.M && j0 + FN * 32 <= p.N;
    float *f32_to = p.ksplit > 1 ? p.Ypart + (size_t)blockIdx.y * p.M * p.N : p.Yf32;
    if (f32_to) {
        const int *exps = p.ksplit > 1 ? nullptr : p.exps;
        if (inside) prefill_store_as<FM, FN, false>(f32_to, p.M, p.N, total, i0, j0, r32, kg, exps);
        else prefill_store_as<FM, FN, true>(f32_to, p.M, p.N, total, i0, j0, r32, kg, exps);
    } else {
        if (inside) prefill_store_as<FM, FN, false>(p.Y, p.M, p.N, total, i0, j0, r32, kg);
        else prefill_store_as<FM, FN, true>(p.Y, p.M, p.N, total, i0, j0, r32, kg);
    }
}

// paired rows: one block of 32 result rows (first row i0 of the result) times 2^exps[row], or unscaled partials
template <int FN, bool CHECKED>
__device__ __forceinline__ void prefill_store_pairs_as(float *__restrict__ dst, const int *__restrict__ exps, int M, int N, const f32x16 (&total)[1][FN], int i0, int j0, int r32, int kg) {
    int e[16];
#pragma unroll
    for (int r = 0; r < 16; r++) e[r] = exps ? exps[min(i0 + kg * 4 + (r >> 2) * 8 + (r & 3), M - 1)] : 0;
#pragma unroll
    for (int j = 0; j < FN; j++) {
        const int gj = j0 + j * 32 + r32;
        float *at = dst + (size_t)(i0 + kg * 4) * N + gj;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int rf = (r >> 2) * 8 + (r & 3);
            if (!CHECKED || (i0 + kg * 4 + rf < M && gj < N)) at[(size_t)rf * N] = ldexpf(total[0][j][r], e[r]);
        }
    }
}
template <int FN>
__device__ __forceinline__ void prefill_store_pairs(const PrefillArgs &p, const f32x16 (&total)[1][FN], int i0, int j0, int r32, int kg) {
    const bool inside = i0 + 32 <= p.pair_rows && j0 + FN * 32 <= p.N;
    float *to = p.ksplit > 1 ? p.Ypart + (size_t)blockIdx.y * p.pair_rows * p.N : p.Yf32;
    const int *exps = p.ksplit > 1 ? nullptr : p.exps;
    if (inside) prefill_store_pairs_as<FN, false>(to, exps, p.pair_rows, p.N, total, i0, j0, r32, kg);
    else prefill_store_pairs_as<FN, true>(to, exps, p.pair_rows, p.N, total, i0, j0, r32, kg);
}

// FULL: K is a multiple of 128, so no stage is partial or missing and nothing needs masking.
template <int SG, int T, bool FULL>
__global__ void __launch_bounds__(256) mmnb_prefill_kernel(const PrefillArgs p) {
    constexpr int kChunks = T / 32;  // 16-byte chunks of the A slab per thread
    constexpr int kPairs = T / 64;   // (weight tile, lane) pairs per thread, two words each
    constexpr int kF = T / 64;       // 32x32 accumulators per wavefront, per direction
    constexpr int kWT = T / 2;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    uint8_t *lds_a = lds_raw;                    // [2][T * kPPitch]
    uint8_t *lds_w = lds_raw + 2 * T * kPPitch;  // [2][T * kPPitch], row = column of W

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int r32 = lane & 31, kg = lane >> 5;

    // one rectangle of the tile grid per XCD (round-robin workgroup ids), as in the int8 kernel
    const int tiles_x = (p.N + T - 1) / T, tiles_y = (p.M + T - 1) / T;
    const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
    const int rows_per = (tiles_y + p.xcd_rows - 1) / p.xcd_rows, cols_per = (tiles_x + p.xcd_cols - 1) / p.xcd_cols;
    const int ty = (xcd / p.xcd_cols) * rows_per + idx / cols_per, tx = (xcd % p.xcd_cols) * cols_per + idx % cols_per;
    if (idx >= rows_per * cols_per || ty >= tiles_y || tx >= tiles_x) return;
    const int i0 = ty * T, j0 = tx * T;

    // A: chunk c = tid + 256 u -> slab row c / 8, 16-byte column c % 8 (8 halves)
    uint32_t a_off[kChunks], a_lds[kChunks];
    int a_k[kChunks];
#pragma unroll
    for (int u = 0; u < kChunks; u++) {
        const int c = tid + 256 * u, row = c >> 3, kc = c & 7;
        a_off[u] = ((uint32_t)min(i0 + row, p.M - 1) * (uint32_t)p.K + kc * 8) * 2;  // rows past M: clamped, never stored
        a_lds[u] = row * kPPitch + kc * 16;
        a_k[u] = kc * 8;
    }
    // W: pair q = tid + 256 u -> weight tile q / 64 of this column range, lane q % 64 of that tile
    uint32_t w_tile[kPairs], w_lds[kPairs], w_sz[kPairs];
#pragma unroll
    for (int u = 0; u < kPairs; u++) {
        const int q = tid + 256 * u, t = q >> 6, l = q & 63;
        const int nt = min(j0 / 16 + t, p.n_tiles - 1);  // tiles past N: clamped, never stored
        w_tile[u] = (uint32_t)nt * (uint32_t)p.n_cg;
        w_lds[u] = (t * 16 + (l & 15)) * kPPitch + (l >> 4) * 16;
        w_sz[u] = (l & 15);
    }
    struct Regs {
        uint4 a[kChunks];
        uint2 w[kPairs];
        uint32_t z[kPairs];  // two (128 + zp) bytes: for word 0 and word 1 of the stage
    };
    const char *a_base = reinterpret_cast<const char *>(p.A);
    auto load_regs = [&](Regs &r, int stage) {
        const int k0 = stage * kPK;
#pragma unroll
        for (int u = 0; u < kChunks; u++) {
            // K is a multiple of 8: a chunk is inside or outside as a whole; one outside is read from the row's last
            // chunk instead (the load is issued whatever the mask says, and past the last row lies the end of A)
            const bool in = FULL || k0 + a_k[u] < p.K;
            const int back = FULL ? 0 : max(0, k0 + a_k[u] - (p.K - 8));
            const uint4 v = HIPC_LOAD_ALWAYS(reinterpret_cast<const uint4 *>(a_base + a_off[u] + ((size_t)k0 - back) * 2));
            r.a[u] = make_uint4(in ? v.x : 0u, in ? v.y : 0u, in ? v.z : 0u, in ? v.w : 0u);
        }
        const int cg = stage >> 1, half = stage & 1;
#pragma unroll
        for (int u = 0; u < kPairs; u++) {
            const uint32_t tile = w_tile[u] + cg;
            const int l = (tid + 256 * u) & 63;
            r.w[u] = *reinterpret_cast<const uint2 *>(reinterpret_cast<const char *>(p.Wq + (size_t)tile * 64 + l) + half * 8);
            const uint8_t *zb = p.Zb + ((size_t)tile * 16 + w_sz[u]) * SG;
            // the scale group of word j (0..3) of a tile: j for SG 4, j / 2 for SG 2, 0 for SG 1
            if (SG == 4) {
                r.z[u] = *reinterpret_cast<const uint16_t *>(zb + half * 2);  // groups 2 half and 2 half + 1
            } else {
                const uint32_t z = zb[SG == 2 ? half : 0];
                r.z[u] = z | (z << 8);
            }
        }
    };
    // a stage past the end reads clamped addresses and stores zeros for A: it adds nothing
    auto store_regs = [&](const Regs &r, int buf, bool live) {
        const uint32_t keep = FULL || live ? 0xffffffffu : 0u;
#pragma unroll
        for (int u = 0; u < kChunks; u++)
            *reinterpret_cast<uint4 *>(lds_a + buf * T * kPPitch + a_lds[u]) =
                make_uint4(r.a[u].x & keep, r.a[u].y & keep, r.a[u].z & keep, r.a[u].w & keep);
#pragma unroll
        for (int u = 0; u < kPairs; u++) {
            uint8_t *dst = lds_w + buf * T * kPPitch + w_lds[u];
            *reinterpret_cast<uint4 *>(dst) = dequant8(r.w[u].x, r.z[u] & 0xffu);        // k = 8 (l >> 4) .. + 8
            *reinterpret_cast<uint4 *>(dst + 64) = dequant8(r.w[u].y, r.z[u] >> 8);     // k + 32
        }
    };

    f32x16 total[kF][kF], raw[kF][kF];
#pragma unroll
    for (int i = 0; i < kF; i++)
#pragma unroll
        for (int j = 0; j < kF; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) total[i][j][r] = 0.f, raw[i][j][r] = 0.f;

    // scales of the lane's columns (one per accumulator column block)
    uint32_t sc_at[kF];
#pragma unroll
    for (int j = 0; j < kF; j++) {
        const int col = wn * kWT + j * 32 + r32;
        const int nt = min((j0 + col) / 16, p.n_tiles - 1);
        sc_at[j] = ((uint32_t)nt * (uint32_t)p.n_cg * 16 + (col & 15)) * SG;
    }
    auto scale_of = [&](int j, int cg, int g) { return p.Sc[sc_at[j] + (uint32_t)cg * 16 * SG + g]; };
    auto fold = [&](const float (&s)[kF]) {
#pragma unroll
        for (int i = 0; i < kF; i++)
#pragma unroll
            for (int j = 0; j < kF; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) total[i][j][r] = fmaf(raw[i][j][r], s[j], total[i][j][r]);
    };

    // One stage = four k steps of 16. `half` is the stage's parity inside its 128-k weight tile;
    // scale groups end after every second step (SG 4), every stage (SG 2) or every odd stage (SG 1).
    // The scales of a stage are requested before the operand loads of the stage after next, so
    // that waiting for them (loads retire in order) never waits for those.
    float s0[kF], s1[kF];
    auto fetch_scales = [&](int stage, int half) {
        const int cg = stage >> 1;
#pragma unroll
        for (int j = 0; j < kF; j++) {
            if (SG == 4) s0[j] = scale_of(j, cg, half * 2), s1[j] = scale_of(j, cg, half * 2 + 1);
            else if (SG == 2) s1[j] = scale_of(j, cg, half);
            else if (half == 1) s1[j] = scale_of(j, cg, 0);
        }
    };
    // the first product of a quantisation block starts from zero instead of from a cleared register
    f32x16 zero;
#pragma unroll
    for (int r = 0; r < 16; r++) zero[r] = 0.f;
    auto compute = [&](int buf, int half) {
        auto opens_block = [&](int step) { return SG == 4 ? (step & 1) == 0 : SG == 2 ? step == 0 : step == 0 && half == 0; };
        const uint8_t *ba = lds_a + buf * T * kPPitch + (wm * kWT + r32) * kPPitch + kg * 16;
        const uint8_t *bw = lds_w + buf * T * kPPitch + (wn * kWT + r32) * kPPitch + kg * 16;
#pragma unroll
        for (int step = 0; step < 4; step++) {
            f16x8 af[kF], wf[kF];
#pragma unroll
            for (int i = 0; i < kF; i++) af[i] = *reinterpret_cast<const f16x8 *>(ba + i * 32 * kPPitch + step * 32);
#pragma unroll
            for (int j = 0; j < kF; j++) wf[j] = *reinterpret_cast<const f16x8 *>(bw + j * 32 * kPPitch + step * 32);
#pragma unroll
            for (int i = 0; i < kF; i++)
#pragma unroll
                for (int j = 0; j < kF; j++)
                    raw[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], wf[j], opens_block(step) ? zero : raw[i][j], 0, 0, 0);
            if (SG == 4 && step == 1) fold(s0);
            if (step == 3 && (SG != 1 || half == 1)) fold(s1);
        }
    };

    const int nk_all = (p.K + kPK - 1) / kPK;
    const int ks0 = blockIdx.y * p.split_stages, nk = min(nk_all, ks0 + p.split_stages);  // this workgroup's stages
    Regs r0, r1;
    load_regs(r0, ks0);
    load_regs(r1, min(ks0 + 1, nk - 1));
    store_regs(r0, 0, true);
    __syncthreads();
    // two stages per trip and no exit in between, so the memory counters stay exact; with an odd
    // stage count the second half of the last trip multiplies a stage whose A is all zeros
    for (int ks = ks0; ks < nk; ks += 2) {
        fetch_scales(ks, 0);
        load_regs(r0, min(ks + 2, nk - 1));
        compute(0, 0);
        store_regs(r1, 1, ks + 1 < nk);
        __syncthreads();
        fetch_scales(min(ks + 1, nk - 1), 1);
        load_regs(r1, min(ks + 3, nk - 1));
        compute(1, 1);
        store_regs(r0, 0, true);
        __syncthreads();
    }

    prefill_store<kF, kF>(p, total, i0 + wm * kWT, j0 + wn * kWT, r32, kg);
}

// ---- the weight never enters LDS --------------------------------------------------------------------------------
// The B operand of v_mfma_f32_32x32x16_f16 is eight k values of one column per lane, and a 32-bit word of the
// prepacked weight is eight k values of one column: tile lane (c, q) of a 128-k weight tile holds, in its word j,
// k = 32 j + 8 q + 0..7 of column c. The wavefront that multiplies a 32-column block reads the words itself (lane
// (r32, kg) takes tile lanes q = 2 kg and 2 kg + 1 of its column: two 16-byte loads per 128 k), turns a word into
// the operand in registers (nine instructions) and uses it for every 32-row block it owns. A k step (j, h) then
// covers k = 32 j + 16 kg + 8 h + 0..7 -- an order of its own, which only has to be the same for both operands: A
// is read from LDS at that offset. With blocks of 16 (SG 8) the lane takes tile lanes q = kg and 2 + kg instead and the step
// covers k = 32 j + 16 h + 8 kg + 0..7: one block, whose scale costs as many vector instructions as two steps of the
// matrix core take (2e10 operations: 24 us with few tiles, 96 with long k; 2341 and 7845 on vector instructions alone). LDS carries A alone (half the traffic and half the writes of the kernel above,
// and no conversion ahead of a barrier).

// NJ: 32-column blocks per wavefront. 2: a 128x128 tile. 3: a 128x192 tile -- a third less LDS traffic per product,
// and a matrix of 512 x 11008 becomes 232 workgroups for 256 CUs where 128x128 tiles make 344, two of them on every
// third CU.
// MI: 32-row blocks per wavefront. 2 with the tiles above; 1 with NJ 1 is a 64x64 tile for matrices that have too few
// of the large ones (four wavefronts of 32x32: a conversion per product, but many short wavefronts per SIMD).
// KG: groups of four wavefronts per workgroup. With 2 (512 threads) each group takes half of the workgroup's k range
// with LDS buffers of its own, and the two sets of accumulators are added through LDS at the end (128-row tiles: each
// group hands over the 32-row blocks the other one stores; 64-row tiles: the second hands everything to the first).
// For launches that leave wavefront slots of the SIMDs empty: a second wavefront issues while the first waits for
// LDS, a barrier or the matrix core.
// WM, WN: the wavefronts of a group, WM along the rows, WN along the columns.
// TERMS: 2 or 3, the row blocks of a wavefront are the terms of the same 32 f32 rows (see nbits_prefill_f32; 0: rows as they
// are). Two terms' products of a quantisation block go into one set of registers, the low ones first, three terms' into three
// that are joined, and scale x (block sum) is added to a running total. With two terms that is one multiply-add per result
// and block, where accumulators of their own cost each term one (blocks of 32: 8 of 14 vector instructions a product), and
// the total is rounded once per block instead of three times: 2.6e-7 -> 1.3e-7 against 64 bits at 333 x 1152 x 13824, 48.2 -> 38.0 us.
template <int SG, int MI, int NJ, int WM, int WN, int KG, int TERMS, bool FULL>
__global__ void __launch_bounds__(64 * WM * WN * KG, KG > 1 ? 1 : MI * NJ == 1 ? 4 : MI * NJ <= 4 ? 2 : 1) mmnb_prefill_direct_kernel(const PrefillArgs p) {
    static_assert(KG == 1 || KG == 2 || (TERMS && KG == 4), "one or two groups; four of paired rows");
    constexpr int GT = 64 * WM * WN;   // threads of a group
    static_assert(TERMS == 0 || MI % TERMS == 0, "all terms in one wavefront");
    constexpr int PB = TERMS ? MI / TERMS : 1, TS = TERMS == 3 ? 3 : 1;   // blocks of 32 f32 rows, sets of sums of each
    constexpr int T = 32 * MI * WM, TN = 32 * NJ * WN, kChunks = T * 8 / GT, kF = MI, kWT = 32 * MI, kWN = 32 * NJ;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    const int grp = KG > 1 ? (int)threadIdx.x / GT : 0;
    uint8_t *lds_a = lds_raw + grp * 2 * T * kPPitch;  // [KG][2][T * kPPitch]

    const int tid = threadIdx.x % GT;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int r32 = lane & 31, kg = lane >> 5;

    const int tiles_x = (p.N + TN - 1) / TN, tiles_y = (p.M + T - 1) / T;
    const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
    const int rows_per = (tiles_y + p.xcd_rows - 1) / p.xcd_rows, cols_per = (tiles_x + p.xcd_cols - 1) / p.xcd_cols;
    const int ty = (xcd / p.xcd_cols) * rows_per + idx / cols_per, tx = (xcd % p.xcd_cols) * cols_per + idx % cols_per;
    if (idx >= rows_per * cols_per || ty >= tiles_y || tx >= tiles_x) return;
    const int i0 = ty * T, j0 = tx * TN;

    // A: chunk c = tid + GT u -> slab row c / 8, 16-byte column c % 8 (8 halves)
    uint32_t a_off[kChunks], a_lds[kChunks];
    int a_k[kChunks];
#pragma unroll
    for (int u = 0; u < kChunks; u++) {
        const int c = tid + GT * u, row = c >> 3, kc = c & 7;
        a_off[u] = ((uint32_t)min(i0 + row, p.M - 1) * (uint32_t)p.K + kc * 8) * 2;  // rows past M: clamped, never stored
        a_lds[u] = row * kPPitch + kc * 16;
        a_k[u] = kc * 8;
    }
    struct ARegs {
        uint4 a[kChunks];
    };
    const char *a_base = reinterpret_cast<const char *>(p.A);
    auto load_a = [&](ARegs &r, int stage) {
        const int k0 = stage * kPK;
#pragma unroll
        for (int u = 0; u < kChunks; u++) {
            // K is a multiple of 8: a chunk is inside or outside as a whole; one outside is read from the row's last
            // chunk instead (the load is issued whatever the mask says, and past the last row lies the end of A)
            const bool in = FULL || k0 + a_k[u] < p.K;
            const uint32_t back = FULL ? 0u : (uint32_t)max(0, k0 + a_k[u] - (p.K - 8)) * 2u;
            const uint4 v = HIPC_LOAD_ALWAYS(reinterpret_cast<const uint4 *>((a_base + (size_t)k0 * 2) + (a_off[u] - back)));   // (uniform part first: a scalar base and a 32-bit lane offset)
            r.a[u] = make_uint4(in ? v.x : 0u, in ? v.y : 0u, in ? v.z : 0u, in ? v.w : 0u);
        }
    };
    // a stage past the end reads clamped addresses and stores zeros for A: it adds nothing
    auto store_a = [&](const ARegs &r, int buf, bool live) {   // (`live` is the same for the whole workgroup group: a branch, no masks)
        if ((FULL && KG == 1) || live) {
#pragma unroll
            for (int u = 0; u < kChunks; u++) *reinterpret_cast<uint4 *>(lds_a + buf * T * kPPitch + a_lds[u]) = r.a[u];
        } else {
#pragma unroll
            for (int u = 0; u < kChunks; u++) *reinterpret_cast<uint4 *>(lds_a + buf * T * kPPitch + a_lds[u]) = make_uint4(0u, 0u, 0u, 0u);
        }
    };

    // B: column block j of the wavefront = 32 columns = two weight tiles; the lane's column is r32 of the block
    uint32_t b_at[NJ], sc_at[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int nt = min(j0 / 16 + wn * (2 * NJ) + j * 2 + (r32 >> 4), p.n_tiles - 1);  // tiles past N: clamped, never stored
        b_at[j] = (uint32_t)nt * (uint32_t)p.n_cg * 64 + (r32 & 15) + (SG == 8 ? 16 : 32) * kg;
        sc_at[j] = ((uint32_t)nt * (uint32_t)p.n_cg * 16 + (r32 & 15)) * SG;
    }
    struct BRegs {
        uint4 w[NJ][2];
        float s[NJ][SG];
        uint32_t z[NJ][SG == 8 ? 2 : 1];  // SG bytes of 128 + zp
    };
    auto load_b = [&](BRegs &b, int cg) {
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const uint4 *src = (p.Wq + (size_t)cg * 64) + b_at[j];
            b.w[j][0] = src[0];
            b.w[j][1] = src[SG == 8 ? 32 : 16];
            const float *sc = (p.Sc + (size_t)cg * 16 * SG) + sc_at[j];
            const uint8_t *zb = (p.Zb + (size_t)cg * 16 * SG) + sc_at[j];
            if (SG >= 4) {
                const float4 v = *reinterpret_cast<const float4 *>(sc);
                b.s[j][0] = v.x, b.s[j][1 % SG] = v.y, b.s[j][2 % SG] = v.z, b.s[j][3 % SG] = v.w;
                if (SG == 8) {
                    const float4 u = *reinterpret_cast<const float4 *>(sc + 4);
                    b.s[j][4 % SG] = u.x, b.s[j][5 % SG] = u.y, b.s[j][6 % SG] = u.z, b.s[j][7 % SG] = u.w;
                    b.z[j][SG == 8] = *reinterpret_cast<const uint32_t *>(zb + 4);
                }
                b.z[j][0] = *reinterpret_cast<const uint32_t *>(zb);
            } else if (SG == 2) {
                const float2 v = *reinterpret_cast<const float2 *>(sc);
                b.s[j][0] = v.x, b.s[j][1 % SG] = v.y;
                b.z[j][0] = *reinterpret_cast<const uint16_t *>(zb);
            } else {
                b.s[j][0] = sc[0];
                b.z[j][0] = zb[0];
            }
        }
    };

    // One set of accumulators, kept in units of the scale of the quantisation block that is open: when the next
    // block opens they are multiplied by (scale of the old block) / (scale of the new one), the products of the new
    // block add to them as they are, and the store multiplies by the last scale. That is one multiplication per
    // accumulator and block, like adding scale x (block sum) to a running total, without the second set of
    // registers for the block sum (which is what lets a wavefront own three 32-column blocks). A scale of magnitude
    // below 2^-64 (a block of zeros carries 0) counts as 2^-64: the quotient stays finite, and what such a block
    // adds, at most 2^-64 x 15 x sum |a|, is far below one unit of the last place of any result that has a block
    // with a real scale; a column without one is stored as 0.
    f32x16 acc[TERMS ? PB * (1 + TS) : kF][NJ];   // TERMS: [0 .. PB - 1] the running totals, behind them the open block's sums
#pragma unroll
    for (int i = 0; i < (TERMS ? PB : kF); i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    float unit[NJ];   // the scale the accumulators of column block j are in
    bool scaled[NJ];  // the lane's column of block j has met a scale of 2^-64 or more
#pragma unroll
    for (int j = 0; j < NJ; j++) unit[j] = 1.f, scaled[j] = false;
    // the scales of a weight tile's groups -> the factors that take the accumulators from each group to the next
    // (worked out when the trip begins, next to the loads, not in front of the products that wait for them)
    auto scales_to_ratios = [&](BRegs &b) {
        if (TERMS) return;
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int g = 0; g < SG; g++) {
                const bool real = !(fabsf(b.s[j][g]) < 0x1p-64f);
                const float s = real ? b.s[j][g] : 0x1p-64f;
                scaled[j] |= real;
                b.s[j][g] = unit[j] * __builtin_amdgcn_rcpf(s);   // (1 ulp: a relative error of 1e-7 in what was added so far)
                unit[j] = s;
            }
    };
    auto reopen = [&](int j, float ratio) {
#pragma unroll
        for (int i = 0; i < kF; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] *= ratio;
    };

    uint32_t ones = 0x64006400u;   // kept in a vector register (see and_or_1024)
#ifndef HIPC_HOST_MODEL
    asm volatile("" : "+v"(ones));
#endif
    // One stage = 64 k = the k steps (j, h) with j = 2 half + 0 / 1 of the weight tile the stage lies in;
    // a scale group opens at every step (SG 8), every second step (SG 4), every stage (SG 2) or every even stage (SG 1).
    // the zero points of a stage as f16 pairs (with one scale group per weight tile: of the whole tile, made once per trip)
    struct ZeroPairs {
        ZeroPair at[NJ][SG == 8 ? 4 : SG == 4 ? 2 : 1];
    };
    auto zero_pairs = [&](const BRegs &b, int half) {
        ZeroPairs zp;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            if constexpr (SG == 8) {
#pragma unroll
                for (int g = 0; g < 4; g++) zp.at[j][g] = zero_pair((b.z[j][half] >> (8 * g)) & 0xffu);
            } else if constexpr (SG == 4) {
                zp.at[j][0] = zero_pair((b.z[j][0] >> (16 * half)) & 0xffu);
                zp.at[j][1] = zero_pair((b.z[j][0] >> (16 * half + 8)) & 0xffu);
            } else {
                zp.at[j][0] = zero_pair(SG == 2 ? (b.z[j][0] >> (8 * half)) & 0xffu : b.z[j][0]);
            }
        }
        return zp;
    };
    auto compute = [&](const BRegs &b, const ZeroPairs &zp, int buf, int half) {   // (b.s holds ratios by now)
        const uint8_t *ba = lds_a + buf * T * kPPitch + (wm * kWT + r32) * kPPitch + kg * (SG == 8 ? 16 : 32);
#pragma unroll
        for (int step = 0; step < 4; step++) {
            const int word = half * 2 + (step >> 1), h = step & 1;
            const bool opens = SG == 8 ? true : SG == 4 ? h == 0 : SG == 2 ? step == 0 : step == 0 && half == 0;
            const int g = (SG == 8 ? 2 * word + h : SG == 4 ? word : SG == 2 ? half : 0) % SG;
            f16x8 af[kF], wf[NJ];
            if (opens && !TERMS) {
#pragma unroll
                for (int j = 0; j < NJ; j++) reopen(j, b.s[j][g]);
            }
#pragma unroll
            for (int i = 0; i < kF; i++) af[i] = *reinterpret_cast<const f16x8 *>(ba + i * 32 * kPPitch + (step >> 1) * 64 + h * (SG == 8 ? 32 : 16));
#pragma unroll
            for (int j = 0; j < NJ; j++) wf[j] = dequant_operand(word_of(b.w[j][h], word), zp.at[j][SG == 8 ? step : SG == 4 ? step >> 1 : 0], ones);
            if constexpr (TERMS > 0) {
                const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                const bool closes = SG == 8 ? true : SG == 4 ? h == 1 : SG == 2 ? step == 3 : step == 3 && half == 1;
#pragma unroll
                for (int t = TERMS - 1; t >= 0; t--)
#pragma unroll
                    for (int i = 0; i < PB; i++)
#pragma unroll
                        for (int j = 0; j < NJ; j++) {
                            f32x16 &sum = acc[PB + i * TS + (TERMS == 3 ? t : 0)][j];
                            sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i * TERMS + t], wf[j], opens && (TERMS == 3 || t == TERMS - 1) ? zero : sum, 0, 0, 0);
                        }
                if (closes) {
#pragma unroll
                    for (int i = 0; i < PB; i++)
#pragma unroll
                        for (int j = 0; j < NJ; j++)
#pragma unroll
                            for (int r = 0; r < 16; r++) {
                                float sum = acc[PB + i * TS][j][r];
                                if constexpr (TERMS == 3) sum = join_terms(sum, acc[PB + i * TS + 1][j][r], acc[PB + i * TS + 2][j][r]);
                                acc[i][j][r] = fmaf(sum, b.s[j][g], acc[i][j][r]);
                            }
                }
                if (SG >= 4) __builtin_amdgcn_sched_barrier(0);   // (left alone, the blocks of a stage are all opened before one is closed)
            } else {
#pragma unroll
                for (int i = 0; i < kF; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], wf[j], acc[i][j], 0, 0, 0);
            }
        }
    };

    const int nk_all = (p.K + kPK - 1) / kPK;
    const int wg_ks0 = blockIdx.y * p.split_stages, wg_nk = min(nk_all, wg_ks0 + p.split_stages);  // this workgroup's stages (wg_ks0 is even)
    // ... and this group's: with two groups the first takes the larger half of the trips; both run as many trips as
    // the first (the barriers are the workgroup's), the second's last one, if it has one less, on zeros
    const int wg_trips = (wg_nk - wg_ks0 + 1) >> 1, my_trips = (wg_trips + KG - 1) / KG;
    const int ks0 = wg_ks0 + grp * 2 * my_trips, nk = KG == 1 ? wg_nk : min(wg_nk, ks0 + 2 * my_trips);
    const int last = min(wg_nk - 1, max(nk - 1, wg_ks0));   // the last stage whose addresses this group may form
    const int cg_last = last >> 1;
    ARegs r0, r1;
    BRegs bc, bn;
    load_b(bc, min(ks0, last) >> 1);
    load_a(r0, min(ks0, last));
    load_a(r1, min(ks0 + 1, last));
    store_a(r0, 0, ks0 < nk);
    __syncthreads();
    // two stages = one weight tile per trip; with an odd stage count the second half of the last trip multiplies
    // a stage whose A is all zeros. (The fences keep the order written here: left alone, the compiler moves the
    // stores -- and with them the wait for the loads they store -- ahead of the products and the next loads behind
    // them, and every half trip then waits out a whole trip to memory.)
    auto trip = [&](BRegs &bcur, BRegs &bnext, int ks) {
        load_b(bnext, min((ks >> 1) + 1, cg_last));
        load_a(r0, min(ks + 2, last));
        scales_to_ratios(bcur);
        ZeroPairs zp = zero_pairs(bcur, 0);
        __builtin_amdgcn_sched_barrier(0);
        compute(bcur, zp, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        store_a(r1, 1, ks + 1 < nk);
        __syncthreads();
        load_a(r1, min(ks + 3, last));
        if (SG != 1) zp = zero_pairs(bcur, 1);
        __builtin_amdgcn_sched_barrier(0);
        compute(bcur, zp, 1, 1);
        __builtin_amdgcn_sched_barrier(0);
        store_a(r0, 0, ks + 2 < nk);
        __syncthreads();
    };
    for (int t = 0; t < my_trips; t += 2) {   // the two register sets of the weight take turns
        trip(bc, bn, ks0 + 2 * t);
        if (t + 1 < my_trips) trip(bn, bc, ks0 + 2 * t + 2);
    }
    if constexpr (TERMS > 0) {
        // the later groups hand their sums to the first ([group - 1][16-byte piece][thread] in LDS), which adds them and stores
        if constexpr (KG > 1) {
            float4 *slot = reinterpret_cast<float4 *>(lds_raw);
            constexpr int kPieces = PB * NJ * 4;
            if (grp > 0) {
#pragma unroll
                for (int i = 0; i < PB; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++)
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            slot[((grp - 1) * kPieces + (i * NJ + j) * 4 + q) * GT + tid] = make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
            }
            __syncthreads();
            if (grp > 0) return;
#pragma unroll
            for (int g = 0; g < KG - 1; g++)
#pragma unroll
                for (int i = 0; i < PB; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++)
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            const float4 o = slot[(g * kPieces + (i * NJ + j) * 4 + q) * GT + tid];
                            acc[i][j][4 * q] += o.x, acc[i][j][4 * q + 1] += o.y, acc[i][j][4 * q + 2] += o.z, acc[i][j][4 * q + 3] += o.w;
                        }
        }
#pragma unroll
        for (int i = 0; i < PB; i++) {
            f32x16 pair[1][NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++) pair[0][j] = acc[i][j];
            prefill_store_pairs<NJ>(p, pair, (i0 + wm * kWT) / TERMS + 32 * i, j0 + wn * kWN, r32, kg);
        }
    } else {
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int i = 0; i < kF; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] *= scaled[j] ? unit[j] : 0.f;
    if constexpr (KG > 1 && MI == 1) {
        // the later groups hand their accumulators to the first: [group - 1][16-byte piece][thread] in LDS (the A
        // buffers are done with: the last barrier of the loop is behind every read of them), added in group order
        float4 *slot = reinterpret_cast<float4 *>(lds_raw);
        if (grp > 0) {
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    slot[((grp - 1) * NJ * 4 + j * 4 + q) * 256 + tid] = make_float4(acc[0][j][4 * q], acc[0][j][4 * q + 1], acc[0][j][4 * q + 2], acc[0][j][4 * q + 3]);
        }
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int g = 1; g < KG; g++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float4 o = slot[((g - 1) * NJ * 4 + j * 4 + q) * 256 + tid];
                    acc[0][j][4 * q] += o.x, acc[0][j][4 * q + 1] += o.y, acc[0][j][4 * q + 2] += o.z, acc[0][j][4 * q + 3] += o.w;
                }
    }
    if constexpr (MI == 1) {
        prefill_store<kF, NJ>(p, acc, i0 + wm * kWT, j0 + wn * kWN, r32, kg);
    } else if constexpr (KG == 2) {
        // group g keeps row block g and hands the other one over: [group][16-byte piece][thread] in LDS (the A
        // buffers are done with: the last barrier of the loop is behind every read of them)
        float4 *mine = reinterpret_cast<float4 *>(lds_raw) + grp * (NJ * 4 * 256), *theirs = reinterpret_cast<float4 *>(lds_raw) + (grp ^ 1) * (NJ * 4 * 256);
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x16 &v = grp == 0 ? acc[1][j] : acc[0][j];
                mine[(j * 4 + q) * 256 + tid] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
            }
        __syncthreads();
        f32x16 sum[1][NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 o = theirs[(j * 4 + q) * 256 + tid];
                const f32x16 &v = grp == 0 ? acc[0][j] : acc[1][j];
                // (first group's share + second group's share, whichever of them adds)
                sum[0][j][4 * q] = grp == 0 ? v[4 * q] + o.x : o.x + v[4 * q];
                sum[0][j][4 * q + 1] = grp == 0 ? v[4 * q + 1] + o.y : o.y + v[4 * q + 1];
                sum[0][j][4 * q + 2] = grp == 0 ? v[4 * q + 2] + o.z : o.z + v[4 * q + 2];
                sum[0][j][4 * q + 3] = grp == 0 ? v[4 * q + 3] + o.w : o.w + v[4 * q + 3];
            }
        prefill_store<1, NJ>(p, sum, i0 + wm * kWT + grp * 32, j0 + wn * kWN, r32, kg);
    } else {
        prefill_store<kF, NJ>(p, acc, i0 + wm * kWT, j0 + wn * kWN, r32, kg);
    }
    }
}

// Y = f16(sum over splits of the f32 partials), in split order; or the f32 sum itself into Yf32. Four results per
// thread; VEC: the element count is a multiple of four and the rows are aligned for 16-byte loads and one 8- or
// 16-byte store. (static: this file is compiled three times)
template <bool VEC>
static __global__ void __launch_bounds__(256)
mmnb_prefill_reduce_kernel(const float *__restrict__ part, __half *__restrict__ Y, float *__restrict__ Yf32, long total, int ksplit,
                           const int *__restrict__ exps, int N) {   // exps: the f32 result's row r times 2^exps[r] (paired rows; VEC then has N a multiple of four)
    const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= total) return;
    if (VEC) {
        float4 v = *reinterpret_cast<const float4 *>(part + i);
        for (int s = 1; s < ksplit; s++) {
            const float4 u = *reinterpret_cast<const float4 *>(part + (size_t)s * total + i);
            v.x += u.x, v.y += u.y, v.z += u.z, v.w += u.w;
        }
        if (exps) {
            const int e = exps[i / N];
            v = make_float4(ldexpf(v.x, e), ldexpf(v.y, e), ldexpf(v.z, e), ldexpf(v.w, e));
        }
        if (Yf32) {
            *reinterpret_cast<float4 *>(Yf32 + i) = v;
        } else {
            *reinterpret_cast<uint2 *>(Y + i) = make_uint2(two_halves(__float2half(v.x), __float2half(v.y)), two_halves(__float2half(v.z), __float2half(v.w)));
        }
        return;
    }
    for (long j = i; j < min(i + 4, total); j++) {
        float v = part[j];
        for (int s = 1; s < ksplit; s++) v += part[(size_t)s * total + j];
        if (exps) v = ldexpf(v, exps[j / N]);
        if (Yf32) Yf32[j] = v;
        else Y[j] = __float2half(v);
    }
}

namespace {

// the rectangles the tile grid is cut into, one per XCD: how many along the rows (of eight)
[[maybe_unused]] int prefill_xcd_rows(int64_t tiles_x, int64_t tiles_y) {
    int best = 8;
    int64_t best_cost = int64_t(1) << 40;
    for (int r = 1; r <= 8; r *= 2) {
        const int64_t cost = ceil_div(tiles_y, r) + ceil_div(tiles_x, 8 / r);
        if (cost < best_cost) best_cost = cost, best = r;
    }
    return best;
}
// The tile grid cut into one rectangle per XCD, the k split (prefill_split option: 0 never splits k, n > 0 forces n
// ways; unset: as a.ksplit says, or, where that is 0, chosen by shape) with its partials in scratch memory; returns the launch grid in *grid.
int prefill_plan(hipc_ctx *ctx, PrefillArgs &a, int TM, int TN, bool may_split, dim3 *grid) {
    const int tiles_x = (int)ceil_div(a.N, TN), tiles_y = (int)ceil_div(a.M, TM);
    a.xcd_rows = prefill_xcd_rows(tiles_x, tiles_y), a.xcd_cols = 8 / a.xcd_rows;
    const unsigned gx = 8u * (unsigned)(ceil_div(tiles_y, a.xcd_rows) * ceil_div(tiles_x, a.xcd_cols));
    // Too few tiles for the chip: split k over workgroups, as many ways as gives every CU a
    // workgroup, at least 32 stages each (with fewer, the second launch and the partials cost more
    // than the idle CUs: 512 x 2048 x 2560 took 27 us split three ways, 21 us on 64x64 tiles). The
    // partials go through scratch memory.
    const int nk = (int)ceil_div(a.K, kPK);
    int ksplit = 1;
    const int g_prefill_split = ctx->tune.prefill_split;
    if (may_split && g_prefill_split != 0) {
        const int tiles = tiles_x * tiles_y;
        const int asked = g_prefill_split > 0 ? g_prefill_split : a.ksplit;
        ksplit = asked > 0 ? asked : std::min(4, ctx->cu_count / std::max(1, tiles));
        ksplit = std::max(1, std::min(ksplit, asked > 0 ? nk / 2 : nk / 32));
    }
    a.split_stages = (int)(ceil_div(ceil_div(nk, ksplit), 2) * 2);
    a.ksplit = (int)ceil_div(nk, a.split_stages);
    a.Ypart = nullptr;
    const size_t part_bytes = (size_t)a.ksplit * (a.pair_rows > 0 ? a.pair_rows : a.M) * a.N * sizeof(float);
    if (a.ksplit > 1 && !scratch_fits(ctx, 0, part_bytes)) a.split_stages = (int)(ceil_div(nk, 2) * 2), a.ksplit = 1;
    if (a.ksplit > 1) {
        void *part = nullptr;
        if (int rc = scratch_get(ctx, 0, part_bytes, &part)) return rc;
        a.Ypart = static_cast<float *>(part);
    }
    *grid = dim3(gx, (unsigned)a.ksplit);
    return HIPC_OK;
}
// the second launch of a k split
int prefill_join_splits(hipc_ctx *ctx, const PrefillArgs &a) {
    if (a.ksplit > 1) {
        const long total = (long)(a.pair_rows > 0 ? a.pair_rows : a.M) * a.N;
        const bool vec = (a.exps ? a.N % 4 == 0 : total % 4 == 0) && (a.Yf32 ? aligned(a.Yf32, 16) : aligned(a.Y, 8));
        if (vec)
            hipLaunchKernelGGL((mmnb_prefill_reduce_kernel<true>), dim3((unsigned)ceil_div(total, 1024)), dim3(256), 0, ctx->stream, a.Ypart, a.Y, a.Yf32, total, a.ksplit, a.exps, a.N);
        else
            hipLaunchKernelGGL((mmnb_prefill_reduce_kernel<false>), dim3((unsigned)ceil_div(total, 1024)), dim3(256), 0, ctx->stream, a.Ypart, a.Y, a.Yf32, total, a.ksplit, a.exps, a.N);
        HIPC_LAUNCHED(ctx);
    }
    return HIPC_OK;
}

// both operands through LDS
template <int SG, int T>
int prefill_launch_tile(hipc_ctx *ctx, PrefillArgs a) {
    const bool full = a.K % (2 * kPK) == 0;
    static bool lds_allowed[2][kMaxDevices] = {};
    if (int rc = full ? allow_dynamic_lds(ctx, mmnb_prefill_kernel<SG, T, true>, prefill_lds(T), lds_allowed[1])
                      : allow_dynamic_lds(ctx, mmnb_prefill_kernel<SG, T, false>, prefill_lds(T), lds_allowed[0]))
        return rc;
    dim3 grid;
    if (int rc = prefill_plan(ctx, a, T, T, T == 128, &grid)) return rc;
    if (full)
        hipLaunchKernelGGL((mmnb_prefill_kernel<SG, T, true>), grid, dim3(256), prefill_lds(T), ctx->stream, a);
    else
        hipLaunchKernelGGL((mmnb_prefill_kernel<SG, T, false>), grid, dim3(256), prefill_lds(T), ctx->stream, a);
    HIPC_LAUNCHED(ctx);
    return prefill_join_splits(ctx, a);
}

// the weight from memory into the operand registers; A alone in LDS
template <int SG, int MI, int NJ, int WM, int WN, int KG, int TERMS>
int prefill_launch_direct_groups(hipc_ctx *ctx, const PrefillArgs &a, dim3 grid) {
    const bool full = a.K % (2 * kPK) == 0;
    constexpr int T = 32 * MI * WM, kThreads = 64 * WM * WN * KG;
    // one group: at most 36 KB, inside the limit that needs no permission; more: their A buffers, then the hand-over
    constexpr size_t hand_over = TERMS ? (size_t)(KG - 1) * (MI / std::max(1, TERMS)) * NJ * 4 * (64 * WM * WN) * 16 : (size_t)(MI == 2 ? 4 : 2 * (KG - 1)) * NJ * 4 * 128 * 16;
    constexpr size_t lds = KG == 1 ? prefill_lds(T) / 2 : std::max(KG * prefill_lds(T) / 2, hand_over);
    if (KG > 1 && lds > 64 * 1024) {
        static bool lds_allowed[2][kMaxDevices] = {};
        if (int rc = full ? allow_dynamic_lds(ctx, mmnb_prefill_direct_kernel<SG, MI, NJ, WM, WN, KG, TERMS, true>, lds, lds_allowed[1])
                          : allow_dynamic_lds(ctx, mmnb_prefill_direct_kernel<SG, MI, NJ, WM, WN, KG, TERMS, false>, lds, lds_allowed[0]))
            return rc;
    }
    if (full)
        hipLaunchKernelGGL((mmnb_prefill_direct_kernel<SG, MI, NJ, WM, WN, KG, TERMS, true>), grid, dim3(kThreads), lds, ctx->stream, a);
    else
        hipLaunchKernelGGL((mmnb_prefill_direct_kernel<SG, MI, NJ, WM, WN, KG, TERMS, false>), grid, dim3(kThreads), lds, ctx->stream, a);
    HIPC_LAUNCHED(ctx);
    return HIPC_OK;
}
template <int SG, int MI, int NJ, int WM, int WN, int TERMS>
int prefill_launch_direct(hipc_ctx *ctx, PrefillArgs a) {
    constexpr int T = 32 * MI * WM, TN = 32 * NJ * WN;
    dim3 grid;
    // (64-row tiles split a long k as the larger ones do when even they are too few: f16 100 x 8192 x 1024, 32 tiles,
    // 32.0 us as they are, 13.7 us four ways)
    if (int rc = prefill_plan(ctx, a, T, TN, true, &grid)) return rc;
    const int trips = (a.split_stages + 1) / 2, forced = ctx->tune.prefill_groups;
    const long wgs = (long)ceil_div(a.M, T) * ceil_div(a.N, TN) * a.ksplit;
    // Two k groups per workgroup (four of paired rows where a group is two wavefronts) when the launch leaves the second
    // wavefront slot of the SIMDs empty (128-row tiles and 96x128 ones of three terms: no more workgroups than CUs, 400 x 1152 x 4096
    // in three terms 26.5 us with one group, 33.4 with two; 64-row tiles: no more than two per CU,
    // 512 x 2048 x 2560: 15.9 against 16.9 us, four groups, 18.3 us, cost more in prologues than they hide) and every group
    // gets two trips or more; prefill_groups 1 / 2 forces the choice. (three column blocks and two groups leave no register
    // for more than one scale per weight tile)
    constexpr int kGroups = WM * WN == 2 ? 4 : 2;
    if constexpr (NJ < 3 || SG == 1) {
        if (forced == 1 ? false : forced == 2 ? true : wgs <= (T < 128 && !(TERMS == 3 && WM * WN == 4) ? 2 : 1) * ctx->cu_count && trips >= 2 * kGroups) {
            if (int rc = prefill_launch_direct_groups<SG, MI, NJ, WM, WN, kGroups, TERMS>(ctx, a, grid)) return rc;
            return prefill_join_splits(ctx, a);
        }
    }
    if (int rc = prefill_launch_direct_groups<SG, MI, NJ, WM, WN, 1, TERMS>(ctx, a, grid)) return rc;
    return prefill_join_splits(ctx, a);
}

}  // namespace

// This file is compiled three times, since where the compiler keeps matrix-core accumulators is a switch of the whole
// compilation. HIPC_PREFILL_WIDE: the kernel that keeps the weight out of LDS, and the 128x128 tiles of the other one, with
// accumulators in ordinary vector registers (the block scales then multiply them without copies out of the accumulation file:
// 48.5 -> 44.7 us for 512 x 2048 x 11008). HIPC_PREFILL_TERMS: the instances for rows in terms, in ordinary registers, too, and without
// sinking (see the Makefile). Without either: the 64x64 tiles with both operands in LDS, which are faster with the accumulation
// file (80.6 against 87.9 us for 512 x 11008 x 2048), the rules and the entry points.
int prefill_launch_wide(hipc_ctx *ctx, const PrefillArgs &a, int SG, int tile);
int prefill_launch_terms(hipc_ctx *ctx, const PrefillArgs &a, int SG, int tile);

#ifdef HIPC_PREFILL_WIDE

int prefill_launch_wide(hipc_ctx *ctx, const PrefillArgs &a, int SG, int tile) {
    if (tile == 192) switch (SG) {
            case 4: return prefill_launch_direct<4, 2, 3, 2, 2, 0>(ctx, a);
            case 2: return prefill_launch_direct<2, 2, 3, 2, 2, 0>(ctx, a);
            default: return prefill_launch_direct<1, 2, 3, 2, 2, 0>(ctx, a);
        }
    if (tile == 64) switch (SG) {
            case 8: return prefill_launch_direct<8, 1, 1, 2, 2, 0>(ctx, a);
            case 4: return prefill_launch_direct<4, 1, 1, 2, 2, 0>(ctx, a);
            case 2: return prefill_launch_direct<2, 1, 1, 2, 2, 0>(ctx, a);
            default: return prefill_launch_direct<1, 1, 1, 2, 2, 0>(ctx, a);
        }
    if (ctx->tune.prefill_direct != 0 || SG == 8) switch (SG) {
            case 8: return prefill_launch_direct<8, 2, 2, 2, 2, 0>(ctx, a);
            case 4: return prefill_launch_direct<4, 2, 2, 2, 2, 0>(ctx, a);
            case 2: return prefill_launch_direct<2, 2, 2, 2, 2, 0>(ctx, a);
            default: return prefill_launch_direct<1, 2, 2, 2, 2, 0>(ctx, a);
        }
    switch (SG) {
        case 4: return prefill_launch_tile<4, 128>(ctx, a);
        case 2: return prefill_launch_tile<2, 128>(ctx, a);
        default: return prefill_launch_tile<1, 128>(ctx, a);
    }
}

#elif defined(HIPC_PREFILL_TERMS)

int prefill_launch_terms(hipc_ctx *ctx, const PrefillArgs &a, int SG, int tile) {
    if (a.terms == 3) {   // (tile: 64 -> 96x64, else 96x128)
        if (tile == 64) switch (SG) {
                case 4: return prefill_launch_direct<4, 3, 1, 1, 2, 3>(ctx, a);
                case 2: return prefill_launch_direct<2, 3, 1, 1, 2, 3>(ctx, a);
                default: return prefill_launch_direct<1, 3, 1, 1, 2, 3>(ctx, a);
            }
        switch (SG) {
            case 4: return prefill_launch_direct<4, 3, 1, 1, 4, 3>(ctx, a);
            case 2: return prefill_launch_direct<2, 3, 1, 1, 4, 3>(ctx, a);
            default: return prefill_launch_direct<1, 3, 1, 1, 4, 3>(ctx, a);
        }
    }
    // (tile: 64 -> 64x64, 128 -> 64x128, 192 -> the larger ones of prefill_pair_tile)
    if (tile == 192) switch (SG) {
            case 4: return prefill_launch_direct<4, 4, 1, 1, 4, 2>(ctx, a);
            case 2: return prefill_launch_direct<2, 2, 2, 1, 4, 2>(ctx, a);
            case 1: return prefill_launch_direct<1, 2, 2, 1, 4, 2>(ctx, a);
        }
    if (tile == 64) switch (SG) {
            case 4: return prefill_launch_direct<4, 2, 1, 1, 2, 2>(ctx, a);
            case 2: return prefill_launch_direct<2, 2, 1, 1, 2, 2>(ctx, a);
            default: return prefill_launch_direct<1, 2, 1, 1, 2, 2>(ctx, a);
        }
    switch (SG) {
        case 4: return prefill_launch_direct<4, 2, 1, 1, 4, 2>(ctx, a);
        case 2: return prefill_launch_direct<2, 2, 1, 1, 4, 2>(ctx, a);
        default: return prefill_launch_direct<1, 2, 1, 1, 4, 2>(ctx, a);
    }
}

#else

namespace {

// Tiles of rows in two terms: 64x64 where there are few tiles, k is not long enough to split three ways over workgroups and no
// XCD gets more workgroups than it has CUs (400 x 1152 x 1152, 234 tiles of which one XCD gets 35: 21.0 us, 15.5 on 64x128); else
// 64x128, or the larger ones where these take fewer rounds of workgroups times stages: 128x128 (64 f32 rows to a wavefront)
// with four scales per weight tile, 64x256 with one or two. They do two 64x128 tiles' work in 15/16 of the time. Measured,
// 64x64 / 64x128 / larger, us: 333 x 1152 x 13824 in blocks of 32 44.0 / 37.1 / 42.1, 1000 x 2048 x 4096 62.1 / 53.1 / 50.4,
// 100 x 2048 x 2560 14.8 / 18.6 / 28.5, 100 x 6912 x 1152 33.3 / 25.2 / 35.7, 300 x 11008 x 2048 90.2 / 72.1 / 54.9; in blocks
// of 128 600 x 8192 x 1024 60.9 / 48.3 / 38.4.
template <int SG>
int prefill_pair_tile(hipc_ctx *ctx, const PrefillArgs &a) {
    const int64_t cus = std::max(1, ctx->cu_count), rows64 = ceil_div(a.M, 64), stages = ceil_div(a.K, kPK);
    const int64_t most = ctx->tune.prefill_split == 0 ? 1 : std::max<int64_t>(1, std::min<int64_t>(4, stages / 32));   // (see prefill_plan)
    const int64_t mid = rows64 * ceil_div(a.N, 128), large = SG <= 2 ? rows64 * ceil_div(a.N, 256) : ceil_div(a.M, 128) * ceil_div(a.N, 128);
    const int64_t cols64 = ceil_div(a.N, 64), xcd_rows = prefill_xcd_rows(cols64, rows64);
    const int64_t per_xcd = ceil_div(rows64, xcd_rows) * ceil_div(cols64, 8 / xcd_rows) * std::max<int64_t>(1, std::min(most, cus / (rows64 * cols64)));
    if (mid <= cus / 2 && most < 3 && 8 * per_xcd <= cus) return 64;
    auto cost = [&](int64_t tiles) {
        const int64_t ways = std::max<int64_t>(1, std::min(most, cus / tiles));
        return ceil_div(tiles * ways, cus) * ceil_div(stages, ways);
    };
    return 2 * 15 * cost(large) < 16 * cost(mid) ? 192 : 128;
}
// Rows in three terms: tiles of 96x64 or 96x128, and how many ways k is split over workgroups, by an estimate of the call in us:
// a workgroup's stages times the rounds of workgroups on the XCD that has most of them (less than proportionally, since rounds overlap;
// 96x64 tiles of one group go two to a CU), and the join of a split's partials. Its constants are a fit to calls of 40 to 1000
// rows, k 1152 to 11008, n 1024 to 6912; over 133 of them what it picks is 1 % behind the best of the eight on average. Measured, us, each
// term's rows by themselves through the kernel for f16 rows / the fewest rounds, split only where that leaves CUs idle / this:
// 64 x 1152 x 1152 in blocks of 32 14.7 / 16.1 / 13.1, 200 x 6912 x 1152 in blocks of 64 43.3 / 47.4 / 39.1, 400 x 4096 x 1152 in blocks
// of 64 41.3 / 54.4 / 35.1, 1000 x 11008 x 1152 in blocks of 32 154 / 187 / 135, 400 x 6912 x 4096 in blocks of 32 166 / 123 / 107; 64 x 11008 x 1024
// in blocks of 128 stays at 28.6 / 33.6 / 30.9.
template <int SG>
int prefill_pinned_tile(hipc_ctx *ctx, const PrefillArgs &a, int *ways_out) {
    const int64_t cus = std::max(1, ctx->cu_count), xcd_cus = std::max<int64_t>(1, cus / 8), stages = ceil_div(a.K, kPK), rows = ceil_div(a.M, 96);
    const double scales = SG == 4 ? 1.07 : SG == 2 ? 1. : 0.85, values = (double)a.pair_rows * a.N;
    const int most = ctx->tune.prefill_split == 0 ? 1 : 4;
    int tile = 128;
    double best = 1e30;
    *ways_out = 1;
    for (int T : {64, 128}) {
        const int64_t cols = ceil_div(a.N, T);
        const int r = prefill_xcd_rows(cols, rows);
        for (int asked = 1; asked <= most; asked++) {   // (as prefill_plan and prefill_launch_direct will have it)
            const int64_t split = std::max<int64_t>(1, std::min<int64_t>(asked, stages / 2)), own = ceil_div(ceil_div(stages, split), 2) * 2, ways = ceil_div(stages, own);
            const bool groups = rows * cols * ways <= (T == 64 ? 2 : 1) * cus && (own + 1) / 2 >= (T == 64 ? 8 : 4);
            const double load = (double)(ceil_div(rows, r) * ceil_div(cols, 8 / r) * ways) / xcd_cus;
            const double rounds = std::max(1., T == 64 && !groups ? std::ceil(2 * load) / 2 : std::ceil(load));
            const double first = T == 64 ? (groups ? 0.33 : 0.39) : 0.48, more = T == 64 ? (groups ? 0.39 : 0.33) : groups ? 0.48 : 0.4;
            double us = (T == 64 ? (groups ? 10.23 : 9.46) : groups ? 8.36 : 7.23) + scales * own * (first + more * (rounds - 1));
            if (ways > 1) us += 2.34 + 1.35e-6 * ways * values;
            if (us < best) best = us, tile = T, *ways_out = asked;
        }
    }
    return tile;
}
template <int SG>
int prefill_launch(hipc_ctx *ctx, const PrefillArgs &a) {
    const int forced = ctx->tune.prefill_tile, g_prefill_split = ctx->tune.prefill_split;
    if (a.pair_rows > 0) {
        PrefillArgs b = a;
        const int tile = forced == 64 || forced == 128 || forced == 192 ? forced : a.terms == 3 ? prefill_pinned_tile<SG>(ctx, a, &b.ksplit) : prefill_pair_tile<SG>(ctx, a);
        return prefill_launch_terms(ctx, b, SG, tile);
    }
    // 128-row tiles when they give every CU a workgroup, directly or (long k) with k split over up
    // to four workgroups per tile; else 64x64
    const int64_t rows128 = ceil_div(a.M, 128), tiles128 = rows128 * ceil_div(a.N, 128), tiles192 = rows128 * ceil_div(a.N, 192);
    const int nk = (int)ceil_div(a.K, kPK);
    const bool by_split = g_prefill_split != 0 && tiles128 * std::min<int64_t>(4, nk / 32) >= 192;
    int tile = tiles128 >= 256 || by_split ? 128 : 64;
    // 128x192 where that shortens the longest queue of a SIMD: rounds of workgroups over the CUs times the wavefront's
    // 32-column blocks (512 x 11008: 344 tiles of 128x128 are two rounds of 2, 232 of 128x192 one round of 3)
    const int64_t cus = std::max(1, ctx->cu_count);
    if (SG != 8 && tile == 128 && tiles128 >= 256 && ctx->tune.prefill_direct != 0 && ceil_div(tiles192, cus) * 3 < ceil_div(tiles128, cus) * 2) tile = 192;
    if (forced == 64 || forced == 128 || (forced == 192 && SG != 8 && ctx->tune.prefill_direct != 0)) tile = forced;
    if constexpr (SG == 8) return prefill_launch_wide(ctx, a, SG, tile);   // (blocks of 16: one kernel; three column blocks leave no registers for the scales)
    else return tile == 64 && ctx->tune.prefill_direct == 0 ? prefill_launch_tile<SG, 64>(ctx, a) : prefill_launch_wide(ctx, a, SG, tile);
}

}  // namespace

bool nbits_prefill_takes(const void *A, const hipc_nbits_weight *w, int64_t M) {
    return M > 16 && w->K % 8 == 0 && aligned(A, 16) && M * w->K < (int64_t(1) << 31);
}

int nbits_prefill(hipc_ctx *ctx, const void *A, const hipc_nbits_weight *w, void *Y, int64_t M) {
    HIPC_REFUSE(ctx, !nbits_prefill_takes(A, w, M), "MatMulNBits prefill: shape or alignment not taken by the tiled kernel");
    PrefillArgs a{};
    a.A = static_cast<const __half *>(A), a.Wq = w->Wq, a.Sc = w->Sc, a.Zb = w->Zb, a.Y = static_cast<__half *>(Y);
    a.M = (int)M, a.K = (int)w->K, a.N = (int)w->N, a.n_tiles = w->n_tiles, a.n_cg = w->n_cg;
    switch (w->SG) {
        case 8: return prefill_launch<8>(ctx, a);
        case 4: return prefill_launch<4>(ctx, a);
        case 2: return prefill_launch<2>(ctx, a);
        default: return prefill_launch<1>(ctx, a);
    }
}

// Rows of f32 activations for the f16 matrix cores: row m becomes two f16 rows, hi = f16(a 2^-e) and
// lo = f16(a 2^-e - hi) (22 significant bits), with 2^e the row's own power of two that brings its
// largest magnitude into [2^14, 2^15) -- exact, and no value of the row leaves the f16 range. The rows
// are stored as A2[m] = hi, A2[M + m] = lo; one workgroup per row. PAIRED: 32 rows of high terms are followed by the
// 32 rows of each further term (row m of two: hi at 64 (m / 32) + m % 32, lo 32 rows on), the grid covers a multiple of 32
// rows and the rows past M are zeros.
template <bool PAIRED, int TERMS = 2>   // TERMS 1: the high terms alone, M rows; 3: a third, unpaired in rows 2 M + m (see split_terms)
static __global__ void __launch_bounds__(256)
mmnb_prefill_split_rows_kernel(const float *__restrict__ A, int M, int K, __half *__restrict__ A2, int *__restrict__ exps) {
    __shared__ float red[4];
    const int m = blockIdx.x, tid = threadIdx.x;
    const size_t step = PAIRED ? 32 : (size_t)M;   // rows from a term to the next
    const size_t hi_at = PAIRED ? (size_t)(32 * TERMS * (m >> 5) + (m & 31)) : (size_t)m, lo_at = hi_at + step;
    if (PAIRED && m >= M) {
#pragma unroll
        for (int t = 0; t < TERMS; t++) {
            uint4 *to = reinterpret_cast<uint4 *>(A2 + (hi_at + t * step) * K);
            for (int c = tid; c < K / 8; c += 256) to[c] = make_uint4(0u, 0u, 0u, 0u);
        }
        return;
    }
    const float4 *row = reinterpret_cast<const float4 *>(A + (size_t)m * K);   // (K is a multiple of 8 and A is aligned: see nbits_prefill_f32_takes)
    const int nv = K / 4;
    constexpr int kHeld = 4;   // 16-byte pieces a thread keeps between the two passes: rows up to 4096 values are read once
    float4 held[kHeld];
    float mx = 0.f;
#pragma unroll
    for (int u = 0; u < kHeld; u++) {
        const int c = tid + 256 * u;
        held[u] = c < nv ? row[c] : make_float4(0.f, 0.f, 0.f, 0.f);
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(held[u].x), fabsf(held[u].y)), fmaxf(fabsf(held[u].z), fabsf(held[u].w))));   // (a NaN does not raise the maximum: it passes through below)
    }
    for (int c = tid + 256 * kHeld; c < nv; c += 256) {
        const float4 v = row[c];
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const int e = row_exponent(__float_as_uint(mx));
    if (tid == 0) exps[m] = e;
    const float down = two_to_minus(e);
    uint2 *hi_row = reinterpret_cast<uint2 *>(A2 + hi_at * K), *lo_row = reinterpret_cast<uint2 *>(A2 + lo_at * K);
    auto split4 = [&](const float4 &v, int c) {
        const float a[4] = {v.x * down, v.y * down, v.z * down, v.w * down};
        _Float16 t[4][TERMS];
#pragma unroll
        for (int i = 0; i < 4; i++) split_terms<TERMS>(a[i], t[i]);
        const auto piece = [&](int e) {
            return make_uint2(two_halves(__builtin_bit_cast(__half, t[0][e]), __builtin_bit_cast(__half, t[1][e])),
                              two_halves(__builtin_bit_cast(__half, t[2][e]), __builtin_bit_cast(__half, t[3][e])));
        };
        hi_row[c] = piece(0);
        if constexpr (TERMS >= 2) lo_row[c] = piece(1);
        if constexpr (TERMS == 3) lo_row[c + step * (K / 4)] = piece(2);
    };
#pragma unroll
    for (int u = 0; u < kHeld; u++)
        if (tid + 256 * u < nv) split4(held[u], tid + 256 * u);
    for (int c = tid + 256 * kHeld; c < nv; c += 256) split4(row[c], c);
}
// Y[m] = (P[m] + P[M + m]) 2^e[m], or with three terms join_terms(P[m], P[M + m], P[2 M + m]) 2^e[m]
template <bool VEC>   // VEC: N is a multiple of four and Y is aligned for 16-byte stores
static __global__ void __launch_bounds__(256)
mmnb_prefill_join_rows_kernel(const float *__restrict__ P, const int *__restrict__ exps, int M, int N, float *__restrict__ Y, int terms) {
    const long i = ((long)blockIdx.x * 256 + threadIdx.x) * (VEC ? 4 : 1), plane = (long)M * N;
    if (i >= plane) return;
    const int e = exps[(int)(i / N)];
    if (VEC) {
        const float4 a = *reinterpret_cast<const float4 *>(P + i), b = *reinterpret_cast<const float4 *>(P + i + plane);
        float4 v = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
        if (terms == 3) {
            const float4 c = *reinterpret_cast<const float4 *>(P + i + 2 * plane);
            v = make_float4(join_terms(a.x, b.x, c.x), join_terms(a.y, b.y, c.y), join_terms(a.z, b.z, c.z), join_terms(a.w, b.w, c.w));
        }
        *reinterpret_cast<float4 *>(Y + i) = make_float4(ldexpf(v.x, e), ldexpf(v.y, e), ldexpf(v.z, e), ldexpf(v.w, e));
    } else {
        Y[i] = ldexpf(terms == 3 ? join_terms(P[i], P[i + plane], P[i + 2 * plane]) : P[i] + P[i + plane], e);
    }
}

// Many rows of f32 activations: each row as one to three f16 rows (11, 22 or all 24 bits) through the same tiled kernel, against
// one pass over the whole weight per 16 rows on the decode kernel. With the kernel that keeps the weight out of LDS the terms
// of a row are row blocks of one wavefront, which adds them and puts the rows' powers of two back itself; else the kernel
// writes a row of f32 results per term and a last launch adds them.
bool nbits_prefill_f32_takes(const void *A, const hipc_nbits_weight *w, int64_t M) {
    return M > 32 && w->K % 8 == 0 && aligned(A, 16) && (3 * M + 96) * w->K < (int64_t(1) << 31) && 3 * M * w->N < (int64_t(1) << 31);
}

namespace {
// the exponents of M rows, padded, in front of the f16 rows
size_t split_exps_bytes(int64_t M) { return ((size_t)M * sizeof(int) + 255) & ~(size_t)255; }
// the kernel that keeps the weight out of LDS takes all terms of a row in one wavefront; for the kernel with both operands in
// LDS, and for blocks of 16 (whose sums and scales would not fit the registers: 130 x 2048 x 2560 58.6 against 30.1 us): `terms`
// M rows, and a launch that adds them
bool split_paired(hipc_ctx *ctx, const hipc_nbits_weight *w, int terms) { return terms >= 2 && w->SG != 8 && ctx->tune.prefill_direct != 0; }
}  // namespace
size_t nbits_split_bytes(int64_t rows, int64_t M, int64_t K) { return (size_t)rows * K * sizeof(__half) + split_exps_bytes(M); }

bool nbits_prefill_f32_fits(hipc_ctx *ctx, const hipc_nbits_weight *w, int64_t M, int terms) {
    const bool paired = split_paired(ctx, w, terms);
    if (!scratch_fits(ctx, 2, nbits_split_bytes(paired ? 32 * terms * ceil_div(M, 32) : terms * M, M, w->K))) return false;
    return terms == 1 || paired || scratch_fits(ctx, 3, (size_t)terms * M * w->N * sizeof(float));
}

int nbits_prefill_f32(hipc_ctx *ctx, const void *A, const hipc_nbits_weight *w, void *Y, int64_t M, int terms) {
    HIPC_REFUSE(ctx, !nbits_prefill_f32_takes(A, w, M), "MatMulNBits prefill: shape or alignment not taken by the tiled kernel");
    if (terms == 1) {
        // one f16 term per row (11 bits beside the row's own power of two): M rows through the kernel, which scales
        // the rows of its f32 result back itself (after a k split, the reduce launch does)
        void *split = nullptr;
        if (int rc = scratch_get(ctx, 2, nbits_split_bytes(M, M, w->K), &split)) return rc;
        __half *A1 = reinterpret_cast<__half *>(static_cast<char *>(split) + split_exps_bytes(M));
        int *exps = static_cast<int *>(split);
        hipLaunchKernelGGL((mmnb_prefill_split_rows_kernel<false, 1>), dim3((unsigned)M), dim3(256), 0, ctx->stream, static_cast<const float *>(A), (int)M, (int)w->K, A1, exps);
        HIPC_LAUNCHED(ctx);
        PrefillArgs a{};
        a.A = A1, a.Wq = w->Wq, a.Sc = w->Sc, a.Zb = w->Zb, a.Y = nullptr, a.Yf32 = static_cast<float *>(Y), a.exps = exps;
        a.M = (int)M, a.K = (int)w->K, a.N = (int)w->N, a.n_tiles = w->n_tiles, a.n_cg = w->n_cg;
        switch (w->SG) {
            case 8: return prefill_launch<8>(ctx, a);
            case 4: return prefill_launch<4>(ctx, a);
            case 2: return prefill_launch<2>(ctx, a);
            default: return prefill_launch<1>(ctx, a);
        }
    }
    const bool paired = split_paired(ctx, w, terms);
    const int64_t rows2 = paired ? 32 * terms * ceil_div(M, 32) : terms * M;
    void *split = nullptr, *sums = nullptr;
    if (int rc = scratch_get(ctx, 2, nbits_split_bytes(rows2, M, w->K), &split)) return rc;
    if (!paired)
        if (int rc = scratch_get(ctx, 3, (size_t)terms * M * w->N * sizeof(float), &sums)) return rc;
    __half *A2 = reinterpret_cast<__half *>(static_cast<char *>(split) + split_exps_bytes(M));
    int *exps = static_cast<int *>(split);
    if (paired && terms == 3)
        hipLaunchKernelGGL((mmnb_prefill_split_rows_kernel<true, 3>), dim3((unsigned)(rows2 / 3)), dim3(256), 0, ctx->stream, static_cast<const float *>(A), (int)M, (int)w->K, A2, exps);
    else if (paired)
        hipLaunchKernelGGL((mmnb_prefill_split_rows_kernel<true, 2>), dim3((unsigned)(rows2 / 2)), dim3(256), 0, ctx->stream, static_cast<const float *>(A), (int)M, (int)w->K, A2, exps);
    else if (terms == 3)
        hipLaunchKernelGGL((mmnb_prefill_split_rows_kernel<false, 3>), dim3((unsigned)M), dim3(256), 0, ctx->stream, static_cast<const float *>(A), (int)M, (int)w->K, A2, exps);
    else
        hipLaunchKernelGGL((mmnb_prefill_split_rows_kernel<false, 2>), dim3((unsigned)M), dim3(256), 0, ctx->stream, static_cast<const float *>(A), (int)M, (int)w->K, A2, exps);
    HIPC_LAUNCHED(ctx);
    PrefillArgs a{};
    a.A = A2, a.Wq = w->Wq, a.Sc = w->Sc, a.Zb = w->Zb, a.Y = nullptr, a.Yf32 = static_cast<float *>(paired ? Y : sums);
    a.M = (int)rows2, a.K = (int)w->K, a.N = (int)w->N, a.n_tiles = w->n_tiles, a.n_cg = w->n_cg;
    if (paired) a.exps = exps, a.pair_rows = (int)M, a.terms = terms;
    int rc;
    switch (w->SG) {
        case 8: rc = prefill_launch<8>(ctx, a); break;
        case 4: rc = prefill_launch<4>(ctx, a); break;
        case 2: rc = prefill_launch<2>(ctx, a); break;
        default: rc = prefill_launch<1>(ctx, a); break;
    }
    if (rc != HIPC_OK || paired) return rc;
    const long total = (long)M * w->N;
    if (w->N % 4 == 0 && aligned(Y, 16))
        hipLaunchKernelGGL((mmnb_prefill_join_rows_kernel<true>), dim3((unsigned)ceil_div(total, 1024)), dim3(256), 0, ctx->stream, static_cast<const float *>(sums), exps, (int)M, (int)w->N, static_cast<float *>(Y), terms);
    else
        hipLaunchKernelGGL((mmnb_prefill_join_rows_kernel<false>), dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, ctx->stream, static_cast<const float *>(sums), exps, (int)M, (int)w->N, static_cast<float *>(Y), terms);
    HIPC_LAUNCHED(ctx);
    return HIPC_OK;
}

// up to 64 rows of f32, split here and multiplied as f16 rows by the kernel for a few rows (matmul_nbits_rows.hip)
int nbits_rows_f32_split(hipc_ctx *ctx, const void *A, const hipc_nbits_weight *w, void *Y, int M, int terms) {
    void *split = nullptr;
    if (int rc = scratch_get(ctx, 2, nbits_split_bytes(terms * M, M, w->K), &split)) return rc;
    __half *A2 = reinterpret_cast<__half *>(static_cast<char *>(split) + split_exps_bytes(M));
    int *exps = static_cast<int *>(split);
    if (terms == 1)
        hipLaunchKernelGGL((mmnb_prefill_split_rows_kernel<false, 1>), dim3((unsigned)M), dim3(256), 0, ctx->stream, static_cast<const float *>(A), M, (int)w->K, A2, exps);
    else if (terms == 3)
        hipLaunchKernelGGL((mmnb_prefill_split_rows_kernel<false, 3>), dim3((unsigned)M), dim3(256), 0, ctx->stream, static_cast<const float *>(A), M, (int)w->K, A2, exps);
    else
        hipLaunchKernelGGL((mmnb_prefill_split_rows_kernel<false, 2>), dim3((unsigned)M), dim3(256), 0, ctx->stream, static_cast<const float *>(A), M, (int)w->K, A2, exps);
    HIPC_LAUNCHED(ctx);
    return nbits_rows_f16(ctx, A2, terms, exps, w, Y, 0, M);
}

#endif  // HIPC_PREFILL_WIDE

}  // namespace hipc
