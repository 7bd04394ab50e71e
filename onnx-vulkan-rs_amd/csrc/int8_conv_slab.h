// Convolutions straight from the NCHW activation, one or two axes, any channel count (group 1).
//
// Reference: crates/onnx-vulkan-core/src/interp.rs:4421-4651, shaders/conv_integer.rs.
//
// The general route first writes the activation out as NHWC (a launch of its own, 2.5 us of 12.7 for 8 x 128 x 28 x 28) and
// its products gather 16-byte pieces of it with two round trips to memory per 128 k. Here a workgroup takes 64 or 128
// consecutive output positions (row after row of the image) and reads the input rows they see -- one contiguous run of every
// channel's plane -- once, transposes it 4 x 4 in registers and keeps it in LDS for the whole product, as
// [16-channel chunk][position of the run][16 channels]. A matrix-core operand is then one 16-byte LDS read at a
// position that a table, also in LDS, names for (tap, output position): that of the tap's input, or, where the tap is
// padding, one behind the run that holds the zero point. A product step is 32 k of one tap (two chunks; with a single chunk
// two neighbouring taps of a filter row), so what moves on from step to step are scalars. Weight fragments come straight
// from memory; the k loop has no barrier. (Working the positions out in the k loop, and divisions where the host's
// multipliers stand now, were 2 us of 8.6 for 192 x 4096, k = 7: a launch starts with an empty instruction cache and lives
// for one pass over its code.)
//
// Before (the general route, or one output per thread for channel counts off 16) -> this: 8 x 128 x 28 x 28, 3 x 3: 12.7 -> 7.2
// us; 5 x 112 -> 224 x 55 x 55 25.3 -> 12.5; 3 x 464 x 2682, k = 5: 51 -> 20.5; pointwise 9 x 128 -> 512 x 47 x 47 67.6 -> 14.1;
// 14 x 3 -> 40 x 224 x 224, 7 x 7 stride 2: 562 -> 32.7. (Twice the channels per wavefront, 128 x 128 tiles, halves the LDS
// reads and measured the same: 21.0, 12.6.)
//
// What bounds it: with few tiles the chain run -> LDS -> products -> epilogue of one workgroup; with many the LDS reads, 64
// positions x 32 bytes for two products of 32 clocks in each of four wavefronts, level with the matrix cores.
#pragma once

#include "int8_gemm.h"

namespace hipc {

// x / d for x < 2^31 as a product and a shift
struct Magic {
    uint32_t m, shift;
};
inline Magic magic_of(uint32_t d) {
    uint32_t s = 0;
    while ((uint64_t(1) << s) < d) s++;
    return {(uint32_t)(((uint64_t(1) << (31 + s)) + d - 1) / d), 31 + s};
}
__device__ __forceinline__ int div_by_magic(int x, const Magic &d) { return (int)(((uint64_t)(uint32_t)x * d.m) >> d.shift); }

struct ConvSlabArgs {
    GemmArgs g;        // (first: gemm_note_scalars names offsets in a GemmArgs) P: the weight, fragment-major, k = step * 32; Q: the activation
    int nch;           // 16-channel chunks
    int SP;            // positions a chunk of the slab has: the run, then one of zeros, then the padding
    int npair, kw2;    // product steps per tap; taps per filter row, or pairs of taps (`pairs`) with a single chunk
    int pairs;
    int steps, frag_steps;   // product steps; 1 KB weight fragments from 32 channels to the next 32
    int adv_tap, adv_q;      // WK product steps on: taps and pairs of chunks
    int tab_at;        // byte offset of the table in LDS
    int o_tiles, p_tiles, items, per_xcd;
    Magic by_o_tiles, by_p_tiles, by_wo;
};

constexpr size_t kSlabLds = 150 * 1024;   // what a slab may take (beyond: the general route)

// any byte address (the hardware takes it)
__device__ __forceinline__ uint32_t load_bytes4(const uint8_t *src) {
    uint32_t v;
    __builtin_memcpy(&v, src, 4);
    return v;
}

// The four wavefronts are WK along k (1 or 4), WP along the positions (1 or 2), the rest along the channels. A wavefront has
// 64 positions and 32 channels; with WK 4, 64 channels (conv_small_finish adds the parts up).
// RAGGED: C is no multiple of 16.
template <int EPI, bool DYN, int WK, int WP, bool RAGGED>
__global__ void __launch_bounds__(256, WK == 4 ? 3 : 4) int8_conv_slab_kernel(const ConvSlabArgs a) {
    constexpr int WO = 4 / (WK * WP), NF = WK == 4 ? 2 : 1, TP = 64 * WP, TO = 32 * NF * WO;
    const GemmArgs &p = a.g;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    uint8_t *slab = lds_raw;                                               // [nch][SP][16]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = WK == 4 ? wave : 0, wo = WK == 4 ? 0 : wave % WO, wp = WK == 4 ? 0 : wave / WO;
    const int r32 = lane & 31, kg = lane >> 5;

    // consecutive items -- the channel tiles of one run, then the next run -- on one XCD: they share what its L2 holds
    const int item = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
    if (item >= a.items) return;
    const int run = div_by_magic(item, a.by_o_tiles), img = div_by_magic(run, a.by_p_tiles);
    const int i0 = (item - run * a.o_tiles) * TO, j0 = (run - img * a.p_tiles) * TP;

    const int zd = (p.host_zp ? p.dyn_zp_value : zp_byte(p.dyn_zp, p.dyn_signed)) - p.dyn_shift;
    const int zc = (p.host_zp ? p.const_zp_value : zp_byte(p.const_zp, p.const_signed)) - p.const_shift;
    const uint32_t flip4 = p.dyn_shift ? 0x80808080u : 0u;

    // P: this wavefront's fragments (with WK 4 the one it finishes first: see conv_small_finish)
    const uint8_t *p_frag[NF];
#pragma unroll
    for (int f = 0; f < NF; f++)
        p_frag[f] = p.P + (size_t)(i0 / 32 + (WK == 4 ? f ^ (wave >> 1) : wo)) * a.frag_steps * 1024 + lane * 16;   // (the weight has rows for whole 128-channel tiles)
    uint4 rp[kSmallSets][NF];
    auto load_p = [&](int set, int stage) {
#pragma unroll
        for (int f = 0; f < NF; f++) rp[set][f] = *reinterpret_cast<const uint4 *>(p_frag[f] + (size_t)min(wk + stage * WK, a.steps - 1) * 1024);
    };
#pragma unroll
    for (int d = 0; d < kSmallSets; d++) load_p(d, d);
    // the epilogue's per-channel constants travel with the first loads
    ConvChannel chan;
    if constexpr (WK == 4) chan = conv_small_channel<EPI>(p, i0);
    else chan = conv_channel<EPI>(p, i0 + wo * 32 + r32);

    // The run: from the first input position a tap of the tile can need to the last. Within one output row that is a stretch
    // of columns, across rows whole rows. (Four positions at a time, from a multiple of four on.)
    const int HW = p.H * p.W;
    int f0, npq;
    {
        const int jl = min(j0 + TP, p.J) - 1;
        const int oh0 = div_by_magic(j0, a.by_wo), oh1 = div_by_magic(jl, a.by_wo);
        const int ih0 = max(oh0 * p.sh - p.pt, 0), ih1 = min(oh1 * p.sh - p.pt + (p.kh - 1) * p.dh, p.H - 1);
        const bool one = oh0 == oh1;
        const int iw0 = one ? max((j0 - oh0 * p.Wo) * p.sw - p.pl, 0) : 0;
        const int iw1 = one ? min((jl - oh1 * p.Wo) * p.sw - p.pl + (p.kw - 1) * p.dw, p.W - 1) : p.W - 1;
        f0 = (ih0 * p.W + iw0) & ~3;
        npq = ih1 >= ih0 && iw1 >= iw0 ? min((ih1 * p.W + iw1 - f0 + 4) >> 2, (a.SP - 2) >> 2) : 0;   // (nothing: every tap is padding)
    }
    // Dealt as in int8_conv_row_kernel: (chunk, quad of positions) pairs, 64 to a step of the workgroup, four lanes to a pair
    const int n_pairs = a.nch * npq;
    const uint8_t *x_img = p.Q + (size_t)img * p.C * HW;
    const int cq4 = (lane & 3) * 4;
    if (npq > 0) {
        const float per = __builtin_amdgcn_rcpf((float)npq);   // (quotients below 65 of numbers below 65: half a unit covers the rounding)
        const int adv_chunk = (int)(64.5f * per), adv_pq = 64 - adv_chunk * npq;
        int pair = wave * 16 + (lane >> 2);
        int chunk = (int)(((float)pair + 0.5f) * per), pq = pair - chunk * npq;
        for (int first = 0; first < n_pairs; first += 64 * kRowBatch) {
            uint32_t in[kRowBatch][4];
            int at[kRowBatch];   // byte offset of the pair's first word in the slab, or -1: nothing to store
#pragma unroll
            for (int u = 0; u < kRowBatch; u++) {
                at[u] = -1;
                if (first + 64 * u >= n_pairs) continue;
                const bool live = pair < n_pairs;
                const int gpos = f0 + 4 * (live ? pq : 0), from = min(gpos, HW - 4), c0 = (live ? chunk : 0) * 16 + cq4;
                const uint8_t *src = x_img + from;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    // (the last quad of a plane is read from where four bytes are left; channels past C hold zeros)
                    const uint32_t v = load_bytes4(src + (size_t)(RAGGED ? min(c0 + i, p.C - 1) : c0 + i) * HW) ^ flip4;
                    in[u][i] = !RAGGED || c0 + i < p.C ? v >> (8 * (gpos - from)) : 0u;
                }
                at[u] = live ? (chunk * a.SP + 4 * pq) * 16 + cq4 : -1;
                pair += 64;
                pq += adv_pq, chunk += adv_chunk;
                if (pq >= npq) pq -= npq, chunk++;
            }
#pragma unroll
            for (int u = 0; u < kRowBatch; u++) {
                if (at[u] < 0) continue;
                const uint32_t lo01 = __builtin_amdgcn_perm(in[u][1], in[u][0], 0x05010400u);  // a0 b0 a1 b1
                const uint32_t hi01 = __builtin_amdgcn_perm(in[u][1], in[u][0], 0x07030602u);  // a2 b2 a3 b3
                const uint32_t lo23 = __builtin_amdgcn_perm(in[u][3], in[u][2], 0x05010400u);  // c0 d0 c1 d1
                const uint32_t hi23 = __builtin_amdgcn_perm(in[u][3], in[u][2], 0x07030602u);  // c2 d2 c3 d3
                uint32_t *dst = reinterpret_cast<uint32_t *>(slab + at[u]);
                dst[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);   // a0 b0 c0 d0: position 4 pq
                dst[4] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
                dst[8] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
                dst[12] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
            }
        }
    }
    // the position of zeros, and the padding: the zero point in every channel there is
    for (int c = tid; c < a.nch * 16; c += 256) {
        uint8_t *at = slab + ((c >> 4) * a.SP + a.SP - 2) * 16 + (c & 15);
        at[0] = 0, at[16] = c < p.C ? (uint8_t)zd : (uint8_t)0;
    }
    // The table: for (filter row, tap, output position of the tile) where in a chunk of the slab the tap's input is. A thread
    // keeps its output position and takes every 256 / TP-th column of taps; with pairs of taps the row's last pair may lack its second.
    const int taps = a.pairs ? 2 * a.kw2 : a.kw2;   // of a filter row
    uint16_t *tab = reinterpret_cast<uint16_t *>(lds_raw + a.tab_at);
    {
        const int pos = tid & (TP - 1), gj = j0 + pos;
        const int oh = div_by_magic(gj, a.by_wo);
        const int ih0 = oh * p.sh - p.pt, iw0 = (gj - oh * p.Wo) * p.sw - p.pl, at0 = ih0 * p.W + iw0 - f0;
        for (int s = tid / TP; s < taps; s += 256 / TP) {
            const bool column = gj < p.J && (unsigned)(iw0 + s * p.dw) < (unsigned)p.W;
            int ih = ih0, from = at0 + s * p.dw;
            for (int r = 0; r < p.kh; r++) {
                tab[(r * taps + s) * TP + pos] = (uint16_t)(s >= p.kw ? a.SP - 2 : column && (unsigned)ih < (unsigned)p.H ? from : a.SP - 1);
                ih += p.dh, from += p.dh * p.W;
            }
        }
    }

    // The product step to be read next: tap (or pair of taps) t, pair of chunks q, both scalars; `at` where the tap puts the
    // lane's two positions (with WK 4 those of the fragment it finishes first), read a step ahead
    const int SP16 = a.SP * 16, last_chunk = (a.nch - 1) * SP16, kg_chunk = a.pairs ? 0 : kg * SP16;
    int n = wk, t = 0, q = wk;
    while (q >= a.npair) q -= a.npair, t++;
    const uint16_t *tab_lane = tab + (a.pairs ? kg * TP : 0) + wp * 64 + r32;
    const int tab_tap = a.pairs ? 2 * TP : TP;
    int at[2];
    auto place = [&] {
#pragma unroll
        for (int f = 0; f < 2; f++) at[f] = tab_lane[t * tab_tap + (WK == 4 ? f ^ (wave & 1) : f) * 32];
    };
    i32x16 acc[2][NF];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < NF; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0;
    int dsum[2] = {0, 0};
    uint4 bq[2][2];
    bool half[2];   // the step's second chunk is there (its weight is zero otherwise, and the sums leave it out)
    auto read_q = [&](int par) {
        const int chunk_at = 2 * q * SP16;
        half[par] = a.pairs || 2 * q + 1 < a.nch;
        // (an odd number of chunks: the second half of the last pair reads the last chunk again)
        const int lane_at = chunk_at + SP16 > last_chunk ? chunk_at : chunk_at + kg_chunk;
#pragma unroll
        for (int f = 0; f < 2; f++) bq[par][f] = *reinterpret_cast<const uint4 *>(slab + at[f] * 16 + lane_at);
        const bool more = n + WK < a.steps;   // (past the last step: the same once more, not used)
        n += more ? WK : 0;
        q += more ? a.adv_q : 0, t += more ? a.adv_tap : 0;
        const bool wrap = q >= a.npair;
        q -= wrap ? a.npair : 0, t += wrap ? 1 : 0;
        place();
    };
    auto compute = [&](int set, int par) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if (DYN) dsum[j] += kg == 0 || half[par] ? dot_ones(bq[par][j]) : 0;
#pragma unroll
            for (int i = 0; i < NF; i++)
                acc[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, bq[par][j]), __builtin_bit_cast(i32x4, rp[set][i]), acc[j][i], 0, 0, 0);
        }
    };

    __syncthreads();
    const int mine = (a.steps - wk + WK - 1) / WK;   // (the host lets wavefronts share k only where there are steps for all)
    place();
    read_q(0);
    int st = 0;
    for (; st + kSmallSets <= mine; st += kSmallSets) {
#pragma unroll
        for (int d = 0; d < kSmallSets; d++) {
            read_q((d + 1) & 1);
            compute(d, d & 1);
            load_p(d, st + d + kSmallSets);
        }
    }
#pragma unroll
    for (int d = 0; d < kSmallSets - 1; d++)
        if (st + d < mine) {
            read_q((d + 1) & 1);
            compute(d, d & 1);
        }
    if constexpr (WK == 4) {
        __syncthreads();   // the hand-over reuses the slab's LDS
        int *lds_acc = reinterpret_cast<int *>(lds_raw);
        conv_small_finish<EPI, DYN>(p, acc, dsum, chan, lds_acc, lds_acc + 4 * 3 * 16 * 64, i0, j0, img, zd, zc);
    } else {
        const int ch = i0 + wo * 32 + r32;
        const int fixed = p.K * zd * zc - zd * chan.csum + (EPI == EPI_REQUANT ? chan.qb : 0);
#pragma unroll
        for (int f = 0; f < 2; f++) {
            if (DYN) dsum[f] += __shfl_xor(dsum[f], 32, 64);   // the two k halves of position f * 32 + r32
            int out[16];
#pragma unroll
            for (int e = 0; e < 16; e++) {
                out[e] = acc[f][0][e] + fixed;
                if (DYN) out[e] -= zc * __shfl(dsum[f], (e >> 2) * 8 + kg * 4 + (e & 3), 64);
            }
            if (ch < p.I) conv_store<EPI>(p, chan, out, img, ch, j0 + wp * 64 + f * 32);
        }
    }
}

}  // namespace hipc
