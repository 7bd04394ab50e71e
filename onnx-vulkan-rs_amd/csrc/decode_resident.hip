// All layers of one decode step in one launch: a grid of one workgroup per CU that stays on the chip and hands its rows
// from phase to phase through memory, instead of five launches per layer.
//
// A launch boundary costs about 2 us before the next kernel's first operand is there (drain, dispatch, arguments, a cold
// scalar cache, the first trip to memory); a token of 26 layers has 130 of them. Handing a row over inside a launch was
// measured (MI355X, per hand-over, all members storing and waiting for all): 0.52 us between the 32 workgroups of an XCD,
// through its L2; 0.87 us between two workgroups of different XCDs, 1.7 us between all 256. So the work is laid out for
// the XCDs:
//   * The q, k and v columns are dealt to all 256 workgroups and handed to the XCDs that want them; XCD x then serves query head
//     x / P (P = 8 / heads XCDs a head), the (x mod P)th part of the context: its 32 workgroups attend to
//     their positions, and multiply their joined, unnormalised outputs by o's rows of the head. What leaves the XCD is one
//     partial row of the o product and the softmax maximum and sum that weigh it.
//   * Workgroup r of every XCD holds the same columns of the hidden row, so a row is summed over the XCDs by eight
//     workgroups that exchange 48 columns each, and gathered inside each XCD again: 1.0 + 0.5 us for an all-reduce.
//   * XCD x holds the ffn columns of the 128-k tiles x, x + 8, ... of the down projection: gate|up columns and down rows
//     of its own, so the gated row never leaves it; the down product's partial rows are summed like o's.
// Per layer four hand-overs stay inside the XCDs and three cross them. Weights and cache rows do not depend on the row, so
// every phase's are asked for two phases ahead, straight into registers (17 MB a layer are 68 KB a workgroup).
//
// Hand-overs carry their own "ready": an empty word is all ones (no result has that pattern, see put()), readers poll the
// words themselves (agent scope loads), so a hand-over is one store and one load, without flags or fences. There are three
// sets of words, taken in turn by the layers. Where layer l begins, a workgroup empties its words of layer l + 1 (they hold
// layer l - 2's): every workgroup it shares words with has then left layer l - 2, since it has handed over attention outputs
// (or partial rows) of layer l - 1; and the emptying has reached memory before the workgroup hands over its own of layer l
// (see the wait before the attention's barrier), without which nobody comes to layer l + 1. Inside an XCD stores go to its
// L2 only (workgroup scope); whether the members of a group really share one is read from the hardware when the launch
// starts, and if not all stores are of agent scope.
//
// Nothing waits for a workgroup that may never come (resident_door.h): the launch begins when all 256 have arrived, which takes
// microseconds on a free device, or else everyone leaves by a deadline of their own, and a launch behind it deals the 256 shares
// of the work to the workgroups that have arrived there; one that arrives later leaves at once. So such launches on one device,
// from other streams or processes, cannot block each other. Waits for workgroups that take part, which are all on the chip,
// are bounded beside that: a thread's polls of a whole launch are counted.
#include <hip/hip_fp16.h>

#include "internal.h"
#include "lanes.h"
#include "lean_ops.h"
#include "resident.h"

namespace hipc {

#ifndef HIPC_HOST_MODEL
#define RES_ONE_PER_CU __attribute__((amdgpu_waves_per_eu(2, 2)))   // two wavefronts a SIMD: 256 registers each
#else
#define RES_ONE_PER_CU
#endif

// phase time stamps (library built with `make stamps` only; see gemv_lean.hip): res_stamps[workgroup][wavefront][phase] of one
// layer, kept in LDS until the layer's end (a store to memory would be waited for by the polls behind it)
#ifdef HIPC_PHASE_STAMPS
constexpr int kStampLayer = 12;
__device__ unsigned long long res_stamps[256 * 8 * 32];
#define RES_STAMP(ph)                                                                      \
    do {                                                                                   \
        const unsigned long long t_ = (unsigned long long)clock64();                       \
        if ((threadIdx.x & 63) == 0) S.stamp[threadIdx.x >> 6][ph] = t_;                   \
    } while (0)
#define RES_STAMPS_OUT()                                                                   \
    do {                                                                                   \
        if (l == kStampLayer && (threadIdx.x & 63) < 32)                                   \
            res_stamps[(blockIdx.x * 8 + (threadIdx.x >> 6)) * 32 + (threadIdx.x & 63)] = S.stamp[threadIdx.x >> 6][threadIdx.x & 63]; \
    } while (0)
#else
#define RES_STAMP(ph)
#define RES_STAMPS_OUT()
#endif
constexpr uint32_t kEmpty = 0xffffffffu;
constexpr int kAgent = 16;        // cache policy of loads and stores at agent scope (sc1)
constexpr int kInXcd = 1;         // ... of stores at workgroup scope (sc0): as far as the XCD's L2
#ifndef HIPC_HOST_MODEL
constexpr int kPollBudget = 1 << 23;                   // polls of one thread in one launch: seconds, where a launch has thousands
#else
constexpr int kPollBudget = 1;                         // (one thread after the other: there is nobody to wait for)
#endif
// How long workgroups that have not started are waited for, in ticks of the 100 MHz clock. All of them, 50 us: they arrive within
// microseconds on a free device, and within the 50 us another decoder's unembedding and token pick keep some CUs. In the
// stand-in until nobody has come for 5 us.
// Beside other work, us a token of gemma3-1b at 2048 (454 alone; launches per product 654 alone), the launches per product / 50 us and
// 256 workgroups standing in / 200 us and 256 / 200 us and 64: beside a softmax of eight workgroups of a millisecond 763 / 773 / 923 / 1602;
// launches that hold 64 CUs for 220 us 730 / 908 / 835 / 1191, 128 CUs for 140 us 788 / 777 / 570 / 569; products that fill the chip for 125 us
// at a time - / 860 / 860 / 872. Two decoders side by side, a token of each: 780 / 878 / 877 / 877; three 918 / 1900 / 2490 / 2060,
// four 1061 / 2190 / 2880 / 2180: launches that each want the whole chip take turns at best, where short ones fill each other's
// gaps (these figures scatter by a fifth), so contexts that decode at the same time are better off with HIPC_DEC_RESIDENT=0.
constexpr int kArriveTicks = 5000, kJoinTicks = 500;
constexpr int kResThreads = 512, kResWaves = 8;
constexpr int kRedPitch = 20;                          // words per column of the reduction area: 16 k tiles, 16-byte rows
constexpr int kSumsAt = 64 * 2 * 4 * 16;               // bytes from the row's terms to their chunks' sums (ResShared)
constexpr int kResUnits = 12;                          // units a thread's wavefront asks for ahead, all phases
constexpr int kEntryWords = (int)(sizeof(ResidentLayer) / 4);

typedef _Float16 rh16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bool any_empty(uint4 v) { return max(max(v.x, v.y), max(v.z, v.w)) == kEmpty; }
// the compiler may neither keep a polled word in a register nor move the loads of weights across a wait
__device__ __forceinline__ void res_reload() { asm volatile("" ::: "memory"); }
#ifndef HIPC_HOST_MODEL
__device__ __forceinline__ void res_stored() {
    res_reload();
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0), in a form the compiler takes into account
    res_reload();
}   // every store of this wavefront is where its scope says
#else
inline void res_stored() {}
#endif

// A wavefront's share of a phase's product: up to U (column tile, k tile) units, one after the other 128 k of 16 columns.
// Which units they are does not change between layers: their byte offsets are worked out once and kept in LDS (kept in
// registers, they and the weights of three phases do not fit).
// The sums of a unit are the same in all four groups of 16 lanes, so one group's are enough: group g takes those of units
// g, 4 + g, ... and holds the scales and zero points of these only, asked for together with three other units'.
template <int U, int SG>
struct Units {
    uint4 wq[U];
    ScaleVecLean<SG> sv[(U + 3) / 4];
    uint32_t live;   // bit i: unit i exists
};

// A product unit against the row's terms in LDS (see mmnb_lean_kernel). The lanes that hold the unit's scales return their column's sum.
template <int SG>
__device__ __forceinline__ float res_unit(const uint4 &wq, const ScaleVecLean<SG> &sv, const char *as, uint32_t o_as, uint32_t nib_mask, uint32_t magic) {
    constexpr int CPG = 4 / SG;
    uint4 a[4];
#pragma unroll
    for (int j = 0; j < 4; j++) a[j] = *reinterpret_cast<const uint4 *>(as + o_as + j * 128);
    const float4 bs = *reinterpret_cast<const float4 *>(as + kSumsAt + ((o_as >> 9) << 4));
    lf32x4 d[SG];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t word = j == 0 ? wq.x : j == 1 ? wq.y : j == 2 ? wq.z : wq.w;
        const uint4 bw = make_uint4((word & nib_mask) | magic, ((word >> 4) & nib_mask) | magic, ((word >> 8) & nib_mask) | magic, ((word >> 12) & nib_mask) | magic);
        const int g = j / CPG;
        d[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lbf16x8, a[j]), __builtin_bit_cast(lbf16x8, bw), (j % CPG) == 0 ? lf32x4{0.f, 0.f, 0.f, 0.f} : d[g], 0, 0, 0);
    }
    float acc = 0.f;
#pragma unroll
    for (int g = 0; g < SG; g++) {
        const float dsum = d[g][0] + d[g][1];
        float asg;
        if (SG == 4) asg = g == 0 ? bs.x : g == 1 ? bs.y : g == 2 ? bs.z : bs.w;
        else if (SG == 2) asg = g == 0 ? bs.x + bs.y : bs.z + bs.w;
        else asg = (bs.x + bs.y) + (bs.z + bs.w);
        const float zb = (float)((sv.z >> (8 * g)) & 0xffu);
        acc = fmaf(sv.s[g], fmaf(-zb, asg, dsum), acc);
    }
    return acc;
}

// gelu_tanh: 0.5 v (1 + tanh u) = v / (1 + exp(-2 u)), without the difference that loses digits where tanh is near -1
__device__ __forceinline__ float res_gelu(float v) {
    return v / (1.f + __expf(-1.5957691216057308f * fmaf(0.044715f, v * v * v, v)));
}

// the LDS of a workgroup
template <int HD>
struct ResShared {
    uint4 As[64 * 2 * 4];                                // the row as two bf16 terms: [32-k chunk][term][8-k group]
    float bsum[64];                                      // the sum of the terms per chunk
    float red[4][64 * kRedPitch];                        // per phase: [column][k tile]; places that no k tile has stay zero
    float trash[64];                                     // where lanes without a result store
    uint2 off[kResUnits][kResThreads];                   // the offsets of every thread's units
    float4 red4[4 * kResWaves];
    float join[kResThreads * 4];
    float rope[2 * HD];
    __half qa[2 * (HD + 8)];
    __half pa[kResWaves][2 * (kAttnPass + 8)];
    float sp[kResWaves][16];
    float kn[HD], vn[HD];
    float sown;
    uint32_t decision[2];
#ifdef HIPC_PHASE_STAMPS
    unsigned long long stamp[kResWaves][32];
#endif
};

// The work of a launch. ALL: the 256 workgroups are there and workgroup v does share v of every phase; what follows needs no
// division and no loop over shares, and weights are asked for phases ahead. Else `n` workgroups take the shares in turn.
template <int HD, int SG, bool ALL>
__device__ __forceinline__ void res_layers(const ResidentArgs &p, ResShared<HD> &S, int first, const int n, const bool wide, uint32_t set, const int pos, int &tries) {
    constexpr int KT3 = HD >= 128 ? HD / 128 : 1;  // k tiles of a head in o's weight (half of one at 64 channels)
    constexpr int KS = HD >= 128 ? HD / 128 : 1;   // 32-channel steps of a wavefront's share of the scores
    constexpr int DQ = HD / (32 * KS);             // wavefronts that share the channels of the scores
    constexpr int NB = HD >= 128 ? HD / 128 : 1;   // 16-channel blocks of a wavefront's outputs
    constexpr int QS = HD + 8, PS = kAttnPass + 8; // halfs per operand row (16 bytes of padding)
    constexpr int NJ = kResThreads * 4 / HD;       // rows of chunks that are joined side by side
    constexpr int U1 = 2, U3 = 1, U4 = 5, U5 = 3;   // units asked for ahead; a wavefront's further ones when it comes to them
    constexpr float NEG = -3.0e38f;

    int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int i16 = lane & 15, g4 = lane >> 4;
    uint32_t magic;
    HIPC_VGPR_FROM_SGPR(magic, p.magic);
    const uint32_t nib_mask = p.nib_mask;
    const int total = pos + 1;
    const __amdgpu_buffer_rsrc_t r_x = lean_rsrc(p.xch, kResSets * kResWords * 4u);
    const char *as = reinterpret_cast<const char *>(S.As);

    // ---- the layer's entry: lane i holds word i of it, a pointer is read from two lanes. (Scalar loads would miss the
    // scalar cache once per phase.) The next layer's is asked for a layer ahead.
    auto entry_of = [&](int l) {
#ifndef HIPC_HOST_MODEL
        return reinterpret_cast<const uint32_t *>(p.table + min(l, p.n_layers - 1))[min(lane, kEntryWords - 1)];
#else
        return (uint32_t)l;
#endif
    };
    uint32_t ent = entry_of(0), ent_next = entry_of(1);
    auto word_of = [&](uint32_t e, int i) {
#ifndef HIPC_HOST_MODEL
        return (uint32_t)__builtin_amdgcn_readlane((int)e, i);
#else
        return reinterpret_cast<const uint32_t *>(p.table + std::min((int)e, p.n_layers - 1))[i];
#endif
    };
    auto ptr_of = [&](uint32_t e, int i) { return reinterpret_cast<void *>(((uint64_t)word_of(e, 2 * i + 1) << 32) | word_of(e, 2 * i)); };
    constexpr int kNorm = 12, kCache = 18, kWindow = 40, kRope = 41;
    static_assert(offsetof(ResidentLayer, norm) == kNorm * 8 && offsetof(ResidentLayer, k_cache) == kCache * 8 && offsetof(ResidentLayer, window) == kWindow * 4, "entries are read as words");

    struct Weight {
        __amdgpu_buffer_rsrc_t q, s, z;
    };
    auto weight = [&](uint32_t e, int which, uint32_t tiles) {
        return Weight{lean_rsrc(ptr_of(e, which), tiles * 1024u), lean_rsrc(ptr_of(e, 4 + which), tiles * 64u * SG), lean_rsrc(ptr_of(e, 8 + which), tiles * 16u * SG)};
    };
    const uint32_t n1 = (uint32_t)(p.tiles_qkv * p.cg_h), n3 = (uint32_t)(p.tiles_h * p.cg_o), n4 = (uint32_t)(2 * p.pairs * p.cg_h), n5 = (uint32_t)(p.tiles_h * p.cg_f);

    // ---- which units share v of a phase has
    struct Unit {
        int tl, kt, t;   // tile of the weight, k tile of the row in LDS, column tile of the workgroup
        bool live;
    };
    auto split_unit = [&](int u, int *kt) {   // unit u = (column tile u / cg_h, k tile u % cg_h)
        const int t = (int)(((uint32_t)u * p.inv_cg_h) >> 16);
        *kt = u - t * p.cg_h;
        return t;
    };
    // q|k|v: column tiles v and v + 256, all of hidden's k tiles
    auto tiles1 = [&](int v) { return (v < p.tiles_qkv) + (v + (int)kResGroups < p.tiles_qkv); };
    auto unit1 = [&](int v, int u) {
        Unit x;
        x.t = split_unit(u, &x.kt);
        x.tl = (v + (int)kResGroups * x.t) * p.cg_h + x.kt;
        x.live = u < tiles1(v) * p.cg_h;
        return x;
    };
    // o: the columns of the hidden row that rank r holds, tiles r, r + 32, ...; the k tiles of the XCD's head
    auto tiles3 = [&](int v) { return (p.tiles_h - (v >> 3) + 31) >> 5; };
    auto unit3 = [&](int v, int u) {
        const int h = (v & 7) >> p.lg_parts;
        Unit x;
        x.t = u / KT3, x.kt = u % KT3;
        x.tl = ((v >> 3) + 32 * x.t) * p.cg_o + (h * HD) / 128 + x.kt;
        x.live = x.t < tiles3(v);
        return x;
    };
    // gate|up: the XCD holds the pairs of the down projection's k tiles x, x + 8, ..., 8 pairs each; rank r its pairs r, r + 32
    auto slice_tiles = [&](int v) { return (p.cg_f - (v & 7) + 7) >> 3; };
    auto pair_of = [&](int v, int q) {   // global pair, or one past the last: nothing there
        const int lp = (v >> 3) + 32 * q;
        return min(((v & 7) + 8 * (lp >> 3)) * 8 + (lp & 7), p.pairs);
    };
    auto pairs4 = [&](int v) {
        const int m = slice_tiles(v) * 8;
        return ((v >> 3) < m) + ((v >> 3) + 32 < m);
    };
    auto unit4 = [&](int v, int u) {
        Unit x;
        x.t = split_unit(u, &x.kt);
        const int pair = pair_of(v, x.t >> 1);
        x.tl = (2 * pair + (x.t & 1)) * p.cg_h + x.kt;
        x.live = u < 2 * pairs4(v) * p.cg_h && pair < p.pairs;
        return x;
    };
    // down: rank r's columns, the XCD's k tiles; unit u = (tile u % tiles, k tile u / tiles), at most four tiles
    auto unit5 = [&](int v, int u) {
        const int tiles = tiles3(v);
        Unit x;
        x.kt = tiles <= 1 ? u : tiles == 2 ? u >> 1 : tiles == 4 ? u >> 2 : (int)(((uint32_t)u * 21846u) >> 16);
        x.t = u - x.kt * tiles;
        x.tl = ((v >> 3) + 32 * x.t) * p.cg_f + (v & 7) + 8 * x.kt;
        x.live = u < tiles * slice_tiles(v);
        return x;
    };
    // the lane's offsets of a unit: in the weight (what its scales' and zero points' follow from); in LDS, the row's operand
    // and in the upper half where the sum goes
    auto offsets_of = [&](const Unit &x, int i, int phase) {
        // (a unit that does not exist loads from past the end of everything: zeros, and no traffic. A load that is skipped
        // would keep the registers of the layer before alive.)
        const uint32_t red = g4 == (i & 3) ? (uint32_t)(phase * 64 * kRedPitch + (x.t * 16 + i16) * kRedPitch + x.kt) : (uint32_t)(4 * 64 * kRedPitch + lane);
        return make_uint2(x.live ? (uint32_t)x.tl * 1024u + (uint32_t)lane * 16u : 0xffff0000u,
                          (uint32_t)x.kt * 512u + (uint32_t)(min(i16 & 3, 1) * 4 + g4) * 16u + (red << 18));
    };
    auto load_scales = [&](const Weight &b, ScaleVecLean<SG> &sv, uint32_t o_wq) {   // of the unit at the lane's o_wq
        const uint32_t o_zb = (o_wq >> 10) * (16u * SG) + (uint32_t)i16 * SG;
        sv.load(b.s, b.z, o_zb * 4u, o_zb, 0);
    };
    // units from .. to - 1 (from: a multiple of four, or 2 with its neighbours' scales already asked for)
    auto load_units = [&](auto &w, int at, const Weight &b, int from = 0, int to = 8) {
        constexpr int U = (int)(sizeof w.wq / sizeof w.wq[0]);
        uint32_t o[U], os[(U + 3) / 4];
#pragma unroll
        for (int i = 0; i < U; i++)
            if (i >= from && i < to) o[i] = S.off[at + i][tid].x;
#pragma unroll
        for (int i = 0; i < U; i += 4)
            if (i >= from && i < to) os[i / 4] = S.off[at + min(i + g4, U - 1)][tid].x;
#pragma unroll
        for (int i = 0; i < U; i++) {
            if (i < from || i >= to) continue;
            if (i % 4 == 0) load_scales(b, w.sv[i / 4], os[i / 4]);
            w.wq[i] = lean_ld16(b.q, o[i], 0);
        }
    };
    auto multiply_one = [&](auto &w, int i, uint32_t o_lds) {
        const float acc = res_unit<SG>(w.wq[i], w.sv[i / 4], as, o_lds & 0xffffu, nib_mask, magic);
        *reinterpret_cast<float *>(reinterpret_cast<char *>(S.red) + (o_lds >> 16)) = acc;
    };
    // a phase's product: what was asked for ahead, then whatever else the share has
    auto multiply = [&](auto &w, int at, uint32_t e, int which, uint32_t tiles, int v, int units, int phase, auto &&unit) {
        constexpr int U = (int)(sizeof w.wq / sizeof w.wq[0]);
        if (ALL) {
            uint32_t o[U];
#pragma unroll
            for (int i = 0; i < U; i++) o[i] = S.off[at + i][tid].y;
#pragma unroll
            for (int i = 0; i < U; i++)
                if ((w.live >> i) & 1u) multiply_one(w, i, o[i]);
        }
        for (int u = wave + (ALL ? 8 * U : 0); u < units; u += 8) {
            const Unit x = unit(v, u);
            if (!x.live) continue;
            Units<1, SG> one;
            const uint2 o = offsets_of(x, 0, phase);
            const Weight b = weight(e, which, tiles);
            load_scales(b, one.sv[0], o.x);
            one.wq[0] = lean_ld16(b.q, o.x, 0);
            multiply_one(one, 0, o.y);
        }
    };
    Units<U1, SG> w1;
    Units<U3, SG> w3;
    Units<U4, SG> w4;
    Units<U5, SG> w5;
    constexpr int kAt1 = 0, kAt3 = U1, kAt4 = U1 + U3, kAt5 = U1 + U3 + U4;
    static_assert(kAt5 + U5 <= kResUnits, "places for the units' offsets");
    if (ALL) {
        auto set_units = [&](auto &w, int at, int phase, auto &&unit) {
            w.live = 0;
            for (int i = 0; i < (int)(sizeof w.wq / sizeof w.wq[0]); i++) {
                const Unit x = unit(first, wave + 8 * i);
                S.off[at + i][tid] = offsets_of(x, i, phase);
                w.live |= x.live ? 1u << i : 0u;
            }
        };
        set_units(w1, kAt1, 0, unit1), set_units(w3, kAt3, 1, unit3), set_units(w4, kAt4, 2, unit4), set_units(w5, kAt5, 3, unit5);
    }

    // ---- the cache rows of a share's positions: 32 at a time
    uint4 kreg[KS], vreg[NB];
    struct Span {
        int begin, end, first;
        bool dead;
    };
    auto span_of = [&](int v, int window) {
        const int base = attn_base(total, window), parts = 1 << p.lg_parts;
        const int per_pass = kAttnPass * (int)kResRanks * parts, len = total - base;
        const int chunk = len <= per_pass ? kAttnPass : kAttnPass * ((len + per_pass - 1) / per_pass);
        Span s;
        s.begin = base + (((v & 7) & (parts - 1)) * (int)kResRanks + (v >> 3)) * chunk;
        s.dead = s.begin >= total;
        s.end = min(total, s.begin + chunk);
        s.first = attn_first(total, window);
        return s;
    };
    const int pb = wave & 1, dq = min(wave >> 1, DQ - 1);
    const uint32_t v_k = (uint32_t)((pb * 16 + i16) * HD + dq * 32 * KS + g4 * 8) * 2u;
    const uint32_t v_v = ((uint32_t)(min(wave * 16 * NB, HD - 16 * NB) + i16) * (uint32_t)p.v_stride + (uint32_t)(g4 * 8)) * 2u;
    auto load_k = [&](__amdgpu_buffer_rsrc_t r, int kvh, int t0) {
        const uint32_t s_k = ((uint32_t)kvh * (uint32_t)p.max_seq + (uint32_t)t0) * HD * 2u;
#pragma unroll
        for (int u = 0; u < KS; u++) kreg[u] = lean_ld16(r, v_k + u * 64u, s_k);
    };
    auto load_v = [&](__amdgpu_buffer_rsrc_t r, int kvh, int t0) {
#pragma unroll
        for (int b = 0; b < NB; b++) vreg[b] = lean_ld16(r, v_v, (((uint32_t)kvh * HD + b * 16u) * (uint32_t)p.v_stride + (uint32_t)t0) * 2u);
    };
    auto rsrc_k = [&](uint32_t e, bool dead) { return lean_rsrc(ptr_of(e, kCache), dead ? 0u : ((uint32_t)p.n_kv * (uint32_t)p.max_seq + 64u) * HD * 2u); };
    auto rsrc_v = [&](uint32_t e, bool dead) { return lean_rsrc(ptr_of(e, kCache + 1), dead ? 0u : (uint32_t)p.n_kv * HD * (uint32_t)p.v_stride * 2u); };
    auto load_kv = [&](uint32_t e, int v) {
        const Span s = span_of(v, (int)word_of(e, kWindow));
        const int kvh = ((v & 7) >> p.lg_parts) >> p.lg_group, t0 = s.dead ? 0 : s.begin;   // (the scalar offset stays inside whatever the descriptor says)
        load_k(rsrc_k(e, s.dead), kvh, t0), load_v(rsrc_v(e, s.dead), kvh, t0);
    };
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    // norm weights of the heads: the query's for wavefront 0, the key's for wavefront 1. (A load under a condition would be
    // waited for where the condition ends: none of the loads ahead has one.)
    float4 head_w = zero4;
    auto load_head_w = [&](uint32_t e) {
        head_w = __builtin_bit_cast(float4, lean_ld16(lean_rsrc(ptr_of(e, kNorm + 4 + (wave & 1)), HD * 4u), (uint32_t)lane * 16u, 0));
    };
    // what a layer's first phases need, asked for while the layer before is in its last one
    auto load_ahead = [&](uint32_t e) {
        load_head_w(e);
        if (ALL) load_units(w1, kAt1, weight(e, 0, n1));
    };

    // ---- hand-overs
    uint32_t cur = set * kResWords * 4u, next = (set == kResSets - 1 ? 0u : set + 1u) * kResWords * 4u;   // byte offsets of this layer's and the next layer's words
    auto store = [&](uint32_t word, uint32_t bits, uint32_t in, bool agent) {
        if (agent) __builtin_amdgcn_raw_buffer_store_b32(bits, r_x, (int)(word * 4u), (int)in, kAgent);
        else __builtin_amdgcn_raw_buffer_store_b32(bits, r_x, (int)(word * 4u), (int)in, kInXcd);
    };
    auto put = [&](uint32_t word, uint32_t bits, bool agent) { store(word, bits == kEmpty ? 0x7fc00000u : bits, cur, agent); };   // (only a NaN has that pattern)
    // share v's words of the next layer, empty (wavefronts 3 to 7, which wait for nothing where this stands)
    auto clear = [&](int v) {
        const uint32_t r = (uint32_t)(v >> 3), x = (uint32_t)(v & 7), mine = x * kResLocal;
        const uint32_t col = (r + 32u * (uint32_t)g4) * 16u + (uint32_t)i16;   // lane's place in a row of tiles r, r + 32, ...
        if (wave == 3) {
#pragma unroll
            for (int i = 0; i < HD / 64; i++) store(mine + kResA + r * HD + (uint32_t)(lane + 64 * i), kEmpty, next, wide);
        } else if (wave == 4) {
            if (lane < tiles1(v) * 16) store(kResQ + (uint32_t)((v + (int)kResGroups * g4) * 16 + i16), kEmpty, next, true);
            if (lane < 2) store(mine + kResML + 2u * r + (uint32_t)lane, kEmpty, next, wide);
        } else if (wave == 5) {
            if (lane < 16 * pairs4(v)) store(mine + kResH + col, kEmpty, next, wide);
            if (lane < 2) store(kResM1 + 32u * r + 2u * x + (uint32_t)lane, kEmpty, next, true);
        } else if (wave >= 6 && lane < tiles3(v) * 16) {
            store(mine + (wave == 6 ? kResY : kResY2) + col, kEmpty, next, wide);
            store((wave == 6 ? kResG1 : kResG2) + r * 512u + x * 64u + (uint32_t)lane, kEmpty, next, true);
        }
    };
    auto take16 = [&](uint32_t word) {
        uint4 v;
        do {
            res_reload();
            v = lean_ld16<kAgent>(r_x, word * 4u, cur);
        } while (any_empty(v) && --tries > 0);
        return v;
    };
    // four values of the row as two bf16 terms into LDS, and their chunk's sum; eight neighbouring threads make a chunk
    auto put_terms = [&](int i4, uint2 hi, uint2 lo) {
        uint2 *dst = reinterpret_cast<uint2 *>(S.As) + (i4 >> 3) * 16 + (i4 & 7);
        dst[0] = hi, dst[8] = lo;
        const lbf16pair ones = __builtin_bit_cast(lbf16pair, 0x3f803f80u);
        float s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(lbf16pair, hi.x), ones, 0.f, false);
        float t = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(lbf16pair, hi.y), ones, 0.f, false);
        s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(lbf16pair, lo.x), ones, s, false);
        t = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(lbf16pair, lo.y), ones, t, false);
        s += t;
        s += lean_dpp<0xB1>(s);
        s += lean_dpp<0x4E>(s);
        s += lean_dpp<0x141>(s);   // row_half_mirror: the other quad of the eight
        if ((i4 & 7) == 0) S.bsum[i4 >> 3] = s;
    };
    auto split_terms4 = [&](int i4, float a, float b, float c, float d) {
        uint2 hi, lo;
        hi.x = __builtin_bit_cast(uint32_t, __builtin_convertvector(lf32x2{a, b}, lbf16x2));
        hi.y = __builtin_bit_cast(uint32_t, __builtin_convertvector(lf32x2{c, d}, lbf16x2));
        a -= __uint_as_float(hi.x << 16), b -= __uint_as_float(hi.x & 0xffff0000u);
        c -= __uint_as_float(hi.y << 16), d -= __uint_as_float(hi.y & 0xffff0000u);
        lo.x = __builtin_bit_cast(uint32_t, __builtin_convertvector(lf32x2{a, b}, lbf16x2));
        lo.y = __builtin_bit_cast(uint32_t, __builtin_convertvector(lf32x2{c, d}, lbf16x2));
        put_terms(i4, hi, lo);
    };
    // stream += rmsnorm(branch, w_post); the row rmsnorm(stream, w_in) goes to LDS. One reduction for both norms (see mmnb_lean_kernel).
    float4 x4 = zero4, y4 = zero4;   // this thread's four values of the stream, and of the branch to be added
    const bool holds = tid * 4 < p.hidden;
    if (holds) x4 = *reinterpret_cast<const float4 *>(p.x_in + tid * 4);
    const int pw = (p.cg_h * 32 + 63) >> 6;   // wavefronts that hold parts of the row
    auto norm_row = [&](const float4 &wp, const float4 &wi) {
        const float4 yw = make_float4(y4.x * wp.x, y4.y * wp.y, y4.z * wp.z, y4.w * wp.w);
        if (wave < pw) {
            float s_yy = fmaf(y4.w, y4.w, fmaf(y4.z, y4.z, fmaf(y4.y, y4.y, y4.x * y4.x)));
            float s_xx = fmaf(x4.w, x4.w, fmaf(x4.z, x4.z, fmaf(x4.y, x4.y, x4.x * x4.x)));
            float s_xy = fmaf(x4.w, yw.w, fmaf(x4.z, yw.z, fmaf(x4.y, yw.y, x4.x * yw.x)));
            float s_ww = fmaf(yw.w, yw.w, fmaf(yw.z, yw.z, fmaf(yw.y, yw.y, yw.x * yw.x)));
            s_yy = lean_row_sum(s_yy), s_xx = lean_row_sum(s_xx), s_xy = lean_row_sum(s_xy), s_ww = lean_row_sum(s_ww);
            if (i16 == 0) S.red4[wave * 4 + g4] = make_float4(s_yy, s_xx, s_xy, s_ww);
        }
        __syncthreads();
        if (wave < pw) {
            const float4 r = lane < pw * 4 ? S.red4[lane & 31] : zero4;
            const float r_yy = lean_row_sum(r.x), r_xx = lean_row_sum(r.y), r_xy = lean_row_sum(r.z), r_ww = lean_row_sum(r.w);
            const float t_yy = lean_lane(r_yy, 0) + lean_lane(r_yy, 16), t_xx = lean_lane(r_xx, 0) + lean_lane(r_xx, 16);
            const float t_xy = lean_lane(r_xy, 0) + lean_lane(r_xy, 16), t_ww = lean_lane(r_ww, 0) + lean_lane(r_ww, 16);
            const float f1 = rsqrtf(t_yy * p.inv_hidden + p.eps);
            const float sq2 = fmaf(f1 * f1, t_ww, fmaf(2.f * f1, t_xy, t_xx));
            const float f2 = rsqrtf(fmaxf(sq2, 0.f) * p.inv_hidden + p.eps);
            x4.x = fmaf(yw.x, f1, x4.x), x4.y = fmaf(yw.y, f1, x4.y), x4.z = fmaf(yw.z, f1, x4.z), x4.w = fmaf(yw.w, f1, x4.w);
            if (tid < p.cg_h * 32) split_terms4(tid, x4.x * f2 * wi.x, x4.y * f2 * wi.y, x4.z * f2 * wi.z, x4.w * f2 * wi.w);
        }
        __syncthreads();
    };
    // the sum of a column's k tiles, in order (places past the last k tile hold zeros)
    auto column = [&](int phase, int col) {
        const float4 *c = reinterpret_cast<const float4 *>(S.red[phase] + col * kRedPitch);
        float4 v[4];
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = c[q];
        return (((v[0].x + v[0].y) + (v[0].z + v[0].w)) + ((v[1].x + v[1].y) + (v[1].z + v[1].w))) +
               (((v[2].x + v[2].y) + (v[2].z + v[2].w)) + ((v[3].x + v[3].y) + (v[3].z + v[3].w)));
    };
    auto zero_red = [&](int phase) {   // (before another share's product, which may have fewer k tiles)
        if (ALL) return;
        for (int i = tid; i < 64 * kRedPitch; i += kResThreads) S.red[phase][i] = 0.f;
        __syncthreads();
    };
    auto row4 = [&](uint32_t e, int which) { return __builtin_bit_cast(float4, lean_ld16(lean_rsrc(ptr_of(e, kNorm + which), (uint32_t)p.hidden * 4u), (uint32_t)tid * 16u, 0)); };   // (past the row: zeros)
    // rank r's columns of a row, summed over the XCDs' partial rows (weighed: with their softmax sums) and given to the XCD
    auto combine = [&](int v, uint32_t g, uint32_t to, bool weighed) {
        const int r = v >> 3, x = v & 7, cols = tiles3(v) * 16;
        const uint32_t base = g + (uint32_t)r * 512u + (uint32_t)min(lane, cols - 1);
        uint32_t part[8];
        uint2 ml = make_uint2(0, 0);
        bool again;
        do {
            res_reload();
            if (weighed) ml = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r_x, (int)((kResM1 + 32u * r + 2u * (lane & 7)) * 4u), (int)cur, kAgent));
#pragma unroll
            for (int s = 0; s < 8; s++) part[s] = __builtin_amdgcn_raw_buffer_load_b32(r_x, (int)((base + 64u * s) * 4u), (int)cur, kAgent);
            again = max(ml.x, ml.y) == kEmpty || max(max(max(part[0], part[1]), max(part[2], part[3])), max(max(part[4], part[5]), max(part[6], part[7]))) == kEmpty;
        } while (again && --tries > 0);
        float y;
        if (weighed) {
            // lane s of every eight: XCD s. The parts of a head are neighbours.
            const float m = __uint_as_float(ml.x), l = __uint_as_float(ml.y);
            float mm = m;
            if (p.lg_parts >= 1) mm = fmaxf(mm, lean_dpp<0xB1>(mm));
            if (p.lg_parts >= 2) mm = fmaxf(mm, lean_dpp<0x4E>(mm));
            if (p.lg_parts >= 3) mm = fmaxf(mm, lean_dpp<0x141>(mm));
            const float e = __expf(m - mm);
            float d = e * l;
            if (p.lg_parts >= 1) d += lean_dpp<0xB1>(d);
            if (p.lg_parts >= 2) d += lean_dpp<0x4E>(d);
            if (p.lg_parts >= 3) d += lean_dpp<0x141>(d);
            const float wgt = e / d;
            float y0 = 0.f, y1 = 0.f;
#pragma unroll
            for (int s = 0; s < 8; s += 2) y0 = fmaf(lean_lane(wgt, s), __uint_as_float(part[s]), y0), y1 = fmaf(lean_lane(wgt, s + 1), __uint_as_float(part[s + 1]), y1);
            y = y0 + y1;
        } else {
            float f[8];
#pragma unroll
            for (int s = 0; s < 8; s++) f[s] = __uint_as_float(part[s]);
            y = ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
        }
        if (lane < cols) put((uint32_t)x * kResLocal + to + (uint32_t)((r + 32 * g4) * 16 + i16), __float_as_uint(y), wide);
    };
    const uint32_t home = (uint32_t)(first & 7) * kResLocal;   // where this workgroup reads rows all XCDs hold
    const int step = ALL ? (int)kResGroups : n;                // (ALL: every loop over shares runs once)
    const int end = ALL ? first + 1 : (int)kResGroups;

    for (int i = tid; i < 4 * 64 * kRedPitch; i += kResThreads) S.red[0][i] = 0.f;
    for (int i = tid; i < 2 * HD; i += kResThreads) S.rope[i] = p.rope[i];
    if (ALL) load_kv(ent, first);
    load_ahead(ent);
    float4 wp = zero4, wi = row4(ent, 0);
    __syncthreads();
    for (int l = 0; l < p.n_layers; l++) {
        // What follows from these is worked out where it is used: kept for all layers it would not fit the registers.
        HIPC_PIN_SGPR(first);
        HIPC_PIN_VGPR(lane);
        HIPC_PIN_VGPR(i16);
        HIPC_PIN_VGPR(g4);
        HIPC_PIN_VGPR(tid);
        // ---- q|k|v of the row
        RES_STAMP(0);
        norm_row(wp, wi);
        if (ALL) load_units(w4, kAt4, weight(ent, 2, n4), 0, 2);
        RES_STAMP(2);
        for (int v = first; v < end; v += step) {
            zero_red(0);
            multiply(w1, kAt1, ent, 0, n1, v, tiles1(v) * p.cg_h, 0, unit1);
            RES_STAMP(3);
            __syncthreads();
            if (wave == 7) {
                const float s = column(0, lane & 31);
                if (lane < tiles1(v) * 16) put(kResQ + (uint32_t)((v + (int)kResGroups * g4) * 16 + i16), __float_as_uint(s), true);
            }
            clear(v);
            if (!ALL) __syncthreads();
        }
        if (ALL) load_units(w3, kAt3, weight(ent, 1, n3));
        RES_STAMP(4);
        // ---- attention: the share's positions for the XCD's head
        for (int v = first; v < end; v += step) {
            const uint32_t mine = (uint32_t)(v & 7) * kResLocal;
            const int h = (v & 7) >> p.lg_parts, kvh = h >> p.lg_group;
            const Span s = span_of(v, (int)word_of(ent, kWindow));
            const bool is_last = !s.dead && s.end == total;
            const int hist_end = min(s.end, pos);
            float rq[4];
            if (wave < 3 && lane < HD / 4) {
                // wavefront 0: the query, 1: the step's key, 2: its value; lane l holds elements 4 l .. + 3
                const float *rope = S.rope + (int)word_of(ent, kRope) * HD + (lane * 4) % (HD / 2);
                const float4 c = *reinterpret_cast<const float4 *>(rope), sn = *reinterpret_cast<const float4 *>(rope + HD / 2);
                const int head = wave == 0 ? h : p.n_q + kvh + (wave == 2 ? p.n_kv : 0);
                const uint4 raw = take16(kResQ + (uint32_t)(head * HD + lane * 4));
                RES_STAMP(1);
                float a[4] = {__uint_as_float(raw.x), __uint_as_float(raw.y), __uint_as_float(raw.z), __uint_as_float(raw.w)};
                if (wave < 2) {
                    float sq = fmaf(a[3], a[3], fmaf(a[2], a[2], fmaf(a[1], a[1], a[0] * a[0])));
                    sq = lean_row_sum(sq);
                    if (HD == 256) sq = (lean_lane(sq, 0) + lean_lane(sq, 16)) + (lean_lane(sq, 32) + lean_lane(sq, 48));
                    if (HD == 128) sq = lean_lane(sq, 0) + lean_lane(sq, 16);
                    const float inv = rsqrtf(sq * (1.f / (float)HD) + p.eps);
                    const float w4n[4] = {head_w.x, head_w.y, head_w.z, head_w.w}, c4[4] = {c.x, c.y, c.z, c.w}, s4[4] = {sn.x, sn.y, sn.z, sn.w};
                    const bool low = lane < HD / 8;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float own = a[e] * inv * w4n[e], pair = __shfl_xor(own, HD / 8, 64);
                        a[e] = low ? own * c4[e] - pair * s4[e] : own * c4[e] + pair * s4[e];
                    }
                }
                if (wave == 0) {
                    __half hi[4], lo[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        rq[e] = a[e] * p.scale;
                        hi[e] = __float2half(rq[e]), lo[e] = __float2half(rq[e] - __half2float(hi[e]));
                    }
                    *reinterpret_cast<uint2 *>(S.qa + lane * 4) = *reinterpret_cast<const uint2 *>(hi);
                    *reinterpret_cast<uint2 *>(S.qa + QS + lane * 4) = *reinterpret_cast<const uint2 *>(lo);
                } else {
                    float *dst = wave == 1 ? S.kn : S.vn;   // as the cache will hold them
                    *reinterpret_cast<float4 *>(dst + lane * 4) = make_float4(__half2float(__float2half(a[0])), __half2float(__float2half(a[1])),
                                                                              __half2float(__float2half(a[2])), __half2float(__float2half(a[3])));
                }
            }
            RES_STAMP(5);
            res_stored();   // this workgroup's words of the next layer are empty before it hands anything over (and o's weights and the cache rows are here)
            RES_STAMP(28);
            if (ALL) load_units(w4, kAt4, weight(ent, 2, n4), 2);
            else load_kv(ent, v);
            RES_STAMP(29);
            __syncthreads();
            RES_STAMP(6);
            if (is_last) {
                if ((h & ((1 << p.lg_group) - 1)) == 0 && tid < HD) {   // one of the heads that share the kv head appends to its cache
                    static_cast<__half *>(ptr_of(ent, kCache))[((size_t)kvh * p.max_seq + pos) * HD + tid] = __float2half(S.kn[tid]);
                    static_cast<__half *>(ptr_of(ent, kCache + 1))[((size_t)kvh * HD + tid) * p.v_stride + pos] = __float2half(S.vn[tid]);
                }
                if (wave == 0) {
                    float dot = 0.f;
                    if (lane < HD / 4)
#pragma unroll
                        for (int e = 0; e < 4; e++) dot = fmaf(rq[e], S.kn[lane * 4 + e], dot);
                    dot = lean_wave_sum(dot);
                    if (lane == 0) S.sown = dot;
                }
            }
            rh16x8 aq[KS];
#pragma unroll
            for (int u = 0; u < KS; u++) {
                uint4 raw = make_uint4(0, 0, 0, 0);
                if (i16 < 2) raw = *reinterpret_cast<const uint4 *>(S.qa + i16 * QS + dq * 32 * KS + u * 32 + g4 * 8);
                aq[u] = __builtin_bit_cast(rh16x8, raw);
            }
            float m_run = NEG, l_run = 0.f;
            lf32x4 o[NB];
#pragma unroll
            for (int b = 0; b < NB; b++) o[b] = lf32x4{0.f, 0.f, 0.f, 0.f};
            auto pass = [&](int t0) {
                const bool more = t0 + kAttnPass < s.end;
                lf32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < KS; u++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(aq[u], __builtin_bit_cast(rh16x8, kreg[u]), acc, 0, 0, 0);
                if (g4 == 0) S.sp[wave][i16] = acc[0] + acc[1];
                if (more) load_k(rsrc_k(ent, false), kvh, t0 + kAttnPass);
                __syncthreads();
                const int t = lane & 31;   // both halves of the wavefront hold the pass's 32 positions
                float part[DQ];
#pragma unroll
                for (int q = 0; q < DQ; q++) part[q] = S.sp[(t >> 4) + 2 * q][t & 15];
                float sc = part[0];
#pragma unroll
                for (int q = 1; q < DQ; q++) sc += part[q];
                const bool valid = t0 + t >= s.first && t0 + t < hist_end;
                sc = valid ? sc : NEG;
                float mx = lean_row_max(sc);
                mx = fmaxf(m_run, fmaxf(lean_lane(mx, 0), lean_lane(mx, 16)));
                const float f = __expf(m_run - mx), e = valid ? __expf(sc - mx) : 0.f;
                if (lane < 32) {
                    const __half hi = __float2half(e);
                    S.pa[wave][t] = hi, S.pa[wave][PS + t] = __float2half(e - __half2float(hi));
                }
                const float es = lean_row_sum(e);
                l_run = fmaf(l_run, f, lean_lane(es, 0) + lean_lane(es, 16));
                m_run = mx;
                // the rows are this wavefront's own: its LDS operations complete in order, the compiler only must not reorder them
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                uint4 praw = make_uint4(0, 0, 0, 0);
                if (i16 < 2) praw = *reinterpret_cast<const uint4 *>(S.pa[wave] + i16 * PS + g4 * 8);
                const rh16x8 ap = __builtin_bit_cast(rh16x8, praw);
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    o[b][0] *= f, o[b][1] *= f;
                    o[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ap, __builtin_bit_cast(rh16x8, vreg[b]), o[b], 0, 0, 0);
                }
                if (more) {
                    load_v(rsrc_v(ent, false), kvh, t0 + kAttnPass);
                    __syncthreads();   // the next pass's scores must not overtake this pass's reads
                }
            };
            // (the first pass apart: its cache rows are here, and a loop that also waits for rows it asks for itself would
            // wait for gate|up's weights with them)
            if (s.begin < s.end) pass(s.begin);
            for (int t0 = s.begin + kAttnPass; t0 < s.end; t0 += kAttnPass) pass(t0);
            RES_STAMP(7);
            float f = 1.f, e_own = 0.f;
            if (is_last) {   // the step's own position
                const float so = S.sown, mx = fmaxf(m_run, so);
                f = __expf(m_run - mx), e_own = __expf(so - mx);
                m_run = mx, l_run = fmaf(l_run, f, e_own);
            }
            if (g4 == 0 && wave * 16 * NB < HD) {
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    const int ch = (wave * NB + b) * 16 + i16;
                    put(mine + kResA + (uint32_t)((v >> 3) * HD + ch), __float_as_uint(fmaf(o[b][0] + o[b][1], f, is_last ? e_own * S.vn[ch] : 0.f)), wide);
                }
                if (wave == 0 && i16 < 2) put(mine + kResML + (uint32_t)(2 * (v >> 3) + i16), __float_as_uint(i16 == 0 ? m_run : l_run), wide);
            }
            if (!ALL) __syncthreads();
        }
        RES_STAMP(8);
        // ---- o: the XCD's chunks joined (unnormalised), times the head's rows of o
        wp = row4(ent, 1), wi = row4(ent, 2);
        for (int v = first; v < end; v += step) {
            const uint32_t mine = (uint32_t)(v & 7) * kResLocal;
            const int h = (v & 7) >> p.lg_parts;
            uint4 ov[HD / 64], ml;
            bool again;
            do {
                res_reload();
                ml = lean_ld16<kAgent>(r_x, (mine + kResML + 4u * (uint32_t)i16) * 4u, cur);
#pragma unroll
                for (int i = 0; i < HD / 64; i++) ov[i] = lean_ld16<kAgent>(r_x, (mine + kResA + (uint32_t)(tid + kResThreads * i) * 4u) * 4u, cur);
                again = any_empty(ml);
#pragma unroll
                for (int i = 0; i < HD / 64; i++) again = again || any_empty(ov[i]);
            } while (again && --tries > 0);
            RES_STAMP(9);
            // lane i16 holds ranks 2 i16 and 2 i16 + 1
            const float m0 = __uint_as_float(ml.x), m1 = __uint_as_float(ml.z);
            const float M = lean_row_max(fmaxf(m0, m1));
            const float e0 = __expf(m0 - M), e1 = __expf(m1 - M);
            const float L = lean_row_sum(fmaf(__uint_as_float(ml.y), e0, __uint_as_float(ml.w) * e1));
            float4 a4 = zero4;
#pragma unroll
            for (int i = 0; i < HD / 64; i++) {
                float e;
                if (HD == 256) {   // a wavefront's 64 pieces are one rank's
                    const int row = wave + 8 * i;
                    e = (row & 1) ? lean_lane(e1, row >> 1) : lean_lane(e0, row >> 1);
                } else {
                    const int row = (tid + kResThreads * i) / (HD / 4);
                    const float ea = __shfl(e0, row >> 1, 64), eb = __shfl(e1, row >> 1, 64);
                    e = (row & 1) ? eb : ea;
                }
                a4.x = fmaf(__uint_as_float(ov[i].x), e, a4.x), a4.y = fmaf(__uint_as_float(ov[i].y), e, a4.y);
                a4.z = fmaf(__uint_as_float(ov[i].z), e, a4.z), a4.w = fmaf(__uint_as_float(ov[i].w), e, a4.w);
            }
            reinterpret_cast<float4 *>(S.join)[tid] = a4;   // [tid / (HD / 4)][HD]
            RES_STAMP(31);
            zero_red(1);
            __syncthreads();
            RES_STAMP(26);
            const int skip = (h * HD) % 128 / 4;            // a head of 64 channels is half of a k tile: the other half counts for nothing
            if (tid < KT3 * 32) {
                const int c = tid - skip;
                float4 sum = zero4;
                if (c >= 0 && c < HD / 4) {
                    float4 t[NJ];
#pragma unroll
                    for (int q = 0; q < NJ; q++) t[q] = reinterpret_cast<const float4 *>(S.join)[q * (HD / 4) + c];
#pragma unroll
                    for (int q = 0; q < NJ; q++) sum.x += t[q].x, sum.y += t[q].y, sum.z += t[q].z, sum.w += t[q].w;
                }
                split_terms4(tid, sum.x, sum.y, sum.z, sum.w);
            }
            __syncthreads();
            RES_STAMP(10);
            const int tiles = tiles3(v);
            multiply(w3, kAt3, ent, 1, n3, v, tiles * KT3, 1, unit3);
            RES_STAMP(11);
            __syncthreads();
            if (wave == 7) {
                const float s = column(1, lane);
                const uint32_t r = (uint32_t)(v >> 3), x = (uint32_t)(v & 7);
                if (lane < 2) put(kResM1 + 32u * r + 2u * x + (uint32_t)lane, __float_as_uint(lane == 0 ? M : L), true);
                if (lane < tiles * 16) put(kResG1 + r * 512u + x * 64u + (uint32_t)lane, __float_as_uint(s), true);
            }
            if (!ALL) __syncthreads();
        }
        RES_STAMP(12);
        if (ALL) load_units(w5, kAt5, weight(ent, 3, n5));
        if (wave == 6)
            for (int v = first; v < end; v += step)
                if (tiles3(v) > 0) combine(v, kResG1, kResY, true);
        RES_STAMP(13);
        // ---- gate | up of the row, and the gated row
        if (holds) {
            const uint4 raw = take16(home + kResY + (uint32_t)tid * 4u);
            y4 = make_float4(__uint_as_float(raw.x), __uint_as_float(raw.y), __uint_as_float(raw.z), __uint_as_float(raw.w));
        }
        RES_STAMP(14);
        if (ALL) load_kv(ent_next, first);   // (behind the last layer: its own again)
        RES_STAMP(25);
        norm_row(wp, wi);
        RES_STAMP(15);
        wp = row4(ent, 3), wi = row4(ent_next, 0);
        for (int v = first; v < end; v += step) {
            zero_red(2);
            multiply(w4, kAt4, ent, 2, n4, v, 2 * pairs4(v) * p.cg_h, 2, unit4);
            RES_STAMP(16);
            __syncthreads();
            if (wave == 7) {
                const int q = (lane >> 4) & 1;
                const float gate = column(2, 32 * q + i16), up = column(2, 32 * q + 16 + i16);
                const float g = pair_of(v, q) < p.pairs ? res_gelu(gate) * up : 0.f;   // columns past ffn: zeros
                uint16_t t[3];
                lean_split1<2>(g, t);
                if (lane < 16 * pairs4(v)) put((uint32_t)(v & 7) * kResLocal + kResH + (uint32_t)(((v >> 3) + 32 * q) * 16 + i16), (uint32_t)t[0] | ((uint32_t)t[1] << 16), wide);
            }
            if (!ALL) __syncthreads();
        }
        RES_STAMP(17);
        // ---- down: the XCD's slice of the gated row times its rows of the weight
        for (int v = first; v < end; v += step) {
            const int nk = slice_tiles(v);
            if (tid < nk * 32) {
                const uint4 w = take16((uint32_t)(v & 7) * kResLocal + kResH + (uint32_t)tid * 4u);
                put_terms(tid, make_uint2(__builtin_amdgcn_perm(w.y, w.x, 0x05040100u), __builtin_amdgcn_perm(w.w, w.z, 0x05040100u)),
                          make_uint2(__builtin_amdgcn_perm(w.y, w.x, 0x07060302u), __builtin_amdgcn_perm(w.w, w.z, 0x07060302u)));
            }
            RES_STAMP(18);
            RES_STAMP(24);
            zero_red(3);
            __syncthreads();
            RES_STAMP(19);
            const int tiles = tiles3(v);
            multiply(w5, kAt5, ent, 3, n5, v, tiles * nk, 3, unit5);
            if (ALL || v == first) load_ahead(ent_next);   // (behind the last layer: its own again)
            RES_STAMP(20);
            __syncthreads();
            if (wave == 7) {
                const float s = column(3, lane);
                if (lane < tiles * 16) put(kResG2 + (uint32_t)(v >> 3) * 512u + (uint32_t)(v & 7) * 64u + (uint32_t)lane, __float_as_uint(s), true);
            }
            if (!ALL) __syncthreads();
        }
        RES_STAMP(21);
        if (wave == 6)
            for (int v = first; v < end; v += step)
                if (tiles3(v) > 0) combine(v, kResG2, kResY2, false);
        RES_STAMP(22);
        if (holds && (l + 1 < p.n_layers || first == 0)) {
            const uint4 raw = take16(home + kResY2 + (uint32_t)tid * 4u);
            y4 = make_float4(__uint_as_float(raw.x), __uint_as_float(raw.y), __uint_as_float(raw.z), __uint_as_float(raw.w));
        }
        RES_STAMP(23);
        RES_STAMPS_OUT();
        cur = next;
        next = next == (kResSets - 1) * kResWords * 4u ? 0u : next + kResWords * 4u;
        ent = ent_next, ent_next = entry_of(l + 2);
    }
    if (first == 0 && holds) {
        *reinterpret_cast<float4 *>(p.x_out + tid * 4) = x4;
        *reinterpret_cast<float4 *>(p.y_out + tid * 4) = y4;
    }
}

// ALL: begins when all 256 workgroups have arrived, or not at all. Else: does the work of a launch of the other form that
// did not begin (`behind` is set), or that was never made, with the workgroups that have arrived by the deadline.
// (Two kernels: in one the second form costs the first 25 us a token, in registers. A launch that finds its work done is 2 us.)
template <int HD, int SG, bool ALL>
__global__ void __launch_bounds__(kResThreads) RES_ONE_PER_CU dec_resident_kernel(const ResidentArgs p) {
    __shared__ __attribute__((aligned(16))) ResShared<HD> S;
    const int pos = *p.pos;
    if (pos >= p.max_seq) return;   // the cache is full: the step is a no-op (the token pick reports it)
    int tries = p.polls;
    int first = blockIdx.x, n = gridDim.x;
    bool wide = false;
    uint32_t set = 0;
#ifndef HIPC_HOST_MODEL
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t epoch = p.sync[0];
    if (!ALL && p.behind && res_decided_for(p.sync[kResAll + kResDecision]) == kResGroups) return;   // done
    uint32_t *words = p.sync + (ALL ? kResAll : kResSome);
    if (ALL && tid == 0) {
        const uint32_t xcc = __builtin_amdgcn_s_getreg((31 << 11) | 20) & 15u;   // XCC_ID
        __hip_atomic_store(words + kResFlags + blockIdx.x, (epoch << 4) | xcc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!ALL) {
        uint32_t here = 0;
        if (tid == 0) S.decision[1] = res_join(words, gridDim.x, (unsigned long long)min(p.arrive, kJoinTicks), &here, tries), S.decision[0] = here;
    } else if (blockIdx.x != 0) {
        if (tid == 0) S.decision[0] = res_await(words, 2ull * (unsigned)p.arrive, tries);
    } else if (wave == 0) {
        const __amdgpu_buffer_rsrc_t r_s = lean_rsrc(words, kResSyncWords * 4u);
        const unsigned long long t0 = wall_clock64();
        const bool taken = lane == 0 && res_take(words);
        uint4 f;   // the flags of workgroups 4 lane ..
        bool all;
        do {
            res_reload();
            f = lean_ld16<kAgent>(r_s, (kResFlags + 4u * lane) * 4u, 0);
            const uint32_t want = epoch << 4;
            all = __all((f.x & ~15u) == want && (f.y & ~15u) == want && (f.z & ~15u) == want && (f.w & ~15u) == want);
        } while (!all && wall_clock64() - t0 < (unsigned long long)p.arrive);
        // one L2 per group: workgroups 8 j + x are group x, this lane holds groups 4 (lane & 1) ..
        const uint32_t gx = __shfl(f.x, lane & 1, 64), gy = __shfl(f.y, lane & 1, 64), gz = __shfl(f.z, lane & 1, 64), gw = __shfl(f.w, lane & 1, 64);
        const bool one_l2 = __all(f.x == gx && f.y == gy && f.z == gz && f.w == gw);
        if (lane == 0) {
            const uint32_t d = all && taken && p.arrive != 0 ? res_decision(kResGroups, one_l2) : res_decision(0, false);
            if (taken) __hip_atomic_store(words + kResDecision, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            S.decision[0] = d;
        }
    }
    __syncthreads();
    {
        const uint32_t d = __builtin_amdgcn_readfirstlane(S.decision[0]);
        if (ALL) {
            if (res_decided_for(d) != kResGroups) {   // the launch does not begin
                if (tries <= 0) *p.broken = 1;
                return;
            }
            wide = p.wide || !(d & 1u);
        } else {
            const uint32_t rank = __builtin_amdgcn_readfirstlane(S.decision[1]);
            if (rank == kResNoRank) {   // ... has begun without this workgroup
                if (tries <= 0) *p.broken = 1;
                return;
            }
            first = (int)rank, n = (int)d, wide = true;
        }
    }
    set = (epoch % kResSets) * ((uint32_t)p.n_layers % kResSets) % kResSets;
#endif
    res_layers<HD, SG, ALL>(p, S, first, n, wide, set, pos, tries);
    if (tries <= 0) *p.broken = 1;
}

__global__ void resident_set_layer_kernel(ResidentLayer *entry, const ResidentLayer value) {
    if (threadIdx.x == 0) *entry = value;
}
__global__ void __launch_bounds__(256) resident_clear_kernel(uint32_t *xch, uint32_t *sync) {
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < kResSets * kResWords; i += gridDim.x * 256) xch[i] = kEmpty;
    if (blockIdx.x == 0)
        for (uint32_t i = threadIdx.x; i < kResSync; i += 256) sync[i] = i == 0 ? 1u : 0u;
}

}  // namespace hipc

using namespace hipc;

#ifdef HIPC_PHASE_STAMPS
extern "C" int hipc_debug_resident_stamps(void *dst, size_t bytes) {
    return (int)hipMemcpyFromSymbol(dst, HIP_SYMBOL(hipc::res_stamps), bytes, 0, hipMemcpyDeviceToHost);
}
#endif

// Heads that divide the eight XCDs, a hidden row the 512 threads hold, k tiles that fit the reduction area (16) and a gated
// slice that fits its words (8 k tiles an XCD).
bool hipc::resident_takes(const hipc_decoder_config &c) {
    const int64_t cg_f = ceil_div(c.ffn, 128);
    return (c.n_q_heads == 1 || c.n_q_heads == 2 || c.n_q_heads == 4 || c.n_q_heads == 8) && (c.head_dim == 64 || c.head_dim == 128 || c.head_dim == 256) &&
           (c.n_q_heads + 2 * c.n_kv_heads) * c.head_dim <= (int)kResMaxQkv && c.hidden % 16 == 0 && c.hidden <= (int)kResMaxHidden && c.ffn % 16 == 0 && cg_f <= 64;
}

// One launch against five per layer: the 256 workgroups read each query head's positions themselves (no more than 8 / heads
// parts of them), where the attention launch spreads them over as many workgroups as it likes, and heads that share a kv head
// there share its reading. So heads and positions decide, whatever the other sizes are. Per product / one launch, us a token of 8 layers (query
// / kv heads of channels, hidden / ffn, at position):
//   8/1 of 256, 2048 / 8192     272 / 259 at 8192, 292 / 308 at 12288, 314 / 350 at 16384
//   8/2 of 64, 512 / 2048       162 / 156 at 8192, 169 / 179 at 12288, 178 / 201 at 16384
//   8/4 of 256, 1152 / 6912     284 / 269 at 12288, 311 / 318 at 16384
//   8/8 of 128, 1024 / 4096     204 / 184 at 8192, 240 / 222 at 12288, 258 / 258 at 16384
//   4/1 of 256, 1152 / 6912     246 / 212 at 16384, 330 / 308 at 32768;  4/4 of 128, 512 / 2048  276 / 251 at 32768
//   2/1 of 128, 512 / 2048      353 / 224 at 65536;  1/1 of 256, 1152 / 6912  804 / 339 at 131072
// and at position 100 one launch takes about three quarters. The position is the device's and a recorded step covers all of
// them, so the rule is on the longest one: no position of a decoder that takes one launch is slower for it.
// Only where every workgroup has a CU: with fewer, all steps would be the stand-in's, whose workgroups take shares in turn (gemma3-1b
// at 2048: 832 us a token with 255 workgroups, 990 with 128, 1680 with 64; 654 by the launches per product, 452 in one launch).
bool hipc::resident_pays(hipc_ctx *ctx, const hipc_decoder_config &c) {
    const int64_t most = c.n_q_heads <= 4 ? 131072 / c.n_q_heads : c.n_kv_heads >= 4 ? 12288 : 8192;
    return ctx->cu_count >= (int)kResGroups && c.max_seq <= most;
}

namespace {

template <int HD, bool ALL>
void launch_sg(hipc_ctx *ctx, int sg, const ResidentArgs &a, int workgroups) {
    switch (sg) {
        case 4: hipLaunchKernelGGL((dec_resident_kernel<HD, 4, ALL>), dim3(workgroups), dim3(kResThreads), 0, ctx->stream, a); break;
        case 2: hipLaunchKernelGGL((dec_resident_kernel<HD, 2, ALL>), dim3(workgroups), dim3(kResThreads), 0, ctx->stream, a); break;
        default: hipLaunchKernelGGL((dec_resident_kernel<HD, 1, ALL>), dim3(workgroups), dim3(kResThreads), 0, ctx->stream, a); break;
    }
}
template <bool ALL>
int launch_hd(hipc_ctx *ctx, int hd, int sg, const ResidentArgs &a, int workgroups) {
    switch (hd) {
        case 64: launch_sg<64, ALL>(ctx, sg, a, workgroups); break;
        case 128: launch_sg<128, ALL>(ctx, sg, a, workgroups); break;
        default: launch_sg<256, ALL>(ctx, sg, a, workgroups); break;
    }
    HIPC_LAUNCHED(ctx);
    return HIPC_OK;
}

}  // namespace

int hipc::resident_launch(hipc_ctx *ctx, const hipc_decoder_config &c, const ResidentArgs &args, int workgroups) {
    ResidentArgs a = args;
    a.hidden = c.hidden, a.cg_h = (int)ceil_div(c.hidden, 128), a.cg_o = (int)ceil_div((int64_t)c.n_q_heads * c.head_dim, 128);
    a.tiles_h = c.hidden / 16, a.tiles_qkv = (c.n_q_heads + 2 * c.n_kv_heads) * c.head_dim / 16;
    a.cg_f = (int)ceil_div(c.ffn, 128), a.pairs = c.ffn / 16;
    a.n_layers = c.n_layers, a.n_q = c.n_q_heads, a.n_kv = c.n_kv_heads;
    a.lg_group = __builtin_ctz((unsigned)(c.n_q_heads / c.n_kv_heads)), a.lg_parts = 3 - __builtin_ctz((unsigned)c.n_q_heads);
    a.max_seq = c.max_seq, a.v_stride = attn_v_stride(c.max_seq);
    a.inv_cg_h = (65536u + (uint32_t)a.cg_h - 1u) / (uint32_t)a.cg_h;
    a.inv_hidden = 1.f / (float)c.hidden;
    a.nib_mask = 0x000f000fu, a.magic = 0x43004300u;
    a.eps = c.rms_eps, a.scale = c.attn_scale > 0.f ? c.attn_scale : 1.f / sqrtf((float)c.head_dim);
    a.arrive = ctx->tune.dec_wait >= 0 ? ctx->tune.dec_wait : kArriveTicks;
    a.polls = ctx->tune.dec_polls > 0 ? ctx->tune.dec_polls : kPollBudget;
    a.wide = ctx->tune.dec_wide > 0;
    const int sg = c.block_size == 32 ? 4 : c.block_size == 64 ? 2 : 1;
    if (workgroups >= (int)kResGroups) {
        int rc = launch_hd<true>(ctx, c.head_dim, sg, a, kResGroups);
        if (rc != HIPC_OK) return rc;
        a.behind = 1, workgroups = kResGroups;   // (where it finds its work done, 256 workgroups that leave at once take no longer than 64)
    }
    return launch_hd<false>(ctx, c.head_dim, sg, a, workgroups);
}

int hipc::resident_set_layer(hipc_ctx *ctx, ResidentLayer *entry, const ResidentLayer &value) {
    hipLaunchKernelGGL((resident_set_layer_kernel), 1, 64, 0, ctx->stream, entry, value);
    HIPC_LAUNCHED(ctx);
    return HIPC_OK;
}

int hipc::resident_clear(hipc_ctx *ctx, uint32_t *xch, uint32_t *sync) {
    hipLaunchKernelGGL((resident_clear_kernel), 128, 256, 0, ctx->stream, xch, sync);
    HIPC_LAUNCHED(ctx);
    return HIPC_OK;
}
