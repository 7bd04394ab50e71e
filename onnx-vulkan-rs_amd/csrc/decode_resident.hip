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
// they are asked for ahead: weights (17 MB a layer are 68 KB a workgroup) into LDS, by wavefronts of their own; cache rows into registers.
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

#include <type_traits>

#include "internal.h"
#include "lanes.h"
#include "lean_ops.h"
#include "resident.h"
#include "row_digits.h"

namespace hipc {

#ifndef HIPC_HOST_MODEL
#define RES_ONE_PER_CU(all) __attribute__((amdgpu_waves_per_eu((all) ? 3 : 2, (all) ? 3 : 2)))   // three (two) wavefronts a SIMD: 168 (256) registers each
#else
#define RES_ONE_PER_CU(all)
#endif

// phase time stamps (library built with `make stamps` only; see gemv_lean.hip): res_stamps[workgroup][wavefront][phase] of one
// layer, kept in LDS until the layer's end (a store to memory would be waited for by the polls behind it)
#ifdef HIPC_PHASE_STAMPS
constexpr int kStampLayer = 12;
__device__ unsigned long long res_stamps[256 * 8 * 32];
#define RES_STAMP(ph)                                                                      \
    do {                                                                                   \
        const unsigned long long t_ = (unsigned long long)clock64();                       \
        if ((threadIdx.x & 63) == 0) S.stamp[threadIdx.x >> 6][ph] = (uint32_t)t_;                   \
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
// Beside other work, us a token of gemma3-1b at 2048, the launches per product / one launch (655 / 445 alone), on another stream without a
// pause: softmaxes of eight workgroups and a millisecond 766 / 511; of 64 workgroups and 220 us 783 / 612; of 128 and 140 us 844 / 585 (the
// softmaxes get on as well beside one launch as beside the other within a fifth); products of 4096^3 of 105 us, which let few small
// launches in between, 3400 / 764. Two decoders side by side, a token of each: 790 / 860; three 928 / 1660 to 2510, four 1585 /
// 2080 to 2720: launches that each want the whole chip take turns at best, where short ones fill each other's gaps, so contexts
// that decode at the same time are better off with HIPC_DEC_RESIDENT=0.
// The two waits are from the kernel before the present one, whose workgroups had eight wavefronts and 94 KB of LDS, so more could share a CU
// with them (launches per product / 50 us and 256 workgroups standing in / 200 us and 256 / 200 us and 64): beside the eight workgroups
// 763 / 773 / 923 / 1602, the 64 730 / 908 / 835 / 1191, the 128 788 / 777 / 570 / 569; three decoders 918 / 1900 / 2490 / 2060.
constexpr int kArriveTicks = 5000, kJoinTicks = 500;
constexpr int kResThreads = 512, kResWaves = 8;        // those that compute
constexpr int kFeedWaves = 4;                          // and, in the launch of all, those that bring the weights: one per product
constexpr int kResSlots = 104;                         // units of weights in LDS (see resident_launch)
constexpr int kRowPitch = 512;                         // bytes of a k tile of the row: four digits of 128 values
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
#define RES_TOGETHER() __builtin_amdgcn_sched_barrier(0)   // no instruction is moved across
#define RES_BARRIER()                  \
    do {                               \
        res_reload();                  \
        __builtin_amdgcn_s_barrier();  \
        res_reload();                  \
    } while (0)   // without a wait for anything
#else
inline void res_stored() {}
#define RES_TOGETHER() ((void)0)
#define RES_BARRIER() __syncthreads()
#endif

// A product is done in units: 128 k (a k tile) of 16 columns (a tile), 1 KB of weight. In the launch of all, four wavefronts of
// their own bring a workgroup's units into LDS (res_feed), one product's each, a whole layer ahead: what a phase has consumed is
// asked for again, for the next layer or for this one, as the product leaves its places. When matters: a CU's loads return in the order
// they were asked for, whichever wavefront asked, so a poll behind weights waits for HBM (measured: a poll of 0.09 us takes up to 1 us
// behind 4 KB of them, 1.5 us behind 36 KB). So they are asked for behind the barrier that follows a poll, with work in front
// of the next one: gate|up's where a layer begins (kFeedFirst units), behind the heads' barrier (up to kFeedHeads) and where
// the chunks have arrived; o's where a layer begins, down's where the hidden row has arrived, the next layer's q|k|v where
// the gated row has. Us for eight tokens of gemma3-1b at 2048 (a row as three bytes a value then): all of a product's at once as soon as its
// places are free 3955; so spread 3560; in the registers of the polling wavefronts, two phases ahead, 3725. (Eight layers of 2048 / 8192 with
// 8/1 heads of 256 at 2040, where those registers held half of the units: 201 -> 185; of 512 / 2048 with 8/2 heads of 64: 123 -> 119.)
//
// The row takes part as whole numbers of four signed bytes (row_digits.h has what that keeps of a value), so a product of a
// unit is two int8 matrix instructions with exact sums, and a weight's nibbles need no conversion beyond being spread to bytes.
// The 16 rows of the matrix operand are the four 32-k chunks times the digits: lane group g ends with the sums of chunk g.
// The digits' own sums, for the zero points, are whole numbers too, so a weight of zero takes nothing from its row's value. Two
// bf16 terms per value took twice the instructions a unit.
typedef int ri32x4 __attribute__((ext_vector_type(4)));

struct UnitWeight {
    uint4 w;
    float s;      // of the lane's column and chunk
    uint32_t z;   // 128 + zero point
};

// the place of column c in a row of words that others turn into digits: a thread takes four words, and the bytes of a digit
// lie as the nibbles of a weight do (0 4 1 5, 2 6 3 7), so bits 1 and 2 change places
__device__ __forceinline__ uint32_t res_place(uint32_t c) { return (c & ~6u) | ((c & 2u) << 1) | ((c & 4u) >> 1); }

template <int CTRL>
__device__ __forceinline__ uint32_t res_dpp(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true); }

// the sum over two neighbouring groups of 16 lanes, in both
__device__ __forceinline__ float res_rows_sum(float v) {
#ifndef HIPC_HOST_MODEL
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
#endif
    return v;
}

// the sum over the four groups of 16 lanes, in all lanes
__device__ __forceinline__ float res_groups_sum(float v) {
#ifndef HIPC_HOST_MODEL
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
#endif
    return res_rows_sum(v);
}

// 16 (4) bytes a lane from memory to LDS, without a register: lane l's to `to` + 16 (4) l
#ifndef HIPC_HOST_MODEL
#define RES_TO_LDS(BYTES, r, to, voff) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)(to), BYTES, (int)(voff), 0, 0, 0)
#else
#define RES_TO_LDS(BYTES, r, to, voff) gpu_model_load<BYTES>(r, (int)(voff), 0, 0, reinterpret_cast<char *>(to) + (threadIdx.x & 63) * BYTES)
#endif

// gelu_tanh: 0.5 v (1 + tanh u) = v / (1 + exp(-2 u)), without the difference that loses digits where tanh is near -1
__device__ __forceinline__ float res_gelu(float v) {
    return v / (1.f + __expf(-1.5957691216057308f * fmaf(0.044715f, v * v * v, v)));
}

// the LDS of a workgroup (the stand-in's, which loads weights where it uses them, fits beside other work's)
template <int HD, int SG, bool ALL>
struct ResShared {
    static constexpr int SLOTS = ALL ? kResSlots : 1;
    union {
        uint32_t row[16 * kRowPitch / 4];                // the row's digits: [k tile][digit, the highest first][128 bytes]
        struct {                                         // (between q|k|v and o)
            __half qa[2 * (HD + 8)];
            __half pa[kResWaves][2 * (kAttnPass + 8)];
            float sp[kResWaves][16];
            float kn[HD], vn[HD];
            float sown;
        };
    };
    int4 chunk[64];                                      // per 32 values: digits_unit(), their sum (two words)
    float4 red4[4 * kResWaves];
    union {
        float red[4 * kResWaves * 64];                   // a product: [tile][part of its k tiles][lane]
        float join[kResThreads * 4];                     // (between two products)
    };
    float rope[2 * HD];
    uint32_t decision[2];
#ifdef HIPC_PHASE_STAMPS
    uint32_t stamp[kResWaves][32];
#endif
    // (last: the others' offsets fit the instructions')
    alignas(16) float sc[SLOTS][16 * SG];
    uint8_t zb[SLOTS][16 * SG];
    uint4 wq[SLOTS][64];                                 // units: as in memory, lane by lane
};
static_assert(sizeof(ResShared<256, 4, true>) <= 160 * 1024, "a workgroup's LDS");

// ---- what a share v (of XCD v & 7, rank v >> 3) has of each product
__device__ __forceinline__ int res_tiles_qkv(const ResidentArgs &p, int v) { return (v < p.tiles_qkv) + (v + (int)kResGroups < p.tiles_qkv); }   // v, v + 256
__device__ __forceinline__ int res_tiles_h(const ResidentArgs &p, int v) { return (p.tiles_h - (v >> 3) + 31) >> 5; }                             // of the hidden row: r, r + 32, ..
__device__ __forceinline__ int res_slice_tiles(const ResidentArgs &p, int v) { return (p.cg_f - (v & 7) + 7) >> 3; }                              // down's k tiles of the XCD
__device__ __forceinline__ int res_pairs(const ResidentArgs &p, int v) {   // (gate, up) pairs: eight per k tile of the slice; r, r + 32
    const int m = res_slice_tiles(p, v) * 8;
    return ((v >> 3) < m) + ((v >> 3) + 32 < m);
}
__device__ __forceinline__ int res_pair(const ResidentArgs &p, int v, int q) {   // global pair, or p.pairs: nothing there
    const int lp = (v >> 3) + 32 * q;
    return min(((v & 7) + 8 * (lp >> 3)) * 8 + (lp & 7), p.pairs);
}
// A share of product `ph`: `tiles` tiles of `kts` k tiles each; unit (t, kt) is number t * kts + kt.
template <int HD>
struct ResShare {
    int v, ph, tiles, kts;
    __device__ __forceinline__ ResShare(const ResidentArgs &p, int v_, int ph_) : v(v_), ph(ph_) {
        tiles = ph == 0 ? res_tiles_qkv(p, v) : ph == 2 ? 2 * res_pairs(p, v) : res_tiles_h(p, v);
        kts = ph == 1 ? (HD >= 128 ? HD / 128 : 1) : ph == 3 ? res_slice_tiles(p, v) : p.cg_h;
    }
    __device__ __forceinline__ bool has(const ResidentArgs &p, int t) const { return ph != 2 || res_pair(p, v, t >> 1) < p.pairs; }
    __device__ __forceinline__ uint32_t at(const ResidentArgs &p, int t, int kt) const {   // which 128 k x 16 columns of the weight
        const int r = v >> 3, x = v & 7;
        if (ph == 0) return (uint32_t)((v + (int)kResGroups * t) * p.cg_h + kt);
        if (ph == 1) return (uint32_t)((r + 32 * t) * p.cg_o + ((x >> p.lg_parts) * HD) / 128 + kt);
        if (ph == 2) return (uint32_t)((2 * res_pair(p, v, t >> 1) + (t & 1)) * p.cg_h + kt);
        return (uint32_t)((r + 32 * t) * p.cg_f + x + 8 * kt);
    }
};
__device__ __forceinline__ uint32_t res_units(const ResidentArgs &p, int ph) {   // of the whole weight
    return (uint32_t)(ph == 0 ? p.tiles_qkv * p.cg_h : ph == 1 ? p.tiles_h * p.cg_o : ph == 2 ? 2 * p.pairs * p.cg_h : p.tiles_h * p.cg_f);
}

// the cache positions of share v: its part of its head's context, 32 at a time
struct ResSpan {
    int begin, end, first;
    bool dead;
    __device__ __forceinline__ ResSpan(const ResidentArgs &p, int v, int total, int window) {
        const int base = attn_base(total, window), lg = p.lg_parts + 10;   // kAttnPass * kResRanks positions a part
        static_assert(kAttnPass * kResRanks == 1 << 10, "positions of a part per pass");
        const int chunk = kAttnPass * max(1, (total - base + (1 << lg) - 1) >> lg);
        begin = base + (((v & 7) & ((1 << p.lg_parts) - 1)) * (int)kResRanks + (v >> 3)) * chunk;
        dead = begin >= total;
        end = min(total, begin + chunk);
        first = attn_first(total, window);
    }
    __device__ __forceinline__ int barriers() const {   // that the passes take: one, and two for each further pass
        const int passes = dead ? 0 : (end - begin + kAttnPass - 1) / kAttnPass;
        return max(0, 2 * passes - 1);
    }
};

// The wavefronts that bring the weights of the launch of all: wavefront `ph` those of product `ph`. It passes the barriers the
// computing wavefronts do, asks for weights behind some of them, and waits for them before the one that opens the product.
// Which units these are does not change: their offsets stay in registers, and each of the four wavefronts has code of its own for
// the fixed places where it asks, so that four units take twelve instructions and the next barrier, which may be 0.3 us away, does
// not wait for this wavefront (one code for all, which skipped what it did not ask for: 3860 us instead of 3560).
// kFeedFirst: as many of gate|up's places are no place of q|k|v's, whose units lie behind them (up to 32, see resident_launch), so
// these can be asked for while q|k|v's product is still to come. kFeedHeads: what the short work in front of the cache passes covers.
// A larger q|k|v share or window moves neither: the places stay free, longer passes leave the later ones more time. Us a token with
// 16/24, 16/16, 16/32, 8/16, 24/24, 24/32: gemma3-1b at 2048 (a vocabulary of 4096) 412 411 421 415 414 415; at 8000, 22 layers with windows
// of 512, 398 392 405 400 395 401; eight layers at 2040 of 2048 / 8192 with 8/1 heads of 256 180 180 181 182 178 178, with 8/8 (two
// tiles of q|k|v a workgroup) 193 195 194 196 192 192; of 1024 / 4096 with 4/4 of 128 121 123 121 121 124 121; of 1152 / 6912 at 16000 220 222
// 225 222 222 223.
constexpr int kFeedFirst = 16, kFeedHeads = 24;
template <int HD, int SG, int ph>
__device__ __forceinline__ void res_feed(const ResidentArgs &p, ResShared<HD, SG, true> &S, const int v, const int total) {
    constexpr int MOST = ph == 0 ? 32 : ph == 1 ? 8 : ph == 2 ? 64 : 32;   // units of a share
    const int lane = threadIdx.x & 63;
    const ResShare<HD> share(p, v, ph);
    const int base = p.slot[ph], units = share.tiles * share.kts;
    const uint32_t tiles = res_units(p, ph);
    constexpr uint32_t none = 0xffff0000u;   // past the end of everything: zeros, and no traffic
    uint32_t o_q[MOST], o_s[MOST / 4];   // (a zero point's is a quarter of its scale's)
    {
        const uint32_t part = (uint32_t)lane / (4 * SG), in = (uint32_t)lane % (4 * SG);   // of four units' scales: whose, and which 16 (4) bytes
        // (tile by tile: worked out unit by unit these would take microseconds of every launch)
        const uint32_t row0 = share.has(p, 0) ? share.at(p, 0, 0) : none, row1 = share.has(p, 1) ? share.at(p, 1, 0) : none;
        const uint32_t row2 = share.has(p, 2) ? share.at(p, 2, 0) : none, row3 = share.has(p, 3) ? share.at(p, 3, 0) : none;
        auto row_of = [&](int t) { return t == 0 ? row0 : t == 1 ? row1 : t == 2 ? row2 : row3; };
        const int kstep = ph == 3 ? 8 : 1;
        int t = 0, kt = 0;
        uint32_t row = row0;
#pragma unroll
        for (int u = 0; u < MOST; u++) {
            if (u % 4 == 0 && u >= units) break;
            const bool live = u < units && row != none;
            const uint32_t tl = row + (uint32_t)(kt * kstep);
            o_q[u] = live ? tl * 1024u + (uint32_t)lane * 16u : none;
            if (u % 4 == 0) o_s[u / 4] = none;
            if (live && part == (uint32_t)(u % 4)) o_s[u / 4] = tl * 64u * SG + in * 16u;
            if (++kt == share.kts) kt = 0, t++, row = row_of(t);
        }
    }
    struct Entry {
        const void *q, *s, *z;
        int window;
    };
    auto entry = [&](int l) {
#ifndef HIPC_HOST_MODEL
        const auto *e = (const __attribute__((address_space(4))) ResidentLayer *)(uintptr_t)(p.table + min(l, p.n_layers - 1));   // (scalar loads: they wait for no weights)
#else
        const ResidentLayer *e = p.table + min(l, p.n_layers - 1);
#endif
        return Entry{e->wq[ph], e->sc[ph], e->zb[ph], e->window};
    };
    auto ask = [&](const Entry &e, auto from, auto to) {   // units from .. to - 1, in whole fours
        const __amdgpu_buffer_rsrc_t q = lean_rsrc(e.q, tiles * 1024u), s = lean_rsrc(e.s, tiles * 64u * SG), z = lean_rsrc(e.z, tiles * 16u * SG);
#pragma unroll
        for (int u = decltype(from)::value; u < decltype(to)::value; u += 4) {
            if (u >= units) break;
#pragma unroll
            for (int i = 0; i < 4; i++) RES_TO_LDS(16, q, S.wq[base + u + i], o_q[u + i]);
            if (lane < 16 * SG) {
                RES_TO_LDS(16, s, S.sc[base + u], o_s[u / 4]);
                RES_TO_LDS(4, z, S.zb[base + u], o_s[u / 4] >> 2);
            }
        }
    };
    Entry e = entry(0), e_next = entry(1);
    constexpr std::integral_constant<int, 0> none_yet{};
    constexpr std::integral_constant<int, kFeedFirst> first{};
    constexpr std::integral_constant<int, kFeedHeads> second{};
    constexpr std::integral_constant<int, MOST> all{};
    if (ph == 0) ask(e, none_yet, all);
    RES_BARRIER();   // (the one in front of the layers)
    for (int l = 0; l < p.n_layers; l++) {
        const int inner = ResSpan(p, v, total, e.window).barriers();
        const int opens = ph == 0 ? 1 : ph == 1 ? 5 + inner : ph == 2 ? 8 + inner : 10 + inner;   // the barrier in front of the product
        for (int b = 0; b < 12 + inner; b++) {
            if (b == opens) res_stored();   // (here: what was asked for has arrived)
            RES_BARRIER();
            if constexpr (ph == 0) {
                if (b == 10 + inner && l + 1 < p.n_layers) ask(e_next, none_yet, all);
            } else if constexpr (ph == 1) {
                if (b == 0) ask(e, none_yet, all);
            } else if constexpr (ph == 2) {
                if (b == 0) ask(e, none_yet, first);
                if (b == 3) ask(e, first, second);
                if (b == 4 + inner) ask(e, second, all);
            } else {
                if (b == 7 + inner) ask(e, none_yet, all);
            }
        }
        e = e_next;
        e_next = entry(l + 2);
    }
}

// The work of a launch. ALL: the 256 workgroups are there and workgroup v does share v of every phase, with the weights in LDS.
// Else `n` workgroups take the shares in turn and load weights where they use them.
// (In the launch of all the loops over shares run once. They stay loops to the compiler, which otherwise moves instructions from phase
// to phase: 3570 against 3650 to 3800 us for eight tokens of gemma3-1b.)
#define RES_SHARES(v) for (int v = first, step_ = ALL ? (int)kResGroups : n, end_ = ALL ? mine + 1 : (int)kResGroups; v < end_; v += step_)
template <int HD, int SG, bool ALL>
__device__ __forceinline__ void res_layers(const ResidentArgs &p, ResShared<HD, SG, ALL> &S, int first, const int n, const bool wide, uint32_t set, const int pos, int &tries) {
    constexpr int KT3 = HD >= 128 ? HD / 128 : 1;  // k tiles of a head in o's weight (half of one at 64 channels)
    constexpr int KS = HD >= 128 ? HD / 128 : 1;   // 32-channel steps of a wavefront's share of the scores
    constexpr int DQ = HD / (32 * KS);             // wavefronts that share the channels of the scores
    constexpr int NB = HD >= 128 ? HD / 128 : 1;   // 16-channel blocks of a wavefront's outputs
    constexpr int QS = HD + 8, PS = kAttnPass + 8; // halfs per operand row (16 bytes of padding)
    constexpr int NJ = kResThreads * 4 / HD;       // rows of chunks that are joined side by side
    constexpr float NEG = -3.0e38f;

    int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int i16 = lane & 15, g4 = lane >> 4;
    const int total = pos + 1, mine = first;
    const __amdgpu_buffer_rsrc_t r_x = lean_rsrc(p.xch, kResSets * kResWords * 4u);

    // ---- the layer's entry: lane i holds word i of it, a pointer is read from two lanes. (Scalar loads would miss the
    // scalar cache once per phase.) The next layer's is asked for a layer ahead.
    auto entry_of = [&](int l) {
#ifndef HIPC_HOST_MODEL
        return reinterpret_cast<const uint32_t *>(p.table + min(l, p.n_layers - 1))[min(lane, kEntryWords - 1)];
#else
        return (uint32_t)l;
#endif
    };
    uint32_t ent = entry_of(0), ent_next = entry_of(1), ent_after = ent_next;
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

    auto tiles1 = [&](int v) { return res_tiles_qkv(p, v); };
    auto tiles3 = [&](int v) { return res_tiles_h(p, v); };
    auto slice_tiles = [&](int v) { return res_slice_tiles(p, v); };
    auto pairs4 = [&](int v) { return res_pairs(p, v); };

    // ---- products
    // NT tiles of a product, t0 .. t0 + NT - 1, over its k tiles kt0, kt0 + step, .. (once: there is no second): this lane's sums
    // for its chunk go to `part`
    auto multiply = [&](auto nt, auto once, int ph, uint32_t e, const ResShare<HD> &share, int t0, int kt0, int step, int part) {
        constexpr int NT = decltype(nt)::value;
        float acc[NT];
#pragma unroll
        for (int j = 0; j < NT; j++) acc[j] = 0.f;
        const int mine = i16 >> 2;
        const char *row = reinterpret_cast<const char *>(S.row) + (i16 & 3) * 128 + mine * 32 + g4 * 8;
        const int4 *chunk = S.chunk + g4;
        const uint32_t m0 = mine == 0 ? ~0u : 0u, m1 = mine == 1 ? ~0u : 0u, m2 = mine == 2 ? ~0u : 0u, m3 = mine == 3 ? ~0u : 0u;
        const int sg = SG == 4 ? g4 : SG == 2 ? g4 >> 1 : 0;
        struct Operands {
            uint2 a;     // the lane's digits of the row
            int4 c;
            UnitWeight w[NT];
        };
        auto row_here = [&](Operands &o, int kt) { o.a = *reinterpret_cast<const uint2 *>(row + kt * kRowPitch), o.c = chunk[kt * 4]; };
        auto product = [&](const Operands &o, const UnitWeight &w, float sum) {
            constexpr uint32_t F = 0x0f0f0f0fu;
            const ri32x4 a0 = {(int)(o.a.x & m0), (int)(o.a.y & m0), (int)(o.a.x & m1), (int)(o.a.y & m1)}, a1 = {(int)(o.a.x & m2), (int)(o.a.y & m2), (int)(o.a.x & m3), (int)(o.a.y & m3)};
            const uint4 q = w.w;
            const ri32x4 b0 = {(int)(q.x & F), (int)((q.x >> 4) & F), (int)(q.y & F), (int)((q.y >> 4) & F)}, b1 = {(int)(q.z & F), (int)((q.z >> 4) & F), (int)(q.w & F), (int)((q.w >> 4) & F)};
            ri32x4 d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, b0, ri32x4{0, 0, 0, 0}, 0, 0, 0);
            d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, b1, d, 0, 0, 0);
            const int nz = 128 - (int)(w.z & 255u);
            const float f = digits_join(d[0] * 256 + d[1] + __mul24(nz, o.c.y), d[2] * 256 + d[3] + __mul24(nz, o.c.z));
            return fmaf(w.s * __builtin_bit_cast(float, o.c.x), f, sum);
        };
        if (ALL) {
            if (kt0 < share.kts) {
                Operands o;
                auto load = [&](int kt) {
                    row_here(o, kt);
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        const int at = p.slot[ph] + (t0 + j) * share.kts + kt;
                        o.w[j] = UnitWeight{S.wq[at][lane], S.sc[at][i16 * SG + sg], S.zb[at][i16 * SG + sg]};
                    }
                };
                load(kt0);
#pragma unroll 1
                for (int kt = kt0 + step; !decltype(once)::value && kt < share.kts; kt += step) {
                    const Operands now = o;
                    load(kt);
#pragma unroll
                    for (int j = 0; j < NT; j++) acc[j] = product(now, now.w[j], acc[j]);
                }
#pragma unroll
                for (int j = 0; j < NT; j++) acc[j] = product(o, o.w[j], acc[j]);
            }
        } else {
#pragma unroll 1
            for (int j = 0, kt = kt0; j < NT && kt0 < share.kts; kt = kt + step < share.kts ? kt + step : (j++, kt0)) {
                if (t0 + j >= share.tiles) break;
                Operands o;
                row_here(o, kt);
                const uint32_t tl = share.at(p, t0 + j, kt), all = res_units(p, ph);
                UnitWeight w;
                w.w = lean_ld16(lean_rsrc(ptr_of(e, ph), all * 1024u), (uint32_t)lane * 16u, tl * 1024u);
                w.s = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(lean_rsrc(ptr_of(e, 4 + ph), all * 64u * SG), (int)((i16 * SG + sg) * 4), (int)(tl * 64u * SG), 0));
                w.z = __builtin_amdgcn_raw_buffer_load_b8(lean_rsrc(ptr_of(e, 8 + ph), all * 16u * SG), i16 * SG + sg, (int)(tl * 16u * SG), 0);
                const float r = product(o, w, 0.f);
#pragma unroll
                for (int i = 0; i < NT; i++)
                    if (i == j) acc[i] += r;
            }
        }
#pragma unroll
        for (int j = 0; j < NT; j++) S.red[((t0 + j) * kResWaves + part) * 64 + lane] = acc[j];
    };
    // the sum of tile t's columns over `parts` parts: column i16's, in all lanes
    auto tile_sum = [&](int t, int parts) {
        const float *r = S.red + t * kResWaves * 64 + lane;
        float s = r[0];
        if (parts >= 2) s += r[64];
        if (parts >= 4) s += r[128] + r[192];
        if (parts >= 8) s += (r[256] + r[320]) + (r[384] + r[448]);
        return res_groups_sum(s);
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    using Three = std::integral_constant<int, 3>;
    using Four = std::integral_constant<int, 4>;

    // ---- the cache rows of a share's positions: 32 at a time
    struct CacheRows {
        uint4 k[KS], v[NB];
    };
    CacheRows kv;
    const int pb = wave & 1, dq = min(wave >> 1, DQ - 1);
    const uint32_t v_k = (uint32_t)((pb * 16 + i16) * HD + dq * 32 * KS + g4 * 8) * 2u;
    const uint32_t v_v = ((uint32_t)(min(wave * 16 * NB, HD - 16 * NB) + i16) * (uint32_t)p.v_stride + (uint32_t)(g4 * 8)) * 2u;
    auto load_k = [&](__amdgpu_buffer_rsrc_t r, int kvh, int t0) {
        const uint32_t s_k = ((uint32_t)kvh * (uint32_t)p.max_seq + (uint32_t)t0) * HD * 2u;
#pragma unroll
        for (int u = 0; u < KS; u++) kv.k[u] = lean_ld16(r, v_k + u * 64u, s_k);
    };
    auto load_v = [&](__amdgpu_buffer_rsrc_t r, int kvh, int t0) {
#pragma unroll
        for (int b = 0; b < NB; b++) kv.v[b] = lean_ld16(r, v_v, (((uint32_t)kvh * HD + b * 16u) * (uint32_t)p.v_stride + (uint32_t)t0) * 2u);
    };
    auto rsrc_k = [&](uint32_t e, bool dead) { return lean_rsrc(ptr_of(e, kCache), dead ? 0u : ((uint32_t)p.n_kv * (uint32_t)p.max_seq + 64u) * HD * 2u); };
    auto rsrc_v = [&](uint32_t e, bool dead) { return lean_rsrc(ptr_of(e, kCache + 1), dead ? 0u : (uint32_t)p.n_kv * HD * (uint32_t)p.v_stride * 2u); };
    auto load_kv = [&](uint32_t e, int v) {
        const ResSpan s(p, v, total, (int)word_of(e, kWindow));
        const int kvh = ((v & 7) >> p.lg_parts) >> p.lg_group, t0 = s.dead ? 0 : s.begin;   // (the scalar offset stays inside whatever the descriptor says)
        load_k(rsrc_k(e, s.dead), kvh, t0), load_v(rsrc_v(e, s.dead), kvh, t0);
    };
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    // norm weights of the heads: the query's for wavefront 0, the key's for wavefront 1; asked for a layer ahead. (A load under a
    // condition would be waited for where the condition ends: none of the loads ahead has one.)
    float4 head_w = zero4;
    auto load_head_w = [&](uint32_t e) {
        head_w = __builtin_bit_cast(float4, lean_ld16(lean_rsrc(ptr_of(e, kNorm + 4 + (wave & 1)), HD * 4u), (uint32_t)lane * 16u, 0));
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
    // four values of the row (words 4 i4 .. of it, see res_place) as digits into LDS; eight neighbouring threads make a chunk.
    // (The sums of the digits from two more matrix instructions against ones per k tile, instead of here: 3710 against 3610 us
    // for eight tokens of gemma3-1b at 2048.)
    auto put_digits = [&](int i4, float a, float b, float c, float d) {
        uint32_t mx = __float_as_uint(__builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(a), fabsf(b)), __builtin_elementwise_maximum(fabsf(c), fabsf(d))));
        mx = max(mx, res_dpp<0xB1>(mx));
        mx = max(mx, res_dpp<0x4E>(mx));
        mx = max(mx, res_dpp<0x141>(mx));   // row_half_mirror: the other quad of the eight
        const uint32_t ex = digits_exponent(mx);
        const float to = digits_scale(ex);
        const uint32_t q0 = digits_of(a * to), q1 = digits_of(c * to), q2 = digits_of(b * to), q3 = digits_of(d * to);   // (in the order of the bytes)
        const uint32_t lo01 = __builtin_amdgcn_perm(q1, q0, 0x05010400u), lo23 = __builtin_amdgcn_perm(q3, q2, 0x05010400u);
        const uint32_t hi01 = __builtin_amdgcn_perm(q1, q0, 0x07030602u), hi23 = __builtin_amdgcn_perm(q3, q2, 0x07030602u);
        uint32_t *dst = S.row + (i4 >> 5) * (kRowPitch / 4) + (i4 & 31);
        const uint32_t w0 = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u), w1 = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
        const uint32_t w2 = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u), w3 = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
        dst[0] = w0, dst[32] = w1, dst[64] = w2, dst[96] = w3;
        auto sum4 = [](uint32_t w, int more) { return __builtin_amdgcn_sdot4((int)w, 0x01010101, more, false); };
        uint32_t hi = (uint32_t)sum4(w1, sum4(w0, 0) * 256), lo = (uint32_t)sum4(w3, sum4(w2, 0) * 256);
        hi += res_dpp<0xB1>(hi), lo += res_dpp<0xB1>(lo);
        hi += res_dpp<0x4E>(hi), lo += res_dpp<0x4E>(lo);
        hi += res_dpp<0x141>(hi), lo += res_dpp<0x141>(lo);
        if ((i4 & 7) == 0) S.chunk[i4 >> 3] = make_int4(__builtin_bit_cast(int, digits_unit(ex)), (int)hi, (int)lo, 0);
    };
    // stream += rmsnorm(branch, w_post); the row rmsnorm(stream, w_in) goes to LDS. One reduction for both norms (see mmnb_lean_kernel).
    float4 x4 = zero4, y4 = zero4;   // this thread's four values of the stream, and of the branch to be added
    const bool holds = tid * 4 < p.hidden;
    auto place = [&] { return (tid >> 1) * 8 + (tid & 1) * 2; };   // its first value's column; the others: + 1, + 4, + 5
    if (holds) {
        const float2 lo = *reinterpret_cast<const float2 *>(p.x_in + place()), hi = *reinterpret_cast<const float2 *>(p.x_in + place() + 4);
        x4 = make_float4(lo.x, lo.y, hi.x, hi.y);
    }
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
            const float4 r = S.red4[lane & 31];   // (zeros behind the wavefronts that hold parts)
            const float r_yy = lean_row_sum(r.x), r_xx = lean_row_sum(r.y), r_xy = lean_row_sum(r.z), r_ww = lean_row_sum(r.w);
            const float t_yy = res_rows_sum(r_yy), t_xx = res_rows_sum(r_xx), t_xy = res_rows_sum(r_xy), t_ww = res_rows_sum(r_ww);
            const float f1 = rsqrtf(t_yy * p.inv_hidden + p.eps);
            const float sq2 = fmaf(f1 * f1, t_ww, fmaf(2.f * f1, t_xy, t_xx));
            const float f2 = rsqrtf(fmaxf(sq2, 0.f) * p.inv_hidden + p.eps);
            x4.x = fmaf(yw.x, f1, x4.x), x4.y = fmaf(yw.y, f1, x4.y), x4.z = fmaf(yw.z, f1, x4.z), x4.w = fmaf(yw.w, f1, x4.w);
            if (tid < p.cg_h * 32) put_digits(tid, x4.x * f2 * wi.x, x4.y * f2 * wi.y, x4.z * f2 * wi.z, x4.w * f2 * wi.w);
        }
        __syncthreads();
    };
    auto row4 = [&](uint32_t e, int which) {   // (past the row: zeros)
        const __amdgpu_buffer_rsrc_t r = lean_rsrc(ptr_of(e, kNorm + which), (uint32_t)p.hidden * 4u);
        const float2 lo = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, place() * 4, 0, 0)), hi = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, place() * 4 + 16, 0, 0));
        return make_float4(lo.x, lo.y, hi.x, hi.y);
    };
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
        if (lane < cols) put((uint32_t)x * kResLocal + to + res_place((uint32_t)((r + 32 * g4) * 16 + i16)), __float_as_uint(y), wide);
    };
    const uint32_t home = (uint32_t)(first & 7) * kResLocal;   // where this workgroup reads rows all XCDs hold

    for (int i = tid; i < 2 * HD; i += kResThreads) S.rope[i] = p.rope[i];
    if (tid < 4 * kResWaves) S.red4[tid] = zero4;
    if (ALL) load_kv(ent, first);
    load_head_w(ent);
    float4 wp = zero4, wi = zero4, wp1 = zero4, wi1 = row4(ent, 0);   // of the norm in the middle of a layer, and where one begins
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
        norm_row(wp1, wi1);
        RES_STAMP(2);
        RES_SHARES(v) {
            const ResShare<HD> share(p, v, 0);
            const int parts = share.tiles == 2 ? 4 : 8;
            if (share.tiles > 0) multiply(One{}, std::false_type{}, 0, ent, share, share.tiles == 2 ? wave >> 2 : 0, wave & (parts - 1), parts, wave & (parts - 1));
            RES_STAMP(3);
            __syncthreads();
            if (wave >= 4 && wave - 4 < share.tiles) {
                const float s = tile_sum(wave - 4, parts);
                if (lane < 16) put(kResQ + (uint32_t)((v + (int)kResGroups * (wave - 4)) * 16 + lane), __float_as_uint(s), true);
            }
            clear(v);
            if (!ALL) __syncthreads();
        }
        RES_STAMP(4);
        // ---- attention: the share's positions for the XCD's head
        RES_SHARES(v) {
            const uint32_t mine = (uint32_t)(v & 7) * kResLocal;
            const int h = (v & 7) >> p.lg_parts, kvh = h >> p.lg_group;
            const ResSpan s(p, v, total, (int)word_of(ent, kWindow));
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
            res_stored();   // this workgroup's words of the next layer are empty before it hands anything over
            RES_STAMP(28);
            if (!ALL) load_kv(ent, v);
            RES_STAMP(29);
            __syncthreads();
            RES_STAMP(6);
            if (ALL) load_head_w(ent_next);
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
                for (int u = 0; u < KS; u++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(aq[u], __builtin_bit_cast(rh16x8, kv.k[u]), acc, 0, 0, 0);
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
                    o[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ap, __builtin_bit_cast(rh16x8, kv.v[b]), o[b], 0, 0, 0);
                }
                if (more) {
                    load_v(rsrc_v(ent, false), kvh, t0 + kAttnPass);
                    __syncthreads();   // the next pass's scores must not overtake this pass's reads
                }
            };
            for (int t0 = s.begin; t0 < s.end; t0 += kAttnPass) pass(t0);
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
        if (!ALL) load_head_w(ent_next);
        // ---- o: the XCD's chunks joined (unnormalised), times the head's rows of o
        RES_SHARES(v) {
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
            if (ALL || v == first) wp = row4(ent, 1), wi = row4(ent, 2);
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
            __syncthreads();
            RES_STAMP(26);
            const int skip = (h * HD) % 128 / 4;            // a head of 64 channels is half of a k tile: the other half counts for nothing
            if (tid < KT3 * 32) {
                const int c = tid - skip;
                float4 sum = zero4;
                if (c >= 0 && c < HD / 4) {
#pragma unroll 1
                    for (int q0 = 0; q0 < NJ; q0 += 8) {
                        float2 lo[8], hi[8];
#pragma unroll
                        for (int q = 0; q < 8; q++) {
                            const float2 *t = reinterpret_cast<const float2 *>(S.join + (q0 + q) * HD + (c >> 1) * 8 + (c & 1) * 2);
                            lo[q] = t[0], hi[q] = t[2];
                        }
#pragma unroll
                        for (int q = 0; q < 8; q++) sum.x += lo[q].x, sum.y += lo[q].y, sum.z += hi[q].x, sum.w += hi[q].y;
                    }
                }
                put_digits(tid, sum.x, sum.y, sum.z, sum.w);
            }
            __syncthreads();
            RES_STAMP(10);
            const ResShare<HD> share(p, v, 1);
            if (wave / KT3 < share.tiles) multiply(One{}, std::true_type{}, 1, ent, share, wave / KT3, wave % KT3, KT3, wave % KT3);
            RES_STAMP(11);
            __syncthreads();
            if (wave >= 4) {
                const uint32_t r = (uint32_t)(v >> 3), x = (uint32_t)(v & 7), t = (uint32_t)wave - 4;
                if (wave == 4 && lane < 2) put(kResM1 + 32u * r + 2u * x + (uint32_t)lane, __float_as_uint(lane == 0 ? M : L), true);
                if ((int)t < share.tiles) {
                    const float s = tile_sum((int)t, KT3);
                    if (lane < 16) put(kResG1 + r * 512u + x * 64u + t * 16u + (uint32_t)lane, __float_as_uint(s), true);
                }
            }
            if (!ALL) __syncthreads();
        }
        RES_STAMP(12);
        if (wave == 6)
            RES_SHARES(v)
                if (tiles3(v) > 0) combine(v, kResG1, kResY, true);
        RES_STAMP(13);
        // ---- gate | up of the row, and the gated row
        if (holds) {
            const uint4 raw = take16(home + kResY + (uint32_t)tid * 4u);
            y4 = make_float4(__uint_as_float(raw.x), __uint_as_float(raw.y), __uint_as_float(raw.z), __uint_as_float(raw.w));
        }
        RES_STAMP(14);
        // What the norm needs is here: said in so many words, and what is asked for next kept together, or the norm's first
        // instructions would be among these loads and wait for them.
        res_stored();
        RES_TOGETHER();
        if (ALL) load_kv(ent_next, first);   // (behind the last layer: its own again)
        wp1 = row4(ent, 3), wi1 = row4(ent_next, 0);
        ent_after = entry_of(l + 2);
        RES_TOGETHER();
        RES_STAMP(25);
        norm_row(wp, wi);
        RES_STAMP(15);
        RES_SHARES(v) {
            const ResShare<HD> share(p, v, 2);
            const int parts = share.tiles == 4 ? 4 : 8, q = share.tiles == 4 ? wave >> 2 : 0;
            // (a pair's k tiles start one wavefront later than the other's: the SIMDs, which have two of the wavefronts each, get as many)
            if (share.tiles > 0 && share.has(p, 2 * q)) multiply(Two{}, std::false_type{}, 2, ent, share, 2 * q, (wave + q) & (parts - 1), parts, wave & (parts - 1));
            RES_STAMP(16);
            __syncthreads();
            if (wave >= 4 && 2 * (wave - 4) < share.tiles) {
                const int t = 2 * (wave - 4);
                const float gate = tile_sum(t, parts), up = tile_sum(t + 1, parts);
                const float g = res_pair(p, v, wave - 4) < p.pairs ? res_gelu(gate) * up : 0.f;   // columns past ffn: zeros
                if (lane < 16) put((uint32_t)(v & 7) * kResLocal + kResH + res_place((uint32_t)(((v >> 3) + 32 * (wave - 4)) * 16 + lane)), __float_as_uint(g), wide);
            }
            if (!ALL) __syncthreads();
        }
        RES_STAMP(17);
        // ---- down: the XCD's slice of the gated row times its rows of the weight
        RES_SHARES(v) {
            const int nk = slice_tiles(v);
            if (tid < nk * 32) {
                const uint4 w = take16((uint32_t)(v & 7) * kResLocal + kResH + (uint32_t)tid * 4u);
                put_digits(tid, __uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w));
            }
            RES_STAMP(18);
            RES_STAMP(24);
            __syncthreads();
            RES_STAMP(19);
            const ResShare<HD> share(p, v, 3);
            // (a k tile per wavefront, which takes all its tiles; one that has none leaves zeros)
            if (share.tiles == 1 || share.tiles == 2) multiply(Two{}, std::true_type{}, 3, ent, share, 0, wave, kResWaves, wave);
            else if (share.tiles == 3) multiply(Three{}, std::true_type{}, 3, ent, share, 0, wave, kResWaves, wave);
            else if (share.tiles == 4) multiply(Four{}, std::true_type{}, 3, ent, share, 0, wave, kResWaves, wave);
            RES_STAMP(20);
            __syncthreads();
            if (wave >= 4 && wave - 4 < share.tiles) {
                const uint32_t t = (uint32_t)wave - 4;
                const float s = tile_sum((int)t, kResWaves);
                if (lane < 16) put(kResG2 + (uint32_t)(v >> 3) * 512u + (uint32_t)(v & 7) * 64u + t * 16u + (uint32_t)lane, __float_as_uint(s), true);
            }
            if (!ALL) __syncthreads();
        }
        RES_STAMP(21);
        if (wave == 6)
            RES_SHARES(v)
                if (tiles3(v) > 0) combine(v, kResG2, kResY2, false);
        RES_STAMP(22);
        if (holds && (l + 1 < p.n_layers || first == 0)) {
            const uint4 raw = take16(home + kResY2 + (uint32_t)tid * 4u);
            y4 = make_float4(__uint_as_float(raw.x), __uint_as_float(raw.y), __uint_as_float(raw.z), __uint_as_float(raw.w));
        }
        RES_STAMP(23);
        res_stored();   // (the next norm's operands are here)
        RES_STAMPS_OUT();
        cur = next;
        next = next == (kResSets - 1) * kResWords * 4u ? 0u : next + kResWords * 4u;
        ent = ent_next, ent_next = ent_after;
    }
    if (first == 0 && holds) {
        float *x = p.x_out + place(), *y = p.y_out + place();
        *reinterpret_cast<float2 *>(x) = make_float2(x4.x, x4.y), *reinterpret_cast<float2 *>(x + 4) = make_float2(x4.z, x4.w);
        *reinterpret_cast<float2 *>(y) = make_float2(y4.x, y4.y), *reinterpret_cast<float2 *>(y + 4) = make_float2(y4.z, y4.w);
    }
}

// ALL: begins when all 256 workgroups have arrived, or not at all. Else: does the work of a launch of the other form that
// did not begin (`behind` is set), or that was never made, with the workgroups that have arrived by the deadline.
// (Two kernels: in one the second form costs the first 25 us a token, in registers. A launch that finds its work done is 4.6 us by kernel trace, the launch itself included.)
template <int HD, int SG, bool ALL>
__global__ void __launch_bounds__(kResThreads + (ALL ? 64 * kFeedWaves : 0)) RES_ONE_PER_CU(ALL) dec_resident_kernel(const ResidentArgs p) {
    __shared__ __attribute__((aligned(16))) ResShared<HD, SG, ALL> S;
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
    if constexpr (ALL) {
        if ((int)threadIdx.x >= kResThreads) {
            switch (__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) - kResWaves) {
                case 0: res_feed<HD, SG, 0>(p, S, first, pos + 1); break;
                case 1: res_feed<HD, SG, 1>(p, S, first, pos + 1); break;
                case 2: res_feed<HD, SG, 2>(p, S, first, pos + 1); break;
                default: res_feed<HD, SG, 3>(p, S, first, pos + 1); break;
            }
            return;
        }
    }
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
//   8/1 of 256, 2048 / 8192     273 / 243 at 8192, 299 / 293 at 12288, 316 / 335 at 16384
//   8/2 of 64, 512 / 2048       162 / 151 at 8192, 171 / 174 at 12288, 179 / 194 at 16384
//   8/4 of 256, 1152 / 6912     285 / 268 at 12288, 312 / 318 at 16384
//   8/8 of 128, 1024 / 4096     207 / 181 at 8192, 242 / 220 at 12288, 259 / 257 at 16384
//   4/1 of 256, 1152 / 6912     247 / 212 at 16384, 327 / 309 at 32768;  4/4 of 128, 512 / 2048  275 / 251 at 32768
//   2/1 of 128, 512 / 2048      353 / 229 at 65536;  1/1 of 256, 1152 / 6912  805 / 341 at 131072
// and at positions 100 and 2040 one launch takes two thirds to four fifths. The position is the device's and a recorded step covers all of
// them, so the rule is on the longest one: no position of a decoder that takes one launch is slower for it.
// Only where every workgroup has a CU: with fewer, all steps would be the stand-in's, whose workgroups take shares in turn (gemma3-1b
// at 2048: 846 us a token with 255 workgroups, 983 with 128, 1672 with 64; 654 by the launches per product, 444 in one launch).
bool hipc::resident_pays(hipc_ctx *ctx, const hipc_decoder_config &c) {
    const int64_t most = c.n_q_heads <= 4 ? 131072 / c.n_q_heads : c.n_kv_heads >= 4 ? 12288 : 8192;
    return ctx->cu_count >= (int)kResGroups && c.max_seq <= most;
}

namespace {

constexpr int whole_units(int units) { return (units + 3) / 4 * 4; }   // four units' scales are asked for together

template <int HD, bool ALL>
void launch_sg(hipc_ctx *ctx, int sg, const ResidentArgs &a, int workgroups) {
    switch (sg) {
        case 4: hipLaunchKernelGGL((dec_resident_kernel<HD, 4, ALL>), dim3(workgroups), dim3(kResThreads + (ALL ? 64 * kFeedWaves : 0)), 0, ctx->stream, a); break;
        case 2: hipLaunchKernelGGL((dec_resident_kernel<HD, 2, ALL>), dim3(workgroups), dim3(kResThreads + (ALL ? 64 * kFeedWaves : 0)), 0, ctx->stream, a); break;
        default: hipLaunchKernelGGL((dec_resident_kernel<HD, 1, ALL>), dim3(workgroups), dim3(kResThreads + (ALL ? 64 * kFeedWaves : 0)), 0, ctx->stream, a); break;
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
    a.inv_hidden = 1.f / (float)c.hidden;
    // Places in LDS for the units of the largest share of each product. q|k|v's are among gate|up's, those that are asked for when
    // the former are done with; the next layer's q|k|v are asked for behind gate|up.
    const int down_kts = (int)ceil_div(a.cg_f, kResXcds), h_tiles = (int)ceil_div(a.tiles_h, kResRanks);
    a.slot[1] = 0;
    a.slot[3] = whole_units(h_tiles * std::max(1, c.head_dim / 128));
    a.slot[2] = a.slot[3] + whole_units(h_tiles * down_kts);
    a.slot[0] = a.slot[2] + kFeedFirst;
    static_assert(whole_units(4 * 2) + whole_units(4 * 8) + std::max(whole_units(4 * 16), kFeedFirst + whole_units(2 * 16)) <= kResSlots, "the largest shapes resident_takes");
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
