// The resident decode kernel (decode_resident.hip): what the decoder hands it.
#pragma once

#include <hip/hip_fp16.h>

#include "internal.h"

namespace hipc {

// One layer as the kernel reads it from device memory (set_linear, set_norm, ... write the entries in stream order).
struct ResidentLayer {
    const uint4 *wq[4];       // q|k|v, o, gate|up (interleaved halves), down
    const float *sc[4];
    const uint8_t *zb[4];
    const float *norm[6];     // input, post_attn, pre_ffn, post_ffn, q, k
    __half *k_cache, *v_cache;
    int window, rope_table;
};

// The words workgroups exchange: three sets, taken in turn by the layers. A region that stays inside an XCD is repeated for each.
constexpr uint32_t kResXcds = 8, kResRanks = 32, kResGroups = kResXcds * kResRanks;
constexpr uint32_t kResMaxHidden = 2048, kResMaxHead = 256, kResMaxSlice = 1024;
constexpr uint32_t kResA = 0;                                          // [rank][head]: unnormalised attention outputs
constexpr uint32_t kResML = kResA + kResRanks * kResMaxHead;           // [rank](max, sum)
constexpr uint32_t kResY = kResML + 2 * kResRanks;                     // the attention branch's row
constexpr uint32_t kResH = kResY + kResMaxHidden;                      // the XCD's slice of the gated row, two bf16 terms a word
constexpr uint32_t kResY2 = kResH + kResMaxSlice;                      // the feed-forward branch's row
constexpr uint32_t kResLocal = kResY2 + kResMaxHidden;                 // words of one XCD
constexpr uint32_t kResG1 = kResXcds * kResLocal;                      // [rank][XCD][64 columns]: o's partial rows
constexpr uint32_t kResM1 = kResG1 + kResRanks * kResXcds * 64;        // [rank][32]: (max, sum) per XCD
constexpr uint32_t kResG2 = kResM1 + kResRanks * 32;                   // [rank][XCD][64 columns]: down's partial rows
constexpr uint32_t kResQ = kResG2 + kResRanks * kResXcds * 64;         // the q|k|v row
constexpr uint32_t kResMaxQkv = 2 * kResGroups * 16;
constexpr uint32_t kResWords = kResQ + kResMaxQkv;                         // words of one set
constexpr uint32_t kResSets = 3;
static_assert(kResA % 32 == 0 && kResML % 32 == 0 && kResY % 32 == 0 && kResH % 32 == 0 && kResY2 % 32 == 0 && kResLocal % 32 == 0,
              "no region shares a 128-byte line with another");
// The words the workgroups of a launch agree through: [0] the step's number, then, for the launch of all workgroups and for
// the one that stands in for it, the decision (0: none yet), one flag and one rank per workgroup. The token pick closes the
// step: it counts the number up and takes both decisions back, so no launch finds one that is not its own, however long ago
// that form last ran. (A flag carries the step's number and needs no clearing; no step has the number 0 that flags begin with.)
constexpr uint32_t kResDecision = 0, kResFlags = 32, kResRankOf = kResFlags + kResGroups, kResSyncWords = kResRankOf + kResGroups;
constexpr uint32_t kResAll = 32, kResSome = kResAll + kResSyncWords, kResSync = kResSome + kResSyncWords;
constexpr uint32_t kResLaunches = kResSets << 26;   // behind the largest number: a multiple of the sets, so that they go on in turn, and 28 bits
constexpr uint32_t kResDecided = 0x80000000u;       // a decision: this, the workgroups that take part, and (bit 0) whether each group of them shares an L2

__host__ __device__ inline uint32_t res_decision(uint32_t workgroups, bool one_l2) { return kResDecided | (workgroups << 1) | (one_l2 ? 1u : 0u); }
__host__ __device__ inline uint32_t res_decided_for(uint32_t decision) { return (decision & ~kResDecided) >> 1; }
// behind a step: the next one's words
__host__ __device__ inline void res_next_step(uint32_t *sync) {
    sync[0] = sync[0] + 1 == kResLaunches ? kResSets : sync[0] + 1;
    sync[kResAll + kResDecision] = sync[kResSome + kResDecision] = 0;
}

struct ResidentArgs {
    const ResidentLayer *table;
    const int *pos;
    int *broken;                 // set when a wait ran out
    const float *x_in, *rope;
    float *x_out, *y_out;        // the stream before the last branch is added, and that branch's row
    uint32_t *xch, *sync;
    int n_layers, hidden, cg_h, cg_o, tiles_h, tiles_qkv, cg_f, pairs;   // cg_*: 128-k tiles of hidden, the heads' channels, ffn; tiles_*: 16-column tiles; pairs: (gate, up) tile pairs
    int n_q, n_kv, lg_group, lg_parts;   // XCDs per head = 1 << lg_parts
    int max_seq, v_stride, behind;
    uint32_t inv_cg_h;                   // 65536 / cg_h, rounded up
    uint32_t nib_mask, magic;
    float eps, scale, inv_hidden;
};

bool resident_takes(const hipc_decoder_config &c);
bool resident_pays(const hipc_decoder_config &c);   // against the launch per product
int resident_launch(hipc_ctx *ctx, const hipc_decoder_config &c, const ResidentArgs &a, int workgroups);
int resident_set_layer(hipc_ctx *ctx, ResidentLayer *entry, const ResidentLayer &value);   // in stream order
int resident_clear(hipc_ctx *ctx, uint32_t *xch, uint32_t *sync);                          // exchange words empty, launch number 1

}  // namespace hipc
