// The resident decode kernel (decode_resident.hip): what the decoder hands it.
#pragma once

#include <hip/hip_fp16.h>

#include "internal.h"
#include "resident_door.h"

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
constexpr uint32_t kResMaxHidden = 2048, kResMaxHead = 256, kResMaxSlice = 1024;
constexpr uint32_t kResA = 0;                                          // [rank][head]: unnormalised attention outputs
constexpr uint32_t kResML = kResA + kResRanks * kResMaxHead;           // [rank](max, sum)
constexpr uint32_t kResY = kResML + 2 * kResRanks;                     // the attention branch's row
constexpr uint32_t kResH = kResY + kResMaxHidden;                      // the XCD's slice of the gated row
constexpr uint32_t kResY2 = kResH + kResMaxSlice;                      // the feed-forward branch's row
constexpr uint32_t kResLocal = kResY2 + kResMaxHidden;                 // words of one XCD
constexpr uint32_t kResG1 = kResXcds * kResLocal;                      // [rank][XCD][64 columns]: o's partial rows
constexpr uint32_t kResM1 = kResG1 + kResRanks * kResXcds * 64;        // [rank][32]: (max, sum) per XCD
constexpr uint32_t kResG2 = kResM1 + kResRanks * 32;                   // [rank][XCD][64 columns]: down's partial rows
constexpr uint32_t kResQ = kResG2 + kResRanks * kResXcds * 64;         // the q|k|v row
constexpr uint32_t kResMaxQkv = 2 * kResGroups * 16;
constexpr uint32_t kResWords = kResQ + kResMaxQkv;                         // words of one set
static_assert(kResA % 32 == 0 && kResML % 32 == 0 && kResY % 32 == 0 && kResH % 32 == 0 && kResY2 % 32 == 0 && kResLocal % 32 == 0,
              "no region shares a 128-byte line with another");

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
    int arrive, polls, wide;             // how long workgroups are waited for, in 10 ns; polls of a thread; stores at agent scope whatever the launch finds
    int slot[4];                         // where the units of product i begin in LDS
    float eps, scale, inv_hidden;
};

// What a reset puts in order behind a step that did not come to its end.
struct ResidentReset {
    uint32_t *xch, *sync;
    const ResidentLayer *table;
    int n_layers, v_rows, v_stride;   // v_rows: channels of all kv heads
};

bool resident_takes(const hipc_decoder_config &c);
bool resident_pays(hipc_ctx *ctx, const hipc_decoder_config &c);   // against the launch per product
int resident_launch(hipc_ctx *ctx, const hipc_decoder_config &c, const ResidentArgs &a, int workgroups);
int resident_set_layer(hipc_ctx *ctx, ResidentLayer *entry, const ResidentLayer &value);   // in stream order
int resident_clear(hipc_ctx *ctx, uint32_t *xch, uint32_t *sync);                          // exchange words empty, launch number 1

}  // namespace hipc
