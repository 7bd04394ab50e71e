// Address model of the decode step: the library's own sources (matmul_nbits.hip, gemv_lean.hip,
// decoder.hip, with prefetch.h and lanes.h) compiled as host code behind gpu_model.h, driven through
// the same entry points a caller uses. Every launch of a step runs thread by thread on the CPU; every
// buffer load is checked against the allocations the library itself made (hipc_decoder_create,
// nbits_prepack: their sizes, byte for byte), under the hardware's rule that the descriptor's range
// check sees the per-lane offset only; every ordinary load and store is checked by AddressSanitizer.
// The read-ahead helper rows are on (kReadAheadVerified is true in this build): what this program
// verifies is exactly what that constant stands for.
//
//   decoder_model full           whole steps at positions around every boundary of the chunking (0, 16, 32, 64, 512,
//                                2048, the windows, the end of the cache), windows 0 / 70 / 512 / 4200, every shape
//                                below: the shapes of the GPU tests and gemma3-1b's (two layers of it, whole vocabulary)
//   decoder_model sweep [threads] the launches whose addresses depend on the position (the q|k|v launch's helper rows,
//                                which read the cache ahead; the attention launch; the output projection's join) at
//                                EVERY position of the cache, the same windows and shapes
//   decoder_model quick [threads] what the test suite runs: the full steps on a shorter list of positions, and the
//                                sweep of gemma3-1b's shape at every position below 96, every 29th beyond and the
//                                last 40, windows 0 and 512
#include <cstdio>
#include <mutex>
#include <thread>
#include <vector>

#include "internal.h"
#include "resident.h"

// ---- what the three sources leave undefined ---------------------------------------------------
namespace hipc {
alignas(16) thread_local uint4 lean_smem[160 * 1024 / 16];   // the kernels' dynamic LDS (`extern __shared__`)
alignas(16) thread_local uint4 smem[160 * 1024 / 16];
thread_local float wgt[40960];
int scratch_get(hipc_ctx *ctx, int slot, size_t bytes, void **out) {
    Scratch &s = ctx->scratch[slot];
    if (s.bytes < bytes) {
        if (s.ptr) gpu_model::release(s.ptr);
        s.ptr = gpu_model::alloc(bytes);   // exactly what was asked for: stricter than the library's rounding
        s.bytes = bytes;
    }
    *out = s.ptr;
    return HIPC_OK;
}
bool nbits_prefill_takes(const void *, const hipc_nbits_weight *, int64_t) { return false; }
int nbits_rows_f32_split(hipc_ctx *, const void *, const hipc_nbits_weight *, void *, int, int) { return HIPC_ERR_UNSUPPORTED; }
int nbits_prefill(hipc_ctx *, const void *, const hipc_nbits_weight *, void *, int64_t) { return HIPC_ERR_UNSUPPORTED; }
bool nbits_prefill_f32_takes(const void *, const hipc_nbits_weight *, int64_t) { return false; }
bool nbits_prefill_f32_fits(hipc_ctx *, const hipc_nbits_weight *, int64_t, int) { return false; }
size_t nbits_split_bytes(int64_t, int64_t, int64_t) { return 0; }
int nbits_prefill_f32(hipc_ctx *, const void *, const hipc_nbits_weight *, void *, int64_t, int) { return HIPC_ERR_UNSUPPORTED; }
}  // namespace hipc
extern "C" {
const char *hipGetErrorString(hipError_t) { return "model"; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamGetCaptureInfo_v2(hipStream_t, hipStreamCaptureStatus *status, unsigned long long *, hipGraph_t *, const hipGraphNode_t **, size_t *n) {
    *status = hipStreamCaptureStatusNone, *n = 0;
    return hipSuccess;
}
}

#define MUST(call)                                                                    \
    do {                                                                              \
        const int rc_ = (call);                                                       \
        if (rc_ != HIPC_OK) {                                                         \
            std::printf("FAILED %s:%d: %s -> %d (%s)\n", __FILE__, __LINE__, #call, rc_, ctx.err.c_str()); \
            std::exit(1);                                                             \
        }                                                                             \
    } while (0)

namespace {

struct Shape {
    const char *name;
    int layers, hidden, ffn, nq, nkv, hd, vocab, max_seq;
};

// which launches of a step run, and which rows of their grids (set per run; read by gpu_model_launch)
struct Select {
    bool on = false;
    int index = 0;                       // launches seen since the step began
    std::function<bool(int, unsigned *, unsigned *)> rows;   // launch index -> run? and its blockIdx.y range
};
thread_local Select g_select;

struct Model {
    hipc_ctx ctx;
    hipc_decoder *dec = nullptr;
    hipc_decoder_config cfg{};
    std::vector<void *> inputs;

    void *input(size_t bytes) {
        void *p = gpu_model::alloc(bytes);
        inputs.push_back(p);
        return p;
    }
    void build(const Shape &s) {
        ctx.tune.dec_prefetch = 31;   // the helper rows are what is being verified
        cfg.n_layers = s.layers, cfg.hidden = s.hidden, cfg.ffn = s.ffn, cfg.n_q_heads = s.nq, cfg.n_kv_heads = s.nkv;
        cfg.head_dim = s.hd, cfg.vocab = s.vocab, cfg.max_seq = s.max_seq, cfg.block_size = 32;
        cfg.rms_eps = 1e-6f, cfg.rope_theta = 10000.f, cfg.attn_scale = 0.f, cfg.embed_scale = 1.f;
        MUST(hipc_decoder_create(&ctx, &cfg, &dec));
        const int64_t qd = (int64_t)s.nq * s.hd, kvd = (int64_t)s.nkv * s.hd;
        auto linear = [&](int layer, int which, int64_t K, int64_t N) {
            const int64_t nb = (K + 31) / 32;
            const size_t b_len = (size_t)N * nb * 16, s_len = (size_t)N * nb, z_len = (size_t)N * ((nb + 1) / 2);
            void *B = input(b_len), *S = input(s_len * 4), *Z = input(z_len);
            MUST(hipc_decoder_set_linear(&ctx, dec, layer, which, B, b_len, S, s_len, Z, z_len));
        };
        for (int li = 0; li < s.layers; li++) {
            linear(li, HIPC_DEC_QKV, s.hidden, qd + 2 * kvd);
            linear(li, HIPC_DEC_O, qd, s.hidden);
            linear(li, HIPC_DEC_GATE_UP, s.hidden, 2 * (int64_t)s.ffn);
            linear(li, HIPC_DEC_DOWN, s.ffn, s.hidden);
            for (int n = 0; n < 6; n++) {
                void *w = input((size_t)std::max(s.hidden, s.hd) * 4);
                MUST(hipc_decoder_set_norm(&ctx, dec, li, n, w));
            }
        }
        linear(0, HIPC_DEC_LM_HEAD, s.hidden, s.vocab);
        MUST(hipc_decoder_set_norm(&ctx, dec, 0, HIPC_DEC_NORM_FINAL, input((size_t)s.hidden * 4)));
        const int64_t nb = (s.hidden + 31) / 32;
        const size_t qb = (size_t)s.vocab * nb * 16, sb = (size_t)s.vocab * nb, zb = (size_t)s.vocab * ((nb + 1) / 2);
        MUST(hipc_decoder_set_embedding(&ctx, dec, input(qb), qb, input(sb * 4), sb, input(zb), zb));
    }
    void step_at(int pos, int token) {
        g_select.index = 0;
        const bool was = g_select.on;
        g_select.on = false;
        MUST(hipc_decoder_reset(&ctx, dec, token, pos));
        g_select.on = was;
        g_select.index = 0;
        MUST(hipc_decoder_step(&ctx, dec));
    }
    void windows(int w) {
        for (int li = 0; li < cfg.n_layers; li++) MUST(hipc_decoder_set_layer_attention(&ctx, dec, li, li == 0 ? w : 0, li == 0 && w ? 1.0e6f : 0.f));
    }
    void destroy() {
        hipc_decoder_destroy(&ctx, dec);
        for (void *p : ctx.deferred) gpu_model::release(p);
        ctx.deferred.clear();
        for (void *p : ctx.deferred_host) gpu_model::release(p);
        ctx.deferred_host.clear();
        for (void *p : inputs) gpu_model::release(p);
        inputs.clear();
        for (hipc::Scratch &s : ctx.scratch)
            if (s.ptr) gpu_model::release(s.ptr), s.ptr = nullptr, s.bytes = 0;
    }
};

const Shape kGemma = {"gemma3-1b (two layers)", 2, 1152, 6912, 4, 1, 256, 262144, 2112};
const Shape kSmall[] = {
    {"small hd 64, 4 q / 2 kv", 2, 128, 256, 4, 2, 64, 512, 80},
    {"small hd 256, 4 q / 1 kv", 2, 128, 256, 4, 1, 256, 512, 2054},
    {"small hd 128, 8 q / 1 kv", 2, 128, 256, 8, 1, 128, 512, 4298},
    {"small hd 64, 2 q / 2 kv", 2, 128, 256, 2, 2, 64, 512, 2308},
    {"small hd 128, 4 q / 2 kv", 2, 128, 256, 4, 2, 128, 512, 517},
    {"small hd 192 (three-kernel attention)", 2, 128, 256, 2, 1, 192, 512, 108},
};

// counters of all host threads (a thread adds its registry's when it is done)
std::mutex g_totals_mu;
size_t g_launches = 0, g_threads = 0, g_loads = 0, g_clipped = 0;
void add_totals() {
    gpu_model::Registry &g = gpu_model::reg();
    std::lock_guard<std::mutex> lock(g_totals_mu);
    g_launches += g.launches, g_threads += g.threads, g_loads += g.loads, g_clipped += g.loads_clipped;
    g.launches = g.threads = g.loads = g.loads_clipped = 0;
}
void report(const char *what) {
    add_totals();
    std::printf("%-44s %7zu launches %11zu threads %11zu buffer loads (%zu answered with zeros)\n", what, g_launches, g_threads, g_loads, g_clipped);
    std::fflush(stdout);
    g_launches = g_threads = g_loads = g_clipped = 0;
}

// The words a step's workgroups agree through must be as new for the next step, whatever they held: a decision that is left
// standing would be taken for the next launch's own.
void step_words() {
    const Shape s = kSmall[0];
    Model m;
    gpu_model::reg().where = "the words of a step";
    m.build(s);
    m.ctx.tune.dec_prefetch = -1;
    uint32_t *sync = nullptr;
    for (const auto &[at, bytes] : gpu_model::reg().blocks)
        if (bytes == hipc::kResSync * sizeof(uint32_t)) sync = reinterpret_cast<uint32_t *>(at);
    using namespace hipc;
    const auto expect = [&](bool ok, const char *what, uint32_t step) {
        if (ok) return;
        std::printf("FAILED: step %u: %s\n", step, what);
        std::exit(1);
    };
    expect(sync != nullptr, "no words found", 0);
    expect(sync[0] == 1, "a new decoder's first step is not number 1", 0);
    hipc_ctx &ctx = m.ctx;
    MUST(hipc_decoder_reset(&ctx, m.dec, 1, 0));
    // (2^22: what a decision once held of the number was all zeros there, as the words are when nothing has been decided)
    for (uint32_t step : {1u, 2u, (1u << 22) - 1, 1u << 22, (1u << 22) + 1, 3u << 22, kResLaunches - 2, kResLaunches - 1}) {
        sync[0] = step;
        sync[kResAll + kResDecision] = res_decision(kResGroups, true), sync[kResSome + kResDecision] = res_decision(3, false);
        MUST(hipc_decoder_step(&ctx, m.dec));
        expect(sync[kResAll + kResDecision] == 0 && sync[kResSome + kResDecision] == 0, "its decisions stand", step);
        expect(sync[0] != 0, "followed by number 0, which the flags begin with", step);
        expect(sync[0] % kResSets == (step + 1) % kResSets, "the sets are not taken in turn", step);
    }
    m.destroy();
    report("the words of a step");
}

// A read brings state, history and logits with pinned host memory and without; the decoder takes none before it, and for logits
// only where they are wanted.
void reads() {
    const Shape s = kSmall[0];
    Model m;
    gpu_model::reg().where = "reads";
    gpu_model::reg().no_pinned = true;
    m.ctx.tune.dec_resident = 0;   // (in the one launch threads wait for each other, which here run in turn)
    m.build(s);
    hipc_ctx &ctx = m.ctx;
    ctx.tune.dec_prefetch = -1;
    const size_t blocks = gpu_model::reg().blocks.size();
    const auto expect = [&](bool ok, const char *what) {
        if (!ok) std::printf("FAILED: a read: %s\n", what), std::exit(1);
    };
    std::vector<float> logits[2];
    std::vector<int32_t> history[2];
    MUST(hipc_decoder_reset(&ctx, m.dec, 1, 5));
    MUST(hipc_decoder_step(&ctx, m.dec));
    for (int pinned = 0; pinned < 2; pinned++) {
        gpu_model::reg().no_pinned = !pinned;
        int32_t token = -1, pos = -1;
        logits[pinned].assign(s.vocab, -1.f), history[pinned].assign(s.max_seq + 3, -7);
        MUST(hipc_decoder_read(&ctx, m.dec, &token, &pos, nullptr, nullptr, 0));
        expect(pos == 6 && token >= 0 && token < s.vocab, "token and position");
        expect(gpu_model::reg().blocks.size() == blocks + pinned, "memory for logits nobody wanted");
        MUST(hipc_decoder_read(&ctx, m.dec, &token, &pos, logits[pinned].data(), history[pinned].data(), s.max_seq + 3));
        expect(gpu_model::reg().blocks.size() == blocks + 2 * pinned, "memory for logits");
        expect(history[pinned][s.max_seq] == -7, "a history longer than there is");
    }
    expect(std::memcmp(logits[0].data(), logits[1].data(), s.vocab * 4) == 0 && history[0] == history[1], "not the same without pinned memory");
    m.destroy();
    report("reads");
}

// Replacing what a layer is made of while graphs live: a new layer table only where a recorded step reads the old one, and
// that one goes when the graphs do.
void table_changes() {
    const Shape s = kSmall[0];
    Model m;
    gpu_model::reg().where = "changes beside graphs";
    m.build(s);
    hipc_ctx &ctx = m.ctx;
    ctx.tune.dec_prefetch = -1;
    const auto change = [&](int times) {
        for (int i = 0; i < times; i++) MUST(hipc_decoder_set_layer_attention(&ctx, m.dec, i % s.layers, 10 + i % 7, 0.f));
    };
    const auto expect = [&](size_t blocks, size_t retained, const char *what) {
        if (gpu_model::reg().blocks.size() == blocks && ctx.retained.size() == retained) return;
        std::printf("FAILED: %s: %zu allocations for %zu, %zu retired for %zu\n", what, gpu_model::reg().blocks.size(), blocks, ctx.retained.size(), retained);
        std::exit(1);
    };
    const auto record = [&] {
        ctx.capturing = true;
        MUST(hipc_decoder_step(&ctx, m.dec));
        ctx.capturing = false, ctx.live_graphs++;
    };
    MUST(hipc_decoder_reset(&ctx, m.dec, 1, 0));
    const size_t before = gpu_model::reg().blocks.size();
    ctx.live_graphs = 1;   // somebody else's
    change(50);
    expect(before, 0, "no recorded step of this decoder");
    record();
    change(50);
    expect(before + 1, 1, "one recorded step");
    record(), record();
    change(50);
    expect(before + 2, 2, "recorded again");
    record();
    // a change for which there was no memory is made up for by the next step: it must not run on what was replaced
    gpu_model::reg().no_memory = true;
    if (hipc_decoder_set_layer_attention(&ctx, m.dec, 0, 77, 0.f) == HIPC_OK || hipc_decoder_step(&ctx, m.dec) == HIPC_OK) {
        std::printf("FAILED: a change without memory, or a step behind it, went through\n");
        std::exit(1);
    }
    gpu_model::reg().no_memory = false;
    MUST(hipc_decoder_step(&ctx, m.dec));
    expect(before + 3, 3, "made up for");
    bool found = false;
    for (const auto &[at, bytes] : gpu_model::reg().blocks)
        found = found || (bytes == s.layers * sizeof(hipc::ResidentLayer) && reinterpret_cast<const hipc::ResidentLayer *>(at)->window == 77);
    if (!found) std::printf("FAILED: the change did not reach the table\n"), std::exit(1);
    ctx.live_graphs = 0;   // all of them destroyed
    for (void *p : ctx.retained) gpu_model::release(p);
    ctx.retained.clear();
    change(50);
    expect(before, 0, "no graph left");
    m.destroy();
    report("changes beside graphs");
}

// Where a decoder takes all layers in one launch by itself: a device with a CU for each workgroup, and contexts up to the
// length where the launches per product, which spread a head over more workgroups, are the faster form.
void which_form() {
    struct Case {
        int cus, nq, nkv, max_seq;
        bool one_launch;
    };
    const Case cases[] = {{256, 4, 2, 80, true}, {255, 4, 2, 80, false}, {64, 4, 2, 80, false}, {304, 4, 2, 80, true},
                          {256, 4, 1, 32768, true}, {256, 4, 1, 32769, false}, {256, 1, 1, 131072, true},
                          {256, 8, 1, 8192, true}, {256, 8, 1, 8193, false}, {256, 8, 2, 8193, false}, {256, 8, 4, 12288, true}, {256, 8, 8, 12289, false}};
    for (const Case &k : cases) {
        hipc_ctx ctx;
        ctx.cu_count = k.cus;
        hipc_decoder_config cfg{};
        cfg.n_layers = 1, cfg.hidden = 128, cfg.ffn = 256, cfg.n_q_heads = k.nq, cfg.n_kv_heads = k.nkv, cfg.head_dim = 64;
        cfg.vocab = 512, cfg.max_seq = k.max_seq, cfg.block_size = 32, cfg.rms_eps = 1e-6f, cfg.rope_theta = 10000.f, cfg.embed_scale = 1.f;
        hipc_decoder *dec = nullptr;
        MUST(hipc_decoder_create(&ctx, &cfg, &dec));
        bool found = false;
        for (const auto &[at, bytes] : gpu_model::reg().blocks) found = found || bytes == hipc::kResSync * sizeof(uint32_t);
        if (found != k.one_launch) {
            std::printf("FAILED: %d CUs, %d / %d heads, %d positions: %s\n", k.cus, k.nq, k.nkv, k.max_seq, found ? "one launch" : "a launch per product");
            std::exit(1);
        }
        hipc_decoder_destroy(&ctx, dec);
        for (void *p : ctx.deferred) gpu_model::release(p);
        for (void *p : ctx.deferred_host) gpu_model::release(p);
    }
    report("which form a decoder takes");
}

bool g_quick = false;
std::vector<int> windows_of(const Shape &s) {
    if (g_quick) return {0, 512};
    std::vector<int> w = {0, 70, 512, 4200};
    w.erase(std::remove_if(w.begin(), w.end(), [&](int v) { return v >= s.max_seq; }), w.end());
    return w;
}

void full(const Shape &s) {
    Model m;
    gpu_model::reg().where = s.name;
    m.build(s);
    const int last = s.max_seq - 1;
    const std::vector<int> all = {0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 69, 70, 71, 511, 512, 513, 527, 528, 1023, 2039, 2040, 2047, 2048, 2049, 4199, 4200, 4201, last - 1, last};
    const std::vector<int> few = {0, 1, 31, 32, 33, 512, 513, 2048, last};
    for (int w : windows_of(s)) {
        m.windows(w);
        for (int pos : g_quick ? few : all)
            if (pos >= 0 && pos <= last) m.step_at(pos, (pos * 7 + 3) % s.vocab);
    }
    // all layers in one launch, where the shape has that: the whole grid, and a smaller one whose workgroups take several shares
    if (s.hd != 192) {
        m.ctx.tune.dec_prefetch = -1;
        for (int w : windows_of(s)) {
            m.windows(w);
            for (int pos : {0, 31, 32, 33, 513, 2048, last})
                if (pos >= 0 && pos <= last) {
                    m.ctx.tune.dec_resident = pos == 33 ? 100 : -1;
                    m.step_at(pos, 1);
                    if (g_quick && s.layers * s.hidden > 1000) break;
                }
        }
        m.ctx.tune.dec_prefetch = 31, m.ctx.tune.dec_resident = -1;
    }
    // a step with the cache full changes nothing and reads nothing out of range
    m.step_at(last, s.vocab - 1);
    {
        hipc_ctx &ctx = m.ctx;
        MUST(hipc_decoder_step(&ctx, m.dec));
        int32_t token = 0, pos = 0;
        const int rc = hipc_decoder_read(&ctx, m.dec, &token, &pos, nullptr, nullptr, 0);
        if (rc == HIPC_OK || pos != s.max_seq) {
            std::printf("FAILED: a step past the end of the cache was not reported (rc %d, position %d)\n", rc, pos);
            std::exit(1);
        }
    }
    m.destroy();
    report(s.name);
}

// The launches whose addresses depend on the position, at every position. In the lean path a layer's
// launches are, from index 1 + 5 layer on: q|k|v (its helper rows read the cache ahead: rows >= 1),
// attention (rows < kv heads: its own; the helper rows behind them read the next launch's weights and
// do not depend on the position), output projection (rows < 8 cover its k slices), gate|up, down.
void sweep(const Shape &s, int threads) {
    // the output projection's own rows: its k slices, as hipc_decoder_create cuts them (one head per slice, at most 8)
    const int n_cg_o = (s.nq * s.hd + 127) / 128;
    int o_tiles = std::max(1, s.hd / 128);
    while ((n_cg_o + o_tiles - 1) / o_tiles > 4 && o_tiles < 4) o_tiles *= 2;
    const unsigned o_slices = (unsigned)((n_cg_o + o_tiles - 1) / o_tiles);
    for (int w : windows_of(s)) {
        std::vector<std::thread> pool;
        for (int t = 0; t < threads; t++) {
            pool.emplace_back([&, t] {
                gpu_model::reg().where = s.name;
                Model m;
                m.build(s);
                m.windows(w);
                g_select.on = true;
                g_select.rows = [&](int index, unsigned *y0, unsigned *y1) {
                    if (index == 1) { *y0 = 1, *y1 = ~0u; return true; }
                    if (index == 2) { *y0 = 0, *y1 = (unsigned)s.nkv; return true; }
                    if (index == 3) { *y0 = 0, *y1 = o_slices; return true; }
                    return false;
                };
                for (int pos = t; pos < s.max_seq; pos += threads)
                    if (!g_quick || pos < 96 || pos % 29 == 0 || pos >= s.max_seq - 40) m.step_at(pos, 1);
                g_select.on = false;
                m.destroy();
                add_totals();
            });
        }
        for (std::thread &th : pool) th.join();
    }
    report(s.name);
}

}  // namespace

int main(int argc, char **argv) {
    const std::string mode = argc > 1 ? argv[1] : "full";
    const int threads = argc > 2 ? std::atoi(argv[2]) : 1;
    gpu_model_select = [](const char *, dim3, unsigned *y0, unsigned *y1) {
        if (!g_select.on) return true;
        return g_select.rows(g_select.index++, y0, y1);
    };
    if (mode != "sweep") step_words(), reads(), table_changes(), which_form();
    if (mode == "full") {
        for (const Shape &s : kSmall) full(s);
        full(kGemma);
    } else if (mode == "quick") {
        g_quick = true;
        for (const Shape &s : kSmall) full(s);
        Shape g = kGemma;
        full(g);
        g.vocab = 4096;   // the unembedding is not part of the swept launches
        sweep(g, threads);
    } else if (mode == "sweep") {
        for (const Shape &s : kSmall)
            if (s.hd != 192) sweep(s, threads);   // (no one-launch attention for that head_dim: nothing of it depends on the position this way)
        Shape g = kGemma;
        g.vocab = 4096;   // the unembedding is not part of the swept launches
        sweep(g, threads);
    } else {
        std::printf("usage: decoder_model full | sweep [threads] | quick [threads]\n");
        return 2;
    }
    std::printf("ok\n");
    return 0;
}
