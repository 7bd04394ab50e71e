// ConvInteger and QLinearConv (static int8, NCHW) for gfx950.
//
// Reference: crates/onnx-vulkan-core/src/interp.rs:3361-3536 (geometry), :4421-4651
// (conv_integer_with routing), :4796-4837 (qlinear_conv), :5680-5748 (HWC weight and
// activation layout); kernels shaders/conv_integer.rs; definition
// tests/conv_integer_im2col.rs:58-89.
//
// The reference materialises an im2col matrix [P, K] and runs its matmul on it
// (interp.rs:5319-5469). Here nothing of size P*K exists: the activation is
// turned once into NHWC (1x its own size, uint8 shifted to signed on the way),
// and the int8 MFMA contraction gathers its k-contiguous 16-byte operand chunks
// straight from it, with K ordered (kh, kw, c) and the weight prepacked to
// match. Padding taps read the zero point, so they contribute nothing and the
// zero-point algebra of the plain matmul applies unchanged
// (shaders/conv_integer.rs:112-119, 350-371).
// That is the general route. What most convolutions take skips even that copy: each workgroup reads the input positions its
// 64 or 128 outputs see straight from NCHW, transposes them in registers and keeps them in LDS for the whole product --
// int8_conv_slab_kernel (int8_conv_slab.h), and for few tiles along one axis int8_conv_row_kernel.
// Depthwise convolutions have a kernel of their own (conv_depth_kernel). Other grouped ones, and what fits neither (channel counts off 16 whose slab exceeds LDS), take a direct kernel, one
// output per thread.
#include <algorithm>
#include <type_traits>

#include "int8_conv_slab.h"

namespace hipc {

// X [C, HW] bytes -> Xt [HW, C] bytes (per image), xor `flip` on the way. 32x32 tiles.
__global__ void __launch_bounds__(256)
nchw_to_nhwc_kernel(const uint8_t *__restrict__ X, uint8_t *__restrict__ Xt, int C, int HW, uint8_t flip) {
    __shared__ uint8_t tile[32][33];
    const size_t img = (size_t)blockIdx.z * C * HW;
    const int hw0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
#pragma unroll
    for (int r = ty; r < 32; r += 8) {
        const int c = c0 + r, hw = hw0 + tx;
        tile[r][tx] = (c < C && hw < HW) ? X[img + (size_t)c * HW + hw] ^ flip : 0;
    }
    __syncthreads();
#pragma unroll
    for (int r = ty; r < 32; r += 8) {
        const int hw = hw0 + r, c = c0 + tx;
        if (c < C && hw < HW) Xt[img + (size_t)hw * C + c] = tile[tx][r];
    }
}

// The same for C and HW multiples of 4 with 4-byte aligned images, 32 bits at a time: a thread reads
// four positions of four channels (16 lanes x 4 bytes are one 64-byte run of a channel), transposes
// the 4 x 4 bytes in registers, and the words change hands through LDS so that the stores run along
// the channels (16 lanes x 4 bytes of one position). 64 channels x 64 positions per workgroup.
__global__ void __launch_bounds__(256)
nchw_to_nhwc4_kernel(const uint8_t *__restrict__ X, uint8_t *__restrict__ Xt, int C, int HW, uint32_t flip4) {
    __shared__ uint32_t words[64][17];  // [position][channel quad], padded
    const size_t img = (size_t)blockIdx.z * C * HW;
    const int hw0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
    const int hq = threadIdx.x & 15, cq = threadIdx.x >> 4;  // position quad, channel quad
    uint32_t in[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int c = c0 + 4 * cq + i, hw = hw0 + 4 * hq;
        in[i] = (c < C && hw < HW) ? *reinterpret_cast<const uint32_t *>(X + img + (size_t)c * HW + hw) ^ flip4 : 0u;
    }
    // out[j] = bytes j of in[0..3]: the four channels of position 4 hq + j
    const uint32_t lo01 = __builtin_amdgcn_perm(in[1], in[0], 0x05010400u);  // a0 b0 a1 b1
    const uint32_t hi01 = __builtin_amdgcn_perm(in[1], in[0], 0x07030602u);  // a2 b2 a3 b3
    const uint32_t lo23 = __builtin_amdgcn_perm(in[3], in[2], 0x05010400u);  // c0 d0 c1 d1
    const uint32_t hi23 = __builtin_amdgcn_perm(in[3], in[2], 0x07030602u);  // c2 d2 c3 d3
    words[4 * hq + 0][cq] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);  // a0 b0 c0 d0
    words[4 * hq + 1][cq] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);  // a1 b1 c1 d1
    words[4 * hq + 2][cq] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
    words[4 * hq + 3][cq] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
    __syncthreads();
    const int oq = threadIdx.x & 15, op = threadIdx.x >> 4;  // channel quad, position (of 16 per pass)
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int pos = op + 16 * r, hw = hw0 + pos, c = c0 + 4 * oq;
        if (c < C && hw < HW) *reinterpret_cast<uint32_t *>(Xt + img + (size_t)hw * C + c) = words[pos][oq];
    }
}

// W [O, C, kh, kw] -> Wp, O_pad x K_pad bytes in the fragment-major order of qfrag_offset,
// k = (r*kw + s)*C + c, signed domain, zero padded;
// rowsum[o] = sum_k Wp[o][k].
__global__ void __launch_bounds__(256)
pack_conv_w_kernel(const uint8_t *__restrict__ W, uint8_t *__restrict__ Wp, int32_t *__restrict__ rowsum, int O, int C,
                   int kh, int kw, int O_pad, int K_pad, int is_signed, int shift) {
    const int o = blockIdx.x;
    const int K = C * kh * kw;
    int local = 0;
    for (int k = threadIdx.x; k < K_pad; k += 256) {
        uint8_t out = 0;
        if (o < O && k < K) {
            const int tap = k / C, c = k - tap * C;
            const uint8_t v = W[((size_t)o * C + c) * kh * kw + tap];
            const int sv = (is_signed ? (int)(int8_t)v : (int)v) - shift;
            local += sv;
            out = (uint8_t)sv;
        }
        Wp[qfrag_offset(o, k, K_pad)] = out;
    }
    __shared__ int part[256];
    part[threadIdx.x] = local;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) rowsum[o] = part[0];
}

// W [O, C, kh, kw] -> fragment-major bytes in the step order of int8_conv_slab_kernel: a step is 32 k of one tap, or, with a
// single 16-channel chunk (kw2: pairs of taps per filter row), 16 channels of two taps. Zeros where there is no channel or tap.
__global__ void __launch_bounds__(256)
pack_conv_slab_kernel(const uint8_t *__restrict__ W, uint8_t *__restrict__ Ws, int32_t *__restrict__ rowsum, int O, int C,
                      int kh, int kw, int kw2, int npair, int steps, int is_signed, int shift) {
    const int o = blockIdx.x;
    const bool tap_pairs = C <= 16;
    int local = 0;
    for (int k = threadIdx.x; k < steps * 32; k += 256) {
        const int step = k >> 5, half = (k >> 4) & 1;
        int r, t, c;
        if (tap_pairs) {
            r = step / kw2, t = 2 * (step - r * kw2) + half, c = k & 15;
        } else {
            const int tap = step / npair;
            r = tap / kw, t = tap - r * kw, c = (step - tap * npair) * 32 + (k & 31);
        }
        uint8_t out = 0;
        if (o < O && c < C && t < kw) {
            const uint8_t v = W[((size_t)o * C + c) * kh * kw + r * kw + t];
            const int sv = (is_signed ? (int)(int8_t)v : (int)v) - shift;
            local += sv;
            out = (uint8_t)sv;
        }
        Ws[qfrag_offset(o, k, steps * 32)] = out;
    }
    __shared__ int part[256];
    part[threadIdx.x] = local;
    __syncthreads();
    for (int n = 128; n > 0; n >>= 1) {
        if (threadIdx.x < n) part[threadIdx.x] += part[threadIdx.x + n];
        __syncthreads();
    }
    if (threadIdx.x == 0) rowsum[o] = part[0];
}

struct DirectConvArgs {
    const uint8_t *X, *W;
    const uint8_t *x_zp, *w_zp;
    int x_signed, w_signed, host_zp, x_zp_value, w_zp_value;
    int n, C, H, Wd, O, kh, kw, sh, sw, dh, dw, pt, pl, group, Ho, Wo;
    void *Y;
    int requant;
    const float *ratio;
    int ratio_step;
    const int32_t *qbias;
    int y_zp, out_signed;
};

__global__ void __launch_bounds__(256) conv_direct_kernel(const DirectConvArgs p) {
    const long total = (long)p.n * p.O * p.Ho * p.Wo;
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int ow = (int)(idx % p.Wo);
    const int oh = (int)((idx / p.Wo) % p.Ho);
    const int o = (int)((idx / ((long)p.Wo * p.Ho)) % p.O);
    const int b = (int)(idx / ((long)p.Wo * p.Ho * p.O));
    const int zx = p.host_zp ? p.x_zp_value : zp_byte(p.x_zp, p.x_signed);
    const int zw = p.host_zp ? p.w_zp_value : zp_byte(p.w_zp, p.w_signed);
    const int cpg = p.C / p.group, opg = p.O / p.group;
    const int grp = o / opg;
    int acc = 0;
    for (int c = 0; c < cpg; c++) {
        const int ci = grp * cpg + c;
        for (int r = 0; r < p.kh; r++) {
            const int ih = oh * p.sh + r * p.dh - p.pt;
            if (ih < 0 || ih >= p.H) continue;
            for (int s = 0; s < p.kw; s++) {
                const int iw = ow * p.sw + s * p.dw - p.pl;
                if (iw < 0 || iw >= p.Wd) continue;
                const uint8_t xv = p.X[(((size_t)b * p.C + ci) * p.H + ih) * p.Wd + iw];
                const uint8_t wv = p.W[(((size_t)o * cpg + c) * p.kh + r) * p.kw + s];
                const int xi = (p.x_signed ? (int)(int8_t)xv : (int)xv) - zx;
                const int wi = (p.w_signed ? (int)(int8_t)wv : (int)wv) - zw;
                acc += xi * wi;
            }
        }
    }
    if (!p.requant) {
        static_cast<int32_t *>(p.Y)[idx] = acc;
    } else {
        if (p.qbias) acc += p.qbias[o];
        int q = (int)rintf(__fmul_rn((float)acc, p.ratio[(size_t)o * p.ratio_step])) + p.y_zp;
        if (p.out_signed)
            static_cast<int8_t *>(p.Y)[idx] = (int8_t)min(max(q, -128), 127);
        else
            static_cast<uint8_t *>(p.Y)[idx] = (uint8_t)min(max(q, 0), 255);
    }
}

// Depthwise convolutions (one input channel per group) with windows up to eight columns wide, no dilation along them and
// strides 1 and 2. One thread makes four neighbouring outputs of a row: per filter row it loads the words its window spans
// (from any byte address; words that reach past the row are loaded from inside it, shifted, and filled up with the zero
// point), and an output is one four-byte dot product per four taps, with the filter row as a word. What bounds it is that
// arithmetic, about 40 instructions per filter row of four outputs; conv_direct_kernel spends as many on one tap of one output,
// and 64-bit divisions. 16 x 48 x 111 x 111, 3 x 3: 85 -> 14.7 us; 8 x 128 x 28 x 28 9.7 -> 4.1.
struct DepthConvArgs {
    GemmArgs g;              // (first: gemm_note_scalars names offsets in a GemmArgs)
    const uint32_t *filter;  // [channel][filter row][NW words], signed, zeros past the window
    int quads;               // groups of four outputs per row
    int total;               // threads
    Magic by_quads, by_ho, by_o, by_per_group;
};

// the weight's rows as words, see DepthConvArgs
__global__ void __launch_bounds__(256)
pack_conv_depth_kernel(const uint8_t *__restrict__ W, uint32_t *__restrict__ F, int32_t *__restrict__ rowsum, int O, int kh, int kw, int words, int is_signed, int shift) {
    const int o = blockIdx.x * 256 + threadIdx.x;
    if (o >= O) return;
    int sum = 0;
    for (int r = 0; r < kh; r++)
        for (int w = 0; w < words; w++) {
            uint32_t v = 0;
            for (int b = 0; b < 4; b++) {
                const int s = 4 * w + b;
                if (s >= kw) continue;
                const uint8_t byte = W[((size_t)o * kh + r) * kw + s];
                const int sv = (is_signed ? (int)(int8_t)byte : (int)byte) - shift;
                sum += sv;
                v |= (uint32_t)(uint8_t)sv << (8 * b);
            }
            F[((size_t)o * kh + r) * words + w] = v;
        }
    rowsum[o] = sum;
}

// SW: stride along the row; NW: words of a filter row; SUMS: the weight's zero point is not zero, which takes the sums of each
// window (calls come here with one of zero; a recorded call may be given another)
template <int EPI, int SW, int NW, bool SUMS>
__global__ void __launch_bounds__(256) conv_depth_kernel(const DepthConvArgs a) {
    constexpr int NB = (3 * SW + 4 * NW + 3) / 4;   // words of input four outputs span
    const GemmArgs &p = a.g;
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= a.total) return;
    const int row = div_by_magic(idx, a.by_quads), ow = (idx - row * a.quads) * 4;
    const int plane = div_by_magic(row, a.by_ho), oh = row - plane * p.Ho;
    const int img = div_by_magic(plane, a.by_o), o = plane - img * p.I;
    const int ci = div_by_magic(o, a.by_per_group);
    const int zd = (p.host_zp ? p.dyn_zp_value : zp_byte(p.dyn_zp, p.dyn_signed)) - p.dyn_shift;
    const uint32_t zd4 = (uint32_t)(zd & 0xff) * 0x01010101u, flip4 = p.dyn_shift ? 0x80808080u : 0u;
    const int zc = SUMS ? p.const_zp_value : 0;
    const ConvChannel chan = conv_channel<EPI>(p, o);

    // word j of the span begins at column iw: where it is loaded from, how far that is off, which of its bytes exist
    int from[NB], off[NB];
    uint32_t keep[NB];
    const auto shifted = [](uint32_t v, int by) { return (uint32_t)(((uint64_t)v << 32) >> (32 + by)); };   // by: -24 .. 24 bits
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int iw = ow * SW - p.pl + 4 * j;
        from[j] = min(max(iw, 0), p.W - 4);
        const int d = iw - from[j];
        off[j] = 8 * min(max(d, -3), 3);
        keep[j] = d > -4 && d < 4 ? shifted(0xffffffffu, off[j]) : 0u;
    }
    const uint8_t *x = p.Q + ((size_t)img * p.C + ci) * p.H * p.W;
    const uint32_t *filter = a.filter + (size_t)o * p.kh * NW;
    int out[4] = {0, 0, 0, 0}, sum[4] = {0, 0, 0, 0};
    for (int r = 0; r < p.kh; r++) {
        const int ih = oh * p.sh - p.pt + r * p.dh;
        const bool inside = ih >= 0 && ih < p.H;
        const uint8_t *src = x + (size_t)min(max(ih, 0), p.H - 1) * p.W;
        uint32_t w[NB + 1];
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const uint32_t m = inside ? keep[j] : 0u, v = shifted(load_bytes4(src + from[j]) ^ flip4, off[j]);
            w[j] = (v & m) | (zd4 & ~m);
        }
        w[NB] = 0;
#pragma unroll
        for (int k = 0; k < NW; k++) {
            const int f = (int)filter[r * NW + k];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int b = i * SW + 4 * k;   // first byte of output i's taps 4 k ..
                out[i] = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_alignbyte(w[b / 4 + 1 < NB ? b / 4 + 1 : NB], w[b / 4], b % 4), f, out[i], false);
            }
            if (SUMS) {
                const int ones = p.kw - 4 * k >= 4 ? 0x01010101 : 0x01010101 & ((1 << (8 * (p.kw - 4 * k))) - 1);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int b = i * SW + 4 * k;
                    sum[i] = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_alignbyte(w[b / 4 + 1 < NB ? b / 4 + 1 : NB], w[b / 4], b % 4), ones, sum[i], false);
                }
            }
        }
    }
    const int fixed = -zd * chan.csum + p.kh * p.kw * zd * zc + (EPI == EPI_REQUANT ? chan.qb : 0);
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] += SUMS ? fixed - zc * sum[i] : fixed;
    const size_t at = (size_t)row * p.Wo + ow;
    if (EPI == EPI_REQUANT) {
        const RequantBytes bytes{chan.ratio, (float)p.y_zp + (p.out_signed ? 128.f : 0.f), p.out_signed ? 0x80808080u : 0u};
        const uint32_t word = gemm_requant4(bytes, out);
        if (ow + 3 < p.Wo) {
            __builtin_memcpy(static_cast<uint8_t *>(p.Y) + at, &word, 4);
            return;
        }
        for (int i = 0; i < 4; i++)
            if (ow + i < p.Wo) static_cast<uint8_t *>(p.Y)[at + i] = (uint8_t)(word >> (8 * i));
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (ow + i < p.Wo) static_cast<int32_t *>(p.Y)[at + i] = out[i];
    }
}

}  // namespace hipc

using namespace hipc;

struct hipc_conv_weight {
    hipc_conv_geom geom{};   // the geometry the weight was packed for (c_out, c_in, kh, kw, group)
    int w_dtype = HIPC_I8;
    uint8_t *raw = nullptr;  // ONNX layout copy, for the direct path
    uint8_t *Wp = nullptr;   // [O_pad, K_pad], (kh, kw, c) order; null when the MFMA path does not apply
    uint8_t *Ws = nullptr;   // the same in the step order of int8_conv_slab_kernel; null where that is Wp's own, or group > 1
    uint32_t *filter = nullptr;   // depthwise: the filter rows as words (conv_depth_kernel)
    int32_t *rowsum = nullptr;
    int O_pad = 0, K_pad = 0;
    mutable hipc::RatioCache ratios;  // QLinearConv's requantisation ratios as last used
};

namespace {

int out_dim(int64_t in, int64_t pb, int64_t pe, int64_t k, int64_t s, int64_t d, int64_t *out) {
    const int64_t span = d * (k - 1) + 1, padded = in + pb + pe;
    if (padded < span) return HIPC_ERR_INVALID;
    *out = (padded - span) / s + 1;
    return HIPC_OK;
}

int check_geom(hipc_ctx *ctx, const hipc_conv_geom *g, int64_t *ho, int64_t *wo) {
    HIPC_REQUIRE(ctx, g, "Conv: null geometry");
    HIPC_REQUIRE(ctx, g->n >= 0 && g->c_in > 0 && g->h > 0 && g->w > 0 && g->c_out > 0 && g->kh > 0 && g->kw > 0,
                 "Conv: non-positive dimension");
    HIPC_REQUIRE(ctx, g->stride_h > 0 && g->stride_w > 0 && g->dil_h > 0 && g->dil_w > 0, "Conv: strides and dilations must be positive");
    HIPC_REQUIRE(ctx, g->pad_top >= 0 && g->pad_left >= 0 && g->pad_bottom >= 0 && g->pad_right >= 0, "Conv: negative padding");
    HIPC_REQUIRE(ctx, g->group > 0 && g->c_in % g->group == 0 && g->c_out % g->group == 0,
                 "Conv: group %ld does not divide the channels (%ld in, %ld out)", (long)g->group, (long)g->c_in, (long)g->c_out);
    HIPC_REQUIRE(ctx,
                 out_dim(g->h, g->pad_top, g->pad_bottom, g->kh, g->stride_h, g->dil_h, ho) == HIPC_OK &&
                     out_dim(g->w, g->pad_left, g->pad_right, g->kw, g->stride_w, g->dil_w, wo) == HIPC_OK,
                 "Conv: the kernel window does not fit the padded input");
    const int64_t big = int64_t(1) << 30;
    HIPC_REQUIRE(ctx, g->n * g->c_out * *ho * *wo < big * 2 && g->n * g->c_in * g->h * g->w < big * 2 && g->c_in * g->kh * g->kw < big,
                 "Conv: tensor too large");
    return HIPC_OK;
}

bool same_weight_shape(const hipc_conv_geom &a, const hipc_conv_geom &b) {
    return a.c_in == b.c_in && a.c_out == b.c_out && a.kh == b.kh && a.kw == b.kw && a.group == b.group;
}

struct ConvEpilogue {
    int requant = 0;
    const float *ratio = nullptr;  // device
    int ratio_step = 0;
    const int32_t *qbias = nullptr;
    int y_zp = 0, out_signed = 0;
};

// one output per thread, any geometry
int run_direct(hipc_ctx *ctx, const void *X, int x_dtype, const hipc_conv_weight *W, const void *x_zp, const void *w_zp,
               int host_zp, int x_zp_value, int w_zp_value, const hipc_conv_geom *g, int64_t ho, int64_t wo, void *Y, const ConvEpilogue &ep) {
    const int64_t total = g->n * g->c_out * ho * wo;
    DirectConvArgs d{};
    d.X = static_cast<const uint8_t *>(X), d.W = W->raw;
    d.x_zp = static_cast<const uint8_t *>(x_zp), d.w_zp = static_cast<const uint8_t *>(w_zp);
    d.x_signed = x_dtype == HIPC_I8, d.w_signed = W->w_dtype == HIPC_I8;
    d.host_zp = host_zp, d.x_zp_value = x_zp_value, d.w_zp_value = w_zp_value;
    d.n = (int)g->n, d.C = (int)g->c_in, d.H = (int)g->h, d.Wd = (int)g->w, d.O = (int)g->c_out;
    d.kh = (int)g->kh, d.kw = (int)g->kw, d.sh = (int)g->stride_h, d.sw = (int)g->stride_w, d.dh = (int)g->dil_h,
    d.dw = (int)g->dil_w, d.pt = (int)g->pad_top, d.pl = (int)g->pad_left, d.group = (int)g->group;
    d.Ho = (int)ho, d.Wo = (int)wo;
    d.Y = Y;
    d.requant = ep.requant, d.ratio = ep.ratio, d.ratio_step = ep.ratio_step, d.qbias = ep.qbias, d.y_zp = ep.y_zp,
    d.out_signed = ep.out_signed;
    hipLaunchKernelGGL((conv_direct_kernel), dim3((unsigned)ceil_div(total, 256)), 256, 0, ctx->stream, d);
    HIPC_LAUNCHED(ctx);
    if (host_zp) {
        note_scalar(ctx, HIPC_SCALAR_A_ZERO_POINT, offsetof(DirectConvArgs, x_zp_value));
        note_scalar(ctx, HIPC_SCALAR_B_ZERO_POINT, offsetof(DirectConvArgs, w_zp_value));
    }
    if (ep.requant) note_scalar(ctx, HIPC_SCALAR_Y_ZERO_POINT, offsetof(DirectConvArgs, y_zp));
    return HIPC_OK;
}

// product steps of int8_conv_slab_kernel: chunks, pairs of them per tap, taps or pairs of taps per filter row
void slab_steps(const hipc_conv_geom &g, ConvSlabArgs *a) {
    a->nch = (int)ceil_div(g.c_in, 16);
    const bool tap_pairs = a->nch == 1;
    a->npair = tap_pairs ? 1 : (a->nch + 1) / 2;
    a->kw2 = (int)(tap_pairs ? ceil_div(g.kw, 2) : g.kw);
    a->pairs = tap_pairs;
    a->steps = (int)g.kh * a->kw2 * a->npair;
}

template <int EPI, bool DYN, int WK, int WP, bool RAGGED>
int slab_launch(hipc_ctx *ctx, const ConvSlabArgs &a, size_t lds) {
    static bool lds_allowed[kMaxDevices] = {};
    if (int rc = allow_dynamic_lds(ctx, int8_conv_slab_kernel<EPI, DYN, WK, WP, RAGGED>, kSlabLds, lds_allowed)) return rc;
    hipLaunchKernelGGL((int8_conv_slab_kernel<EPI, DYN, WK, WP, RAGGED>), dim3(8u * (unsigned)a.per_xcd), 256, lds, ctx->stream, a);
    HIPC_LAUNCHED(ctx);
    const void *with_sums = nullptr;
    if (!DYN && ctx->capturing) {
        static bool sums_allowed[kMaxDevices] = {};
        if (int rc = allow_dynamic_lds(ctx, int8_conv_slab_kernel<EPI, true, WK, WP, RAGGED>, kSlabLds, sums_allowed)) return rc;
        with_sums = reinterpret_cast<const void *>(int8_conv_slab_kernel<EPI, true, WK, WP, RAGGED>);
    }
    gemm_note_scalars(ctx, a.g, DYN, with_sums);
    return HIPC_OK;
}
template <int EPI, bool DYN, int WK, int WP>
int slab_launch_ragged(hipc_ctx *ctx, const ConvSlabArgs &a, size_t lds) {
    return a.g.C % 16 ? slab_launch<EPI, DYN, WK, WP, true>(ctx, a, lds) : slab_launch<EPI, DYN, WK, WP, false>(ctx, a, lds);
}
template <int WK, int WP>
int slab_launch_as(hipc_ctx *ctx, ConvSlabArgs a, size_t lds, bool requant, bool sums) {
    a.adv_tap = WK / a.npair, a.adv_q = WK % a.npair;
    if (requant) return sums ? slab_launch_ragged<EPI_REQUANT, true, WK, WP>(ctx, a, lds) : slab_launch_ragged<EPI_REQUANT, false, WK, WP>(ctx, a, lds);
    return sums ? slab_launch_ragged<EPI_I32, true, WK, WP>(ctx, a, lds) : slab_launch_ragged<EPI_I32, false, WK, WP>(ctx, a, lds);
}

// positions a slab of int8_conv_slab_kernel needs for `tile` consecutive outputs, whichever they are: rounded up to fours
// from a multiple of four on, and the padding position
int64_t slab_positions(const hipc_conv_geom &g, int64_t ho, int64_t wo, int64_t tile) {
    tile = std::min(tile, ho * wo);
    const int64_t rows = wo % tile == 0 ? 1 : tile % wo == 0 ? tile / wo : std::min(ho, (tile + wo - 2) / wo + 1);
    const int64_t span = (g.kh - 1) * g.dil_h + 1;
    const int64_t within = (std::min(g.h, span) - 1) * g.w + std::min(g.w, (std::min(tile, wo) - 1) * g.stride_w + (g.kw - 1) * g.dil_w + 1);
    const int64_t across = rows > 1 ? std::min(g.h, (rows - 1) * g.stride_h + span) * g.w : 0;
    return (std::max(within, across) + 3 + 3) / 4 * 4 + 2;
}

// The slab kernel, where what 64 outputs see of the input fits LDS (*taken).
int run_slab(hipc_ctx *ctx, const GemmArgs &ga, const hipc_conv_weight *W, const hipc_conv_geom *g, int64_t ho, int64_t wo, bool requant, bool sums, bool *taken) {
    *taken = false;
    if (g->h * g->w < 4) return HIPC_OK;
    ConvSlabArgs a{};
    a.g = ga;
    slab_steps(*g, &a);
    a.frag_steps = W->Ws ? a.steps : W->K_pad / 32;
    if (W->Ws) a.g.P = W->Ws;
    const auto slab_of = [&](int64_t tile) { return (size_t)a.nch * slab_positions(*g, ho, wo, tile) * 16; };
    const auto lds_of = [&](int64_t tile) { return slab_of(tile) + (size_t)(g->kh * a.kw2 * (a.pairs ? 2 : 1) * tile * 2); };
    const int64_t J = ho * wo, cus = std::max(1, ctx->cu_count), o64 = ceil_div(g->c_out, 64);
    // Few tiles of 64 x 64 and enough steps to share: the four wavefronts of a workgroup split k. Else a wavefront keeps its k
    // to itself and takes 32 channels: 128 channels x 64 positions, or, where the channels would leave wavefronts of the
    // last tile idle, 64 x 128.
    const bool by_k = o64 * ceil_div(J, 64) * g->n <= 2 * cus && a.steps >= 8;
    const bool wide = !by_k && o64 % 2 == 1 && o64 <= 3 && J > 64 && lds_of(128) <= kSlabLds;
    const int tile = wide ? 128 : 64;
    size_t lds = lds_of(tile);
    if (lds > kSlabLds) return HIPC_OK;
    *taken = true;
    if (by_k) lds = std::max(lds, kSmallLds);
    a.SP = (int)slab_positions(*g, ho, wo, tile), a.tab_at = (int)slab_of(tile);
    a.o_tiles = (int)(by_k || wide ? o64 : ceil_div(g->c_out, 128)), a.p_tiles = (int)ceil_div(J, tile);
    a.items = (int)((int64_t)a.o_tiles * a.p_tiles * g->n), a.per_xcd = (int)ceil_div(a.items, 8);
    a.by_o_tiles = magic_of((uint32_t)a.o_tiles), a.by_p_tiles = magic_of((uint32_t)a.p_tiles), a.by_wo = magic_of((uint32_t)wo);
    return by_k ? slab_launch_as<4, 1>(ctx, a, lds, requant, sums) : wide ? slab_launch_as<1, 2>(ctx, a, lds, requant, sums) : slab_launch_as<1, 1>(ctx, a, lds, requant, sums);
}

// Depthwise, where conv_depth_kernel has the case
int depth_words(const hipc_conv_geom &g) { return g.group == g.c_in && g.kw <= 8 ? (int)ceil_div(g.kw, 4) : 0; }
template <int EPI>
int depth_launch(hipc_ctx *ctx, const DepthConvArgs &a, int words) {
    const auto run = [&](auto stride, auto nw) -> int {
        constexpr int SW = decltype(stride)::value, NW = decltype(nw)::value;
        hipLaunchKernelGGL((conv_depth_kernel<EPI, SW, NW, false>), dim3((unsigned)ceil_div(a.total, 256)), 256, 0, ctx->stream, a);
        HIPC_LAUNCHED(ctx);
        gemm_note_scalars(ctx, a.g, false, reinterpret_cast<const void *>(conv_depth_kernel<EPI, SW, NW, true>));
        return HIPC_OK;
    };
    constexpr std::integral_constant<int, 1> one{};
    constexpr std::integral_constant<int, 2> two{};
    if (a.g.sw == 1) return words == 1 ? run(one, one) : run(one, two);
    return words == 1 ? run(two, one) : run(two, two);
}

int run_conv(hipc_ctx *ctx, const void *X, int x_dtype, const hipc_conv_weight *W, const void *x_zp, const void *w_zp,
             int host_zp, int x_zp_value, int w_zp_value, const hipc_conv_geom *g, void *Y, const ConvEpilogue &ep) {
    int64_t ho = 0, wo = 0;
    int rc = check_geom(ctx, g, &ho, &wo);
    if (rc != HIPC_OK) return rc;
    HIPC_REQUIRE(ctx, W, "Conv: null weight");
    HIPC_REQUIRE(ctx, same_weight_shape(*g, W->geom), "Conv: the weight was prepacked for a different shape");
    HIPC_REFUSE(ctx, !is_byte_dtype(x_dtype), "Conv: X must be uint8 or int8, got %d", x_dtype);
    const int64_t total = g->n * g->c_out * ho * wo;
    if (total == 0) return HIPC_OK;
    HIPC_REQUIRE(ctx, X && Y, "Conv: null tensor");

    if (W->rowsum) {
        GemmArgs ga{};
        ga.P = W->Wp;
        ga.const_sum = W->rowsum;
        ga.dyn_zp = static_cast<const uint8_t *>(x_zp), ga.const_zp = static_cast<const uint8_t *>(w_zp);
        ga.dyn_shift = x_dtype == HIPC_U8 ? 128 : 0, ga.const_shift = W->w_dtype == HIPC_U8 ? 128 : 0;
        ga.dyn_signed = x_dtype == HIPC_I8, ga.const_signed = W->w_dtype == HIPC_I8;
        ga.host_zp = host_zp, ga.dyn_zp_value = x_zp_value, ga.const_zp_value = w_zp_value;
        ga.I = (int)g->c_out, ga.J = (int)(ho * wo), ga.K = (int)(g->c_in * g->kh * g->kw), ga.K_pad = W->K_pad;
        ga.C = (int)g->c_in, ga.H = (int)g->h, ga.W = (int)g->w, ga.Ho = (int)ho, ga.Wo = (int)wo;
        ga.kh = (int)g->kh, ga.kw = (int)g->kw, ga.sh = (int)g->stride_h, ga.sw = (int)g->stride_w;
        ga.dh = (int)g->dil_h, ga.dw = (int)g->dil_w, ga.pt = (int)g->pad_top, ga.pl = (int)g->pad_left;
        ga.Y = Y;
        ga.ratio = ep.ratio, ga.ratio_step = ep.ratio_step, ga.qbias = ep.qbias, ga.y_zp = ep.y_zp,
        ga.out_signed = ep.out_signed;
        // the row sums of the activations only matter when the weight's zero point, in the signed domain, is not zero
        const bool zero_known = ga.const_shift == 0 && (host_zp ? w_zp_value == 0 : w_zp == nullptr);
        ga.Q = static_cast<const uint8_t *>(X);
        if (W->filter) {
            const int64_t quads = ceil_div(wo, 4), threads = g->n * g->c_out * ho * quads;
            if (!zero_known || g->dil_w != 1 || g->stride_w > 2 || g->w < 4)   // (a weight zero point needs the sums of each output's window)
                return run_direct(ctx, X, x_dtype, W, x_zp, w_zp, host_zp, x_zp_value, w_zp_value, g, ho, wo, Y, ep);
            DepthConvArgs a{};
            a.g = ga, a.filter = W->filter, a.quads = (int)quads, a.total = (int)threads;
            a.by_quads = magic_of((uint32_t)quads), a.by_ho = magic_of((uint32_t)ho), a.by_o = magic_of((uint32_t)g->c_out);
            a.by_per_group = magic_of((uint32_t)(g->c_out / g->group));
            return ep.requant ? depth_launch<EPI_REQUANT>(ctx, a, depth_words(*g)) : depth_launch<EPI_I32>(ctx, a, depth_words(*g));
        }
        // few 64x64 tiles and a long k: the wavefronts of a workgroup split k and the weight stays out of LDS
        // (the gemm_small option, 0 / 1, overrides: tuning, tests)
        const int forced = ctx->tune.gemm_small;
        const int64_t tiles64 = ceil_div(ga.I, 64) * ceil_div(ga.J, 64) * g->n;
        const bool small = forced >= 0 ? forced != 0 : (tiles64 <= 2 * (int64_t)ctx->cu_count && ga.K_pad >= 4 * kBK);

        // A convolution along W alone with few tiles, whose input slab fits LDS: the kernel made for it, one instruction
        // cheaper wherever int8_conv_slab_kernel allows for rows, padding and odd addresses (192 x 4096, k = 7: 6.5 against
        // 7.0 us; with more tiles than two per CU that kernel does not split k and is the faster one).
        // The conv_row option set to 0 takes the general route (tuning, tests).
        const bool row_off = ctx->tune.conv_row == 0;
        const int64_t slab_pos = (3 + 63 * g->stride_w + (g->kw - 1) * g->dil_w + 1 + 3) / 4 * 4;
        const size_t slab_bytes = (size_t)(slab_pos * g->c_in);
        if (W->Wp && !row_off && tiles64 <= 2 * (int64_t)ctx->cu_count && g->h == 1 && g->kh == 1 && ho == 1 && g->pad_top == 0 && g->w % 4 == 0 && aligned(X, 4) &&
            slab_bytes <= 64 * 1024) {
            ga.slab_pos = (int)slab_pos;
            const size_t lds = std::max(kSmallLds, slab_bytes);
            const dim3 grid(gemm_grid(ga, 64), 1, (unsigned)g->n);
            if (ep.requant) {
                if (zero_known) hipLaunchKernelGGL((int8_conv_row_kernel<EPI_REQUANT, false>), grid, 256, lds, ctx->stream, ga);
                else hipLaunchKernelGGL((int8_conv_row_kernel<EPI_REQUANT, true>), grid, 256, lds, ctx->stream, ga);
            } else {
                if (zero_known) hipLaunchKernelGGL((int8_conv_row_kernel<EPI_I32, false>), grid, 256, lds, ctx->stream, ga);
                else hipLaunchKernelGGL((int8_conv_row_kernel<EPI_I32, true>), grid, 256, lds, ctx->stream, ga);
            }
            HIPC_LAUNCHED(ctx);
            gemm_note_scalars(ctx, ga, !zero_known);
            return HIPC_OK;
        }

        // any other whose slab fits
        bool taken = false;
        if (!row_off) {
            rc = run_slab(ctx, ga, W, g, ho, wo, ep.requant != 0, !zero_known, &taken);
            if (taken) return rc;
        }
        if (!W->Wp) return run_direct(ctx, X, x_dtype, W, x_zp, w_zp, host_zp, x_zp_value, w_zp_value, g, ho, wo, Y, ep);
        HIPC_REQUIRE(ctx, g->n <= 65535, "Conv: batch %ld too large", (long)g->n);
        // NHWC copy of the activation, shifted to the signed domain
        void *xt = nullptr;
        const size_t x_bytes = (size_t)(g->n * g->c_in * g->h * g->w);
        rc = scratch_get(ctx, 1, x_bytes + 16, &xt);
        if (rc != HIPC_OK) return rc;
        const int HW = (int)(g->h * g->w);
        if (g->c_in % 4 == 0 && HW % 4 == 0 && aligned(X, 4))
            hipLaunchKernelGGL((nchw_to_nhwc4_kernel), dim3((unsigned)ceil_div(HW, 64), (unsigned)ceil_div(g->c_in, 64), (unsigned)g->n), 256, 0, ctx->stream, static_cast<const uint8_t *>(X), static_cast<uint8_t *>(xt), (int)g->c_in, HW,
                                                  x_dtype == HIPC_U8 ? 0x80808080u : 0u);
        else
            hipLaunchKernelGGL((nchw_to_nhwc_kernel), dim3((unsigned)ceil_div(HW, 32), (unsigned)ceil_div(g->c_in, 32), (unsigned)g->n), 256, 0, ctx->stream, static_cast<const uint8_t *>(X), static_cast<uint8_t *>(xt), (int)g->c_in, HW,
                                                 x_dtype == HIPC_U8 ? 0x80 : 0);
        HIPC_LAUNCHED(ctx);
        ga.Q = static_cast<const uint8_t *>(xt);
        if (small) {
            const dim3 grid(gemm_grid(ga, 64), 1, (unsigned)g->n);
            if (ep.requant) {
                if (zero_known) hipLaunchKernelGGL((int8_conv_small_kernel<EPI_REQUANT, false>), grid, 256, kSmallLds, ctx->stream, ga);
                else hipLaunchKernelGGL((int8_conv_small_kernel<EPI_REQUANT, true>), grid, 256, kSmallLds, ctx->stream, ga);
            } else {
                if (zero_known) hipLaunchKernelGGL((int8_conv_small_kernel<EPI_I32, false>), grid, 256, kSmallLds, ctx->stream, ga);
                else hipLaunchKernelGGL((int8_conv_small_kernel<EPI_I32, true>), grid, 256, kSmallLds, ctx->stream, ga);
            }
            HIPC_LAUNCHED(ctx);
            gemm_note_scalars(ctx, ga, !zero_known);
            return HIPC_OK;
        }
        return ep.requant ? gemm_launch<MODE_CONV, EPI_REQUANT, true>(ctx, ga, (unsigned)g->n)
                          : gemm_launch<MODE_CONV, EPI_I32, true>(ctx, ga, (unsigned)g->n);
    }

    return run_direct(ctx, X, x_dtype, W, x_zp, w_zp, host_zp, x_zp_value, w_zp_value, g, ho, wo, Y, ep);
}

}  // namespace

extern "C" {

int hipc_conv_out_shape(const hipc_conv_geom *g, int64_t *h_out, int64_t *w_out) {
    if (!g || !h_out || !w_out) return HIPC_ERR_INVALID;
    if (g->kh <= 0 || g->kw <= 0 || g->stride_h <= 0 || g->stride_w <= 0 || g->dil_h <= 0 || g->dil_w <= 0)
        return HIPC_ERR_INVALID;
    if (out_dim(g->h, g->pad_top, g->pad_bottom, g->kh, g->stride_h, g->dil_h, h_out) != HIPC_OK) return HIPC_ERR_INVALID;
    return out_dim(g->w, g->pad_left, g->pad_right, g->kw, g->stride_w, g->dil_w, w_out);
}

void hipc_same_pads(int64_t in, int64_t kernel, int64_t stride, int64_t dilation, int upper, int64_t *pad_begin,
                    int64_t *pad_end) {
    const int64_t out = (in + stride - 1) / stride;
    const int64_t span = dilation * (kernel - 1) + 1;
    int64_t total = (out - 1) * stride + span - in;
    if (total < 0) total = 0;
    const int64_t small = total / 2, large = total - small;
    *pad_begin = upper ? small : large;
    *pad_end = upper ? large : small;
}

int hipc_prepack_conv_w(hipc_ctx *ctx, const void *W, int w_dtype, const hipc_conv_geom *g, hipc_conv_weight **out) {
    if (!out) return HIPC_ERR_INVALID;
    return entry(ctx, [&]() -> int {
        *out = nullptr;
        HIPC_REFUSE(ctx, ctx->capturing, "Conv prepack while a capture is open");
        HIPC_REFUSE(ctx, !is_byte_dtype(w_dtype), "Conv: W must be uint8 or int8, got %d", w_dtype);
        HIPC_REQUIRE(ctx, W && g, "Conv prepack: null argument");
        HIPC_REQUIRE(ctx, g->c_in > 0 && g->c_out > 0 && g->kh > 0 && g->kw > 0 && g->group > 0 && g->c_in % g->group == 0 &&
                              g->c_out % g->group == 0 && g->c_in * g->kh * g->kw < (int64_t(1) << 30),
                     "Conv prepack: bad weight shape");
        hipc_conv_weight *w = new hipc_conv_weight();
        w->geom = *g;
        w->w_dtype = w_dtype;
        const size_t raw_bytes = (size_t)(g->c_out * (g->c_in / g->group) * g->kh * g->kw);
        hipError_t e = hipMalloc(reinterpret_cast<void **>(&w->raw), raw_bytes);
        if (e == hipSuccess)
            e = hipMemcpyAsync(w->raw, W, raw_bytes, hipMemcpyDeviceToDevice, ctx->stream);
        const bool mfma = g->group == 1 && g->c_in % 16 == 0;
        if (e == hipSuccess && g->group == 1) {
            w->O_pad = (int)(ceil_div(g->c_out, kBM) * kBM);
            e = hipMalloc(reinterpret_cast<void **>(&w->rowsum), (size_t)w->O_pad * 4);
        }
        if (e == hipSuccess && g->group > 1 && depth_words(*g) > 0) {
            e = hipMalloc(reinterpret_cast<void **>(&w->rowsum), (size_t)g->c_out * 4);
            if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(&w->filter), (size_t)(g->c_out * g->kh * depth_words(*g)) * 4);
            if (e == hipSuccess) {
                hipLaunchKernelGGL((pack_conv_depth_kernel), dim3((unsigned)ceil_div(g->c_out, 256)), 256, 0, ctx->stream, static_cast<const uint8_t *>(W), w->filter, w->rowsum, (int)g->c_out, (int)g->kh, (int)g->kw,
                    depth_words(*g), w_dtype == HIPC_I8, w_dtype == HIPC_U8 ? 128 : 0);
                e = hipGetLastError();
            }
        }
        if (e == hipSuccess && g->group == 1 && g->c_in % 32 != 0) {
            ConvSlabArgs a{};
            slab_steps(*g, &a);
            e = hipMalloc(reinterpret_cast<void **>(&w->Ws), (size_t)w->O_pad * a.steps * 32);
            if (e == hipSuccess) {
                hipLaunchKernelGGL((pack_conv_slab_kernel), dim3((unsigned)w->O_pad), 256, 0, ctx->stream, static_cast<const uint8_t *>(W), w->Ws, w->rowsum, (int)g->c_out, (int)g->c_in, (int)g->kh, (int)g->kw,
                    a.kw2, a.npair, a.steps, w_dtype == HIPC_I8, w_dtype == HIPC_U8 ? 128 : 0);
                e = hipGetLastError();
            }
        }
        if (e == hipSuccess && mfma) {
            w->K_pad = (int)(ceil_div(g->c_in * g->kh * g->kw, kBK) * kBK);
            e = hipMalloc(reinterpret_cast<void **>(&w->Wp), (size_t)w->O_pad * w->K_pad);
            if (e == hipSuccess) {
                hipLaunchKernelGGL((pack_conv_w_kernel), dim3((unsigned)w->O_pad), 256, 0, ctx->stream, static_cast<const uint8_t *>(W), w->Wp, w->rowsum, (int)g->c_out, (int)g->c_in, (int)g->kh, (int)g->kw,
                    w->O_pad, w->K_pad, w_dtype == HIPC_I8, w_dtype == HIPC_U8 ? 128 : 0);
                e = hipGetLastError();
            }
        }
        if (e != hipSuccess) {
            if (w->raw) (void)hipFree(w->raw);
            if (w->Wp) (void)hipFree(w->Wp);
            if (w->Ws) (void)hipFree(w->Ws);
            if (w->filter) (void)hipFree(w->filter);
            if (w->rowsum) (void)hipFree(w->rowsum);
            delete w;
            return fail(ctx, HIPC_ERR_BACKEND, "Conv prepack: %s", hipGetErrorString(e));
        }
        *out = w;
        return HIPC_OK;
    });
}

void hipc_conv_weight_destroy(hipc_ctx *ctx, hipc_conv_weight *w) {
    if (!w) return;
    entry_void(ctx, [&] {
        if (w->raw) ctx->deferred.push_back(w->raw);
        if (w->Wp) ctx->deferred.push_back(w->Wp);
        if (w->Ws) ctx->deferred.push_back(w->Ws);
        if (w->filter) ctx->deferred.push_back(w->filter);
        if (w->rowsum) ctx->deferred.push_back(w->rowsum);
        ratio_release(ctx, w->ratios);
        delete w;
    });
}

int hipc_conv_integer(hipc_ctx *ctx, const void *X, int x_dtype, const hipc_conv_weight *W, const void *x_zp,
                      const void *w_zp, const hipc_conv_geom *g, void *Y) {
    return entry(ctx, [&]() -> int {
        return run_conv(ctx, X, x_dtype, W, x_zp, w_zp, 0, 0, 0, g, Y, ConvEpilogue{});
    });
}

int hipc_qlinear_conv(hipc_ctx *ctx, const void *X, int x_dtype, float x_scale, int32_t x_zp, const hipc_conv_weight *W,
                      const float *w_scale, int64_t n_w_scale, int32_t w_zp, float y_scale, int32_t y_zp, int y_dtype,
                      const void *bias, const hipc_conv_geom *g, void *Y) {
    return entry(ctx, [&]() -> int {
        HIPC_REQUIRE(ctx, g && w_scale, "QLinearConv: null geometry or scale");
        HIPC_REFUSE(ctx, !is_byte_dtype(y_dtype), "QLinearConv: output must be uint8 or int8, got %d", y_dtype);
        // the accepted envelope of `unsupported_quantization` (interp.rs:781-847)
        HIPC_REQUIRE(ctx, n_w_scale == 1 || n_w_scale == g->c_out, "QLinearConv: %ld weight scales for %ld channels",
                     (long)n_w_scale, (long)g->c_out);
        HIPC_REFUSE(ctx, n_w_scale > 1 && w_zp != 0, "QLinearConv: w per-channel zero point is not zero (asymmetric weights)");
        HIPC_REQUIRE(ctx, y_scale != 0.f, "QLinear: y_scale is zero");
        HIPC_REQUIRE(ctx, W, "QLinearConv: null weight");
        // a per-tensor scale is broadcast to c_out so the bias stays per channel (interp.rs:4815-4823)
        const float *dratio = nullptr;
        int rc = ratio_resident(ctx, W->ratios, x_scale, w_scale, n_w_scale, y_scale, g->c_out, &dratio);
        if (rc != HIPC_OK) return rc;
        ConvEpilogue ep;
        ep.requant = 1;
        ep.ratio = dratio, ep.ratio_step = 1;
        ep.qbias = static_cast<const int32_t *>(bias);
        ep.y_zp = y_zp, ep.out_signed = y_dtype == HIPC_I8;
        return run_conv(ctx, X, x_dtype, W, nullptr, nullptr, 1, x_zp, w_zp, g, Y, ep);
    });
}

}  // extern "C"
