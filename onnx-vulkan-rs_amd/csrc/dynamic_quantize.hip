// DynamicQuantizeLinear for gfx950.
//
// Reference: crates/onnx-vulkan-core/src/shaders/dynamic_quantize.rs:106-222 (the two
// passes and the range slot), interp.rs:1945-2085 (host side), definition
// tests/dynamic_quantize.rs:16-26.
//
// The range slot is 8 bytes {bits(-min), bits(max)}. The range always contains 0,
// so both values are >= 0 and their bit patterns order like the values: an
// unsigned atomicMax on the words is a float max, independent of the order the
// workgroups arrive in. The reference replaces `/` by a double-single reciprocal
// because Vulkan's OpFDiv may be 2.5 ULP off; here `__fdiv_rn` is the IEEE
// division, so the operator's definition is evaluated as written.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "internal.h"
#include "lanes.h"

namespace hipc {

// Up to how many values dql_small_kernel, whose every workgroup reads (of a GELU: evaluates) all of them, beats the launch whose
// workgroups tell each other their ranges. Us, both: 32768 values 4.04 / 4.62, 40960 4.36 / 4.62, 65536 5.7 / 4.65; of a GELU
// 4097 4.31 / 4.9, 6000 4.59 / 4.9, 8192 5.1 / 5.0, 16384 6.7 / 5.0.
constexpr int64_t kSmallPlain = 40960, kSmallGelu = 6144;
constexpr long kMeetTicks = 1000;   // 10 us: twice what the workgroups of a launch are apart on a chip of their own (16 M values: 20.3 us with 5 us and more, 28 with 2 us)


// Range partials of hipc_dynamic_quantize_linear_static: {bits(-min), bits(max)} per workgroup of
// the first pass, kParamPartsMax pairs = 16 KiB, part of the library's device image. In host code
// this name is a stand-in, not a device address: dql_static_init asks the runtime where the array
// lives on the context's device, and every launch gets that pointer.
static __device__ __align__(256) __attribute__((used)) uint32_t scratch[2 * kParamPartsMax];

int dql_static_init(hipc_ctx *ctx) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) return HIPC_ERR_BACKEND;
    ctx->dql_static = ptr;
    return HIPC_OK;
}

// Division by a value that is the same for every element (a quantizer's scale, GELU's divisor), correctly rounded, in five
// instructions instead of the ten of a general IEEE division: q = v * rc with rc = 1 / d rounded to nearest is within 1.5 ulp,
// and each correction adds the exactly formed remainder times rc. After the first one q is within just over half an ulp; the
// second one then rounds what the true quotient rounds to: its error is below b 2^-26 ulp for a divisor mantissa b < 2,
// while a quotient is never closer than 2^-24 / b ulp to a midpoint (Markstein's theorem). No remainder may be lost below
// the smallest number and no product may overflow: the callers see to that.
__device__ __forceinline__ float div_by(float v, float d, float rc) {
    float q = v * rc;
    q = fmaf(fmaf(-q, d, v), rc, q);
    return fmaf(fmaf(-q, d, v), rc, q);
}

// What the quantizer reads: x itself, or DecomposedGelu(x), the exact GELU written out as
// Div -> Erf -> Add -> Mul -> Mul and fused by the reference (rewrite.rs:683-735). Every one of the five rounds
// on its own, as the kernels it replaces do (shaders/elementwise.rs:71-118): this file is
// compiled with floating-point contraction off, so the fused quantizer and the plain GELU kernel
// below evaluate bit for bit the same function.
enum { GELU_OFF = 0, GELU_SQRT2 = 1, GELU_ANY = 2 };   // GELU_SQRT2: the divisor is sqrt(2) as a float, which exported graphs have
struct GeluParams {
    int on;             // one of the above (the kernels are instantiated on it)
    float divisor, offset, factor;
    int factor_first;   // x * ((erf + offset) * factor) instead of (x * (erf + offset)) * factor
};

// shaders/elementwise.rs:71-80 (Abramowitz-Stegun 7.1.26); |x| <= 32. The passes over a GELU are bound by these
// instructions (16 M values: 21 us a pass at 40 of them, for 65 MB), so:
//   * 1 / (1 + p a), an argument in [1, 12]: the hardware's estimate and one correction, which for every one of the 2^23
//     mantissas gives the correctly rounded reciprocal;
//   * exp(-a^2) as 2^h times (1 + r ln 2), h + r being -a^2 log2(e) to 48 bits: no range reduction, since the hardware's
//     exponential takes the whole range and nothing here overflows.
__device__ __forceinline__ float erf_approx(float x) {
    const float a = fabsf(x);
    const float y = fmaf(0.3275911f, a, 1.f);
    const float r0 = __builtin_amdgcn_rcpf(y);
    const float t = fmaf(fmaf(-y, r0, 1.f), r0, r0);
    const float poly = t * fmaf(t, fmaf(t, fmaf(t, fmaf(t, 1.061405429f, -1.453152027f), 1.421413741f), -0.284496736f), 0.254829592f);
    constexpr float log2e = 1.44269502f, ln2 = 0.693147181f;
    const float s = -(a * a), h = s * log2e, r = fmaf(s, log2e, -h);
    const float e2 = __builtin_amdgcn_exp2f(h), e = fmaf(e2, r * ln2, e2);
    return copysignf(fmaf(-poly, e, 1.f), x);   // (for x = 0 the caller multiplies by 0)
}

// Past 32 the error function has long been 1 (from 10.2 on): clamping there keeps infinities out of the quotient and the square.
template <int GELU>
__device__ __forceinline__ float gelu_load(float v, const GeluParams &g) {
    if (GELU == GELU_OFF) return v;
    float x;
    if (GELU == GELU_SQRT2) {
        // div_by with a single correction: for this divisor it gives the IEEE quotient for every one of the 2^23 mantissas
        constexpr float d = 1.41421356f, rc = 1.f / d;
        const float c = __builtin_amdgcn_fmed3f(v, -64.f, 64.f), q = c * rc;
        x = fmaf(fmaf(-q, d, c), rc, q);
    } else {
        x = fminf(fmaxf(v / g.divisor, -32.f), 32.f);
    }
    const float e = erf_approx(x) + g.offset;
    return g.factor_first ? v * (e * g.factor) : (v * e) * g.factor;
}
template <int GELU>
__device__ __forceinline__ float4 gelu_load4(float4 v, const GeluParams &g) {
    return make_float4(gelu_load<GELU>(v.x, g), gelu_load<GELU>(v.y, g), gelu_load<GELU>(v.z, g), gelu_load<GELU>(v.w, g));
}

template <int GELU>
__global__ void __launch_bounds__(256)
decomposed_gelu_kernel(const float *__restrict__ x, long n, GeluParams g, float *__restrict__ y) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = gelu_load<GELU>(x[i], g);
}

__global__ void dql_clear_range_kernel(uint32_t *range) {
    if (threadIdx.x < 2) range[threadIdx.x] = 0u;
}

// min and max of zero and `n` values at x, taken by `nthreads` threads of which this one is `tid`
template <int GELU>
__device__ __forceinline__ void dql_scan(const float *__restrict__ x, long n, long tid, long nthreads, int vec_ok, const GeluParams &g, float &mn, float &mx) {
    mn = 0.f, mx = 0.f;
    auto take = [&](float4 v) {
        v = gelu_load4<GELU>(v, g);
        mn = fminf(mn, fminf(fminf(v.x, v.y), fminf(v.z, v.w)));
        mx = fmaxf(mx, fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)));
    };
    long i = tid;
    if (vec_ok) {
        const long n4 = n >> 2;
        const float4 *x4 = reinterpret_cast<const float4 *>(x);
        for (; i + 3 * nthreads < n4; i += 4 * nthreads) {  // four independent loads in flight
            const float4 a = x4[i], b = x4[i + nthreads], c = x4[i + 2 * nthreads], d = x4[i + 3 * nthreads];
            take(a), take(b), take(c), take(d);
        }
        for (; i < n4; i += nthreads) take(x4[i]);
        i = (n4 << 2) + tid;
    }
    for (; i < n; i += nthreads) {
        const float v = gelu_load<GELU>(x[i], g);
        mn = fminf(mn, v);
        mx = fmaxf(mx, v);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        mn = fminf(mn, __shfl_xor(mn, off, 64));
        mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    }
}

template <int GELU>
__global__ void __launch_bounds__(256)
dql_range_kernel(const float *__restrict__ x, long n, uint32_t *__restrict__ range, int vec_ok, int per_block, GeluParams g) {
    float mn, mx;
    dql_scan<GELU>(x, n, (long)blockIdx.x * 256 + threadIdx.x, (long)gridDim.x * 256, vec_ok, g, mn, mx);
    __shared__ float smn[4], smx[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) smn[wave] = mn, smx[wave] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        mn = fminf(fminf(smn[0], smn[1]), fminf(smn[2], smn[3]));
        mx = fmaxf(fmaxf(smx[0], smx[1]), fmaxf(smx[2], smx[3]));
        // -0.0 counts as 0: drop the sign bit
        if (per_block) {  // one {bits(-min), bits(max)} pair per workgroup, joined by the quantize pass
            range[2 * blockIdx.x] = __float_as_uint(-mn) & 0x7fffffffu;
            range[2 * blockIdx.x + 1] = __float_as_uint(mx) & 0x7fffffffu;
        } else {
            atomicMax(&range[0], __float_as_uint(-mn) & 0x7fffffffu);
            atomicMax(&range[1], __float_as_uint(mx) & 0x7fffffffu);
        }
    }
}

__device__ __forceinline__ void dql_params(const uint32_t *range, float &scale, float &zp) {
    const float neg_min = __uint_as_float(range[0]);
    const float mx = __uint_as_float(range[1]);
    // max - min with min = -neg_min; max == min only when both are 0
    const float span = __fadd_rn(mx, neg_min);
    scale = span == 0.f ? 1.f : __fdiv_rn(span, 255.f);
    zp = rintf(fminf(fmaxf(__fdiv_rn(neg_min, scale), 0.f), 255.f));
}

// The codes of four values: sat(rte(v / scale) + zp), packed. `rcp` is 1 / scale where div_by may be used -- a scale within
// 2^-100 .. 2^100, so that the remainders of every quotient that does not round to 0 stay in range -- and 0 where it may not.
// Values beyond 1024 scale, which only a caller's own range lets through, saturate like that one (NaN becomes code 0 either way).
template <bool FAST>
__device__ __forceinline__ uint32_t dql_four_by(float4 v, float scale, float rcp, float zp) {
    const float in[4] = {v.x, v.y, v.z, v.w};
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float q = FAST ? div_by(__builtin_amdgcn_fmed3f(in[j], -1024.f * scale, 1024.f * scale), scale, rcp) : __fdiv_rn(in[j], scale);
        w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_amdgcn_fmed3f(__fadd_rn(rintf(q), zp), 0.f, 255.f), j, w);
    }
    return w;
}
__device__ __forceinline__ uint32_t dql_four(float4 v, float scale, float rcp, float zp) {
    return rcp != 0.f ? dql_four_by<true>(v, scale, rcp, zp) : dql_four_by<false>(v, scale, rcp, zp);
}
__device__ __forceinline__ float dql_rcp(float scale) { return scale >= 0x1p-100f && scale <= 0x1p100f ? __fdiv_rn(1.f, scale) : 0.f; }

// 256 threads join `nparts` {bits(-min), bits(max)} pairs; the maximum of non-negative floats is the maximum of their
// bit patterns
__device__ __forceinline__ void dql_join(const uint32_t *__restrict__ pairs, int nparts, uint32_t (&joined)[2]) {
    __shared__ uint32_t wave_max[4][2];
    uint32_t a = 0, b = 0;
    for (int i = threadIdx.x; i < nparts; i += 256) a = max(a, pairs[2 * i]), b = max(b, pairs[2 * i + 1]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        a = max(a, (uint32_t)__shfl_xor((int)a, off, 64));
        b = max(b, (uint32_t)__shfl_xor((int)b, off, 64));
    }
    if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6][0] = a, wave_max[threadIdx.x >> 6][1] = b;
    __syncthreads();
    joined[0] = max(max(wave_max[0][0], wave_max[1][0]), max(wave_max[2][0], wave_max[3][0]));
    joined[1] = max(max(wave_max[0][1], wave_max[1][1]), max(wave_max[2][1], wave_max[3][1]));
}

// V runs of four values per thread, 1024 values apart, each packed into one 32-bit store where the output allows it; the
// values are asked for before the range pairs are joined
template <int GELU, int V>
__global__ void __launch_bounds__(256)
dql_quantize_kernel(const float *__restrict__ x, long n, const uint32_t *__restrict__ range, int nparts,
                    uint8_t *__restrict__ y, float *__restrict__ scale_out, uint8_t *__restrict__ zp_out, int vec_ok,
                    GeluParams g) {
    const long first = (long)blockIdx.x * (256 * V) + threadIdx.x;   // this thread's first run, counted in runs
    float4 v[V];
#pragma unroll
    for (int u = 0; u < V; u++) {
        const long run = first + 256 * u, base = run << 2;
        v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (vec_ok && base + 4 <= n) {
            v[u] = reinterpret_cast<const float4 *>(x)[run];
        } else {
            if (base < n) v[u].x = x[base];
            if (base + 1 < n) v[u].y = x[base + 1];
            if (base + 2 < n) v[u].z = x[base + 2];
            if (base + 3 < n) v[u].w = x[base + 3];
        }
    }
    float scale, zp;
    if (nparts > 0) {
        uint32_t joined[2];
        dql_join(range, nparts, joined);
        dql_params(joined, scale, zp);
    } else {
        dql_params(range, scale, zp);
    }
    const float rcp = dql_rcp(scale);
    if (first == 0) {
        *scale_out = scale;
        *zp_out = (uint8_t)zp;
    }
#pragma unroll
    for (int u = 0; u < V; u++) {
        const long run = first + 256 * u, base = run << 2;
        const uint32_t w = dql_four(gelu_load4<GELU>(v[u], g), scale, rcp, zp);
        if (vec_ok && base + 4 <= n) {
            reinterpret_cast<uint32_t *>(y)[run] = w;
        } else {
            for (int j = 0; j < 4; j++)
                if (base + j < n) y[base + j] = (uint8_t)(w >> (8 * j));
        }
    }
}

// Few values: every workgroup takes the range of all of them and quantizes its own 4096; what that reads again comes from the
// caches and costs less than a second launch (1.6 us, 2.2 us of the host's time) or telling each other (1.3 us).
template <int GELU>
__global__ void __launch_bounds__(1024)
dql_small_kernel(const float *__restrict__ x, long n, uint8_t *__restrict__ y, float *__restrict__ scale_out, uint8_t *__restrict__ zp_out, GeluParams g) {
    const long run = (long)blockIdx.x * 1024 + threadIdx.x, base = run << 2;
    float4 own = make_float4(0.f, 0.f, 0.f, 0.f);
    if (base + 4 <= n) {
        own = reinterpret_cast<const float4 *>(x)[run];
    } else {
        if (base < n) own.x = x[base];
        if (base + 1 < n) own.y = x[base + 1];
        if (base + 2 < n) own.z = x[base + 2];
    }
    own = gelu_load4<GELU>(own, g);
    float mn, mx;
    if (gridDim.x == 1) {
        mn = fminf(0.f, fminf(fminf(own.x, own.y), fminf(own.z, own.w))), mx = fmaxf(0.f, fmaxf(fmaxf(own.x, own.y), fmaxf(own.z, own.w)));
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            mn = fminf(mn, __shfl_xor(mn, off, 64));
            mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        }
    } else {
        dql_scan<GELU>(x, n, threadIdx.x, 1024, 1, g, mn, mx);
    }
    __shared__ float smn[16], smx[16];
    if ((threadIdx.x & 63) == 0) smn[threadIdx.x >> 6] = mn, smx[threadIdx.x >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 16; w++) mn = fminf(mn, smn[w]), mx = fmaxf(mx, smx[w]);
    const uint32_t joined[2] = {__float_as_uint(-mn) & 0x7fffffffu, __float_as_uint(mx) & 0x7fffffffu};   // (-0.0 counts as 0)
    float scale, zp;
    dql_params(joined, scale, zp);
    if (run == 0) *scale_out = scale, *zp_out = (uint8_t)zp;
    const uint32_t w = dql_four(own, scale, dql_rcp(scale), zp);
    if (base + 4 <= n) {
        reinterpret_cast<uint32_t *>(y)[run] = w;
    } else {
        for (int j = 0; j < 3; j++)
            if (base + j < n) y[base + j] = (uint8_t)(w >> (8 * j));
    }
}

// All of it in one launch, for as many values as the chip's registers hold: 1024 threads keep V runs of four values each, through
// the GELU where there is one, publish the workgroup's range, wait for the ranges of all workgroups and quantize what they hold.
// Every value is read once and every GELU taken once; two launches do both twice. As few runs per thread as 256 workgroups
// allow, since waiting for 256 costs little more than for 64: 1 M values 5.2 us with one run, 5.3, 5.9 and 7.8 with two, four
// and eight. What bounds it: 1 M values the launch, the trip for the values and the two of the hand-over (4.9 us of which 1 us
// is the copy's time), 4 M through a GELU its instructions (4.8 of 9.0 us), 8 M the memory (9.4 us, 4.5 TB/s). Against two
// launches, us: 64 K values 4.6 / 5.2, 1 M 4.9 / 6.1, 4 M 6.3 / 9.2, 8 M 9.4 / 18.2, 16 M 20.3 / 31.3; through a GELU 64 K 5.2 / 6.2,
// 1 M 5.5 / 7.7, 4 M 9.0 / 14.3, 8 M 14.1 / 26.3, 16 M 29.4 / 42.2.
//
// The ranges are published eight times over and each workgroup reads one copy with one wavefront: all 256 workgroups polling
// one copy with four wavefronts each took 8 us for what takes one.
//
// No workgroup depends on the others being on the chip with it. One that has waited long enough says so beside its range and
// leaves, which makes room for one that has not started: of each XCD (to which a launch's workgroups are dealt in turn) the first
// after `ticks`, then two, four, ... more at a time, the last after twice `ticks`, so that about as many leave as are missing.
// Whoever finds all ranges there takes parts of those that left, one at a time. (A workgroup that leaves looks once more after it
// has said so: either it finds all ranges, or the one that publishes last looks for leavers after that, and takes what
// nobody else takes. Both may write the same values; no other order is possible.)
// Calls waited for one by one, beside launches that hold CUs whole, us, two launches / one: 128 CUs for 140 us at a time, 4 M values
// 24 / 21, 8 M 32 / 50, 16 M 45 / 62; 200 CUs, 1 M 19 / 33, 16 M 50 / 140; beside products that fill the chip for 125 us 220 / 110 to
// 124 at any size. (When all left after 50 us and the last workgroup did their parts alone: 16 M beside 64 CUs held 1610.)
//
// A call uses one of two sets of words, empties the other, which nobody reads any more, and then makes that the next call's.
#ifndef HIPC_HOST_MODEL
__device__ __forceinline__ void dql_stored() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }   // this wavefront's stores are where everyone sees them
__device__ __forceinline__ long dql_now() { return (long)wall_clock64(); }
#else   // (threads of the address model run one after the other: nobody waits)
inline void dql_stored() {}
inline long dql_now() { return 0; }
#endif
constexpr uint64_t kThere = 0x80000000ull, kLeft = 0x8000000000000000ull;   // (the sign bits, which a range does not need)
template <int GELU, int V>
__global__ void __launch_bounds__(1024)
dql_once_kernel(const float *__restrict__ x, long n, uint32_t *meet, uint8_t *__restrict__ y, float *__restrict__ scale_out, uint8_t *__restrict__ zp_out, long ticks, GeluParams g) {
    HIPC_PIN_SGPR(ticks);   // (read with the first arguments, not when the waiting begins)
    __shared__ float slow[16], shigh[16];
    __shared__ uint32_t joined[2];
    __shared__ int seen[2];   // all ranges; that some left
    __shared__ uint64_t free_parts[kMeetMax / 64];
    __shared__ int mine_now;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, groups = gridDim.x;
    // the 4096 values of run `r` of a workgroup, four to a thread
    auto load = [&](long r) {
        const float *xr = x + r * 4096;
        const int count = (int)max(min(n - r * 4096, 4096l), 0l), base = 4 * tid;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (__builtin_expect(base + 4 <= count, 1)) {
            v = reinterpret_cast<const float4 *>(xr)[tid];
        } else {
            if (base < count) v.x = xr[base];
            if (base + 1 < count) v.y = xr[base + 1];
            if (base + 2 < count) v.z = xr[base + 2];
        }
        return v;
    };
    auto store = [&](long r, uint32_t w) {
        uint8_t *yr = y + r * 4096;
        const int count = (int)max(min(n - r * 4096, 4096l), 0l), base = 4 * tid;
        if (__builtin_expect(base + 4 <= count, 1)) {
            reinterpret_cast<uint32_t *>(yr)[tid] = w;
        } else {
            for (int j = 0; j < 3; j++)
                if (base + j < count) yr[base + j] = (uint8_t)(w >> (8 * j));
        }
    };
    const long first = (long)blockIdx.x * V;
    float4 v[V];
#pragma unroll
    for (int u = 0; u < V; u++) v[u] = load(first + u);
    const uint32_t set = __builtin_amdgcn_readfirstlane(meet[0]) & 1u;   // (asked for behind the values)
    uint32_t *here = meet + 64 + set * (kMeetSet / 4), *other = meet + 64 + (set ^ 1u) * (kMeetSet / 4);
    float mn = 0.f, mx = 0.f;
#pragma unroll
    for (int u = 0; u < V; u++) {
        v[u] = gelu_load4<GELU>(v[u], g);
        mn = fminf(mn, fminf(fminf(v[u].x, v[u].y), fminf(v[u].z, v[u].w)));
        mx = fmaxf(mx, fmaxf(fmaxf(v[u].x, v[u].y), fmaxf(v[u].z, v[u].w)));
    }
    float low = lean_wave_max(-mn), high = lean_wave_max(mx);
    if (lane == 0) slow[wave] = low, shigh[wave] = high;
    __syncthreads();
    uint64_t *copies = reinterpret_cast<uint64_t *>(here);
    uint32_t *taken = here + 2 * kMeetMax * kMeetCopies;
    uint64_t own = kThere;
    auto publish = [&](uint64_t left) {
        if (tid < kMeetCopies) __hip_atomic_store(copies + tid * kMeetMax + blockIdx.x, own | left, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (wave == 0) dql_stored();
    };
    if (tid < kMeetCopies) {
#pragma unroll
        for (int w = 0; w < 16; w++) low = fmaxf(low, slow[w]), high = fmaxf(high, shigh[w]);
        own |= ((uint64_t)(__float_as_uint(low) & 0x7fffffffu) << 32) | (__float_as_uint(high) & 0x7fffffffu);   // (-0.0 counts as 0)
    }
    publish(0);
    const uint64_t *mine = copies + (blockIdx.x % kMeetCopies) * kMeetMax;
    auto look = [&](long wait) -> bool {   // are all ranges there, within `wait`?
        if (wave == 0) {
            uint64_t pair[kMeetMax / 64];
            bool all, left;
            const long t0 = dql_now();
            for (;;) {
                bool there = true;
                left = false;
#pragma unroll
                for (int q = 0; q < kMeetMax / 64; q++) {
                    pair[q] = kThere;
                    if (lane + 64 * q < groups) pair[q] = __hip_atomic_load(mine + lane + 64 * q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
#pragma unroll
                for (int q = 0; q < kMeetMax / 64; q++) there &= (pair[q] & kThere) != 0, left |= (pair[q] & kLeft) != 0;
                all = __all(there);
                if (all || dql_now() - t0 >= wait) break;
            }
            low = high = 0.f;
#pragma unroll
            for (int q = 0; q < kMeetMax / 64; q++)
                low = fmaxf(low, __uint_as_float((uint32_t)(pair[q] >> 32) & 0x7fffffffu)), high = fmaxf(high, __uint_as_float((uint32_t)pair[q] & 0x7fffffffu));
            low = lean_wave_max(low), high = lean_wave_max(high);
            left = __any(left);
            if (lane == 0) joined[0] = __float_as_uint(low), joined[1] = __float_as_uint(high), seen[0] = all, seen[1] = left;
        }
        __syncthreads();
        return seen[0];
    };
    if (__builtin_expect(!look(ticks + ticks / 5 * (31 - __builtin_clz((blockIdx.x >> 3) + 1))), 0)) {
        __syncthreads();
        publish(kLeft);
        if (!look(0)) return;
    }
    float scale, zp;
    dql_params(joined, scale, zp);
    const float rcp = dql_rcp(scale);
    // workgroup 0, or who does its part, tells the scale and makes the other set the next call's
    auto once = [&] {
        for (int i = tid; i < (int)(kMeetSet / 16); i += 1024) reinterpret_cast<uint4 *>(other)[i] = make_uint4(0, 0, 0, 0);
        if (tid == 0) *meet = set ^ 1u, *scale_out = scale, *zp_out = (uint8_t)zp;
    };
    if (blockIdx.x == 0) once();
#pragma unroll
    for (int u = 0; u < V; u++) store(first + u, dql_four(v[u], scale, rcp, zp));
    if (__builtin_expect(!seen[1], 1)) return;
    for (;;) {   // (every round somebody takes a part: there are no more rounds than parts)
        if (wave < kMeetMax / 64) {
            bool free = false;
            if (tid < groups && tid != (int)blockIdx.x)
                free = (__hip_atomic_load(mine + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kLeft) && !__hip_atomic_load(taken + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint64_t parts = __ballot(free);
            if (lane == 0) free_parts[wave] = parts;
        }
        __syncthreads();
        int count = 0;
#pragma unroll
        for (int q = 0; q < kMeetMax / 64; q++) count += __popcll(free_parts[q]);
        if (count == 0) return;
        // not everyone the same: the workgroup's number modulo how many there are
        int nth = (int)blockIdx.x % count, q = 0;
        while (nth >= __popcll(free_parts[q])) nth -= __popcll(free_parts[q++]);
        uint64_t parts = free_parts[q];
        while (nth-- > 0) parts &= parts - 1;
        const int i = 64 * q + __builtin_ctzll(parts);
        if (tid == 0) mine_now = __hip_atomic_exchange(taken + i, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
        __syncthreads();
        if (!mine_now) continue;
        if (i == 0) once();
#pragma unroll 1
        for (int u = 0; u < V; u++) store((long)i * V + u, dql_four(gelu_load4<GELU>(load((long)i * V + u), g), scale, rcp, zp));
    }
}

__global__ void dql_empty_kernel(float *scale_out, uint8_t *zp_out) {
    if (threadIdx.x == 0) {
        *scale_out = 1.f;
        *zp_out = 0;
    }
}

}  // namespace hipc

using namespace hipc;

namespace {

// `parts`: where the per-workgroup range pairs of a call without a caller-owned slot go (the
// context's own block, or this device's static array)
int dql_launch(hipc_ctx *ctx, const void *X, int64_t n, void *Y, void *scale_out, void *zp_out, void *range, int range_ready,
               const GeluParams &gelu, uint32_t *parts = nullptr) {
    HIPC_REQUIRE(ctx, n >= 0, "DynamicQuantizeLinear: negative length");
    HIPC_REQUIRE(ctx, scale_out && zp_out, "DynamicQuantizeLinear: null scale or zero-point output");
    HIPC_REQUIRE(ctx, aligned(scale_out, 4), "DynamicQuantizeLinear: scale output must be 4-byte aligned");
    if (n == 0) {  // empty input: y empty, scale 1, zero point 0 (interp.rs:1949-1966)
        hipLaunchKernelGGL((dql_empty_kernel), 1, 64, 0, ctx->stream, static_cast<float *>(scale_out), static_cast<uint8_t *>(zp_out));
        HIPC_LAUNCHED(ctx);
        return HIPC_OK;
    }
    HIPC_REQUIRE(ctx, X && Y, "DynamicQuantizeLinear: null tensor");
    HIPC_REQUIRE(ctx, aligned(X, 4), "DynamicQuantizeLinear: input must be 4-byte aligned");
    uint32_t *slot = static_cast<uint32_t *>(range ? range : static_cast<void *>(static_cast<char *>(ctx->params) + kParamRange));
    HIPC_REQUIRE(ctx, aligned(slot, 4), "DynamicQuantizeLinear: range slot must be 4-byte aligned");
    HIPC_REQUIRE(ctx, !(range_ready && !range), "DynamicQuantizeLinear: range_ready needs a caller-owned range slot");
    const int vec_ok = aligned(X, 16) && aligned(Y, 4);
    const float *x = static_cast<const float *>(X);
    auto launch = [&](auto gelu_kind) -> int {
        constexpr int GELU = decltype(gelu_kind)::value;
        if (!range_ready && !range && vec_ok && n <= (GELU ? kSmallGelu : kSmallPlain)) {
            hipLaunchKernelGGL((dql_small_kernel<GELU>), (unsigned)ceil_div(n, 4096), 1024, 0, ctx->stream, x, (long)n, static_cast<uint8_t *>(Y),
                               static_cast<float *>(scale_out), static_cast<uint8_t *>(zp_out), gelu);
            HIPC_LAUNCHED(ctx);
            return HIPC_OK;
        }
        // one launch while a workgroup per CU holds all values (16 runs of four per thread at most: 107 registers of the 128
        // that 1024 threads may have); the forms that must not use the context's memory, and unaligned tensors, keep two
        const int64_t groups = std::min<int64_t>(ctx->cu_count, kMeetMax);
        if (!range_ready && !range && !parts && vec_ok && n <= groups * 16 * 4096 && ctx->tune.dql_wait != 0) {
            const long ticks = ctx->tune.dql_wait > 0 ? ctx->tune.dql_wait : kMeetTicks;
            auto once = [&](auto runs) {
                constexpr int V = decltype(runs)::value;
                hipLaunchKernelGGL((dql_once_kernel<GELU, V>), (unsigned)ceil_div(n, 4096 * V), 1024, 0, ctx->stream, x, (long)n,
                                   reinterpret_cast<uint32_t *>(static_cast<char *>(ctx->params) + kParamMeet), static_cast<uint8_t *>(Y), static_cast<float *>(scale_out),
                                   static_cast<uint8_t *>(zp_out), ticks, gelu);
            };
            if (n <= groups * 4096) once(std::integral_constant<int, 1>{});
            else if (n <= groups * 2 * 4096) once(std::integral_constant<int, 2>{});
            else if (n <= groups * 4 * 4096) once(std::integral_constant<int, 4>{});
            else if (n <= groups * 8 * 4096) once(std::integral_constant<int, 8>{});
            else once(std::integral_constant<int, 16>{});
            HIPC_LAUNCHED(ctx);
            return HIPC_OK;
        }
        int nparts = 0;
        if (!range_ready && !range) {
            // no slot of the caller's to fill: per-workgroup pairs in the context's block, joined by the
            // second pass -- no clearing launch and no atomics
            slot = parts ? parts : reinterpret_cast<uint32_t *>(static_cast<char *>(ctx->params) + kParamParts);
            nparts = (int)std::min<long>(std::max<long>(ceil_div(n, 256 * 16), 1), kParamPartsMax);
            hipLaunchKernelGGL((dql_range_kernel<GELU>), (unsigned)nparts, 256, 0, ctx->stream, x, (long)n, slot, vec_ok, 1, gelu);
            HIPC_LAUNCHED(ctx);
        } else if (!range_ready) {
            hipLaunchKernelGGL((dql_clear_range_kernel), 1, 64, 0, ctx->stream, slot);
            HIPC_LAUNCHED(ctx);
            // enough workgroups to pull from every HBM channel, few enough that the atomics are noise
            const long want = ceil_div(n, 256 * 16);
            const unsigned grid = (unsigned)std::min<long>(std::max<long>(want, 1), 8L * ctx->cu_count);
            hipLaunchKernelGGL((dql_range_kernel<GELU>), grid, 256, 0, ctx->stream, x, (long)n, slot, vec_ok, 0, gelu);
            HIPC_LAUNCHED(ctx);
        }
        // sixteen values per thread where that leaves every SIMD a wavefront: a workgroup joins all the range pairs, a trip
        // to memory of its own (4 M values through a GELU: 13.2 -> 11.0 us); else four
        const long quads = ceil_div(n, 4);
        HIPC_REQUIRE(ctx, ceil_div(quads, 256) < (int64_t(1) << 31), "DynamicQuantizeLinear: tensor too large");
        if (quads >= 4 * 256 * (int64_t)ctx->cu_count)
            hipLaunchKernelGGL((dql_quantize_kernel<GELU, 4>), (unsigned)ceil_div(quads, 4 * 256), 256, 0, ctx->stream, x, (long)n, slot, nparts, static_cast<uint8_t *>(Y),
                               static_cast<float *>(scale_out), static_cast<uint8_t *>(zp_out), vec_ok, gelu);
        else
            hipLaunchKernelGGL((dql_quantize_kernel<GELU, 1>), (unsigned)ceil_div(quads, 256), 256, 0, ctx->stream, x, (long)n, slot, nparts, static_cast<uint8_t *>(Y),
                               static_cast<float *>(scale_out), static_cast<uint8_t *>(zp_out), vec_ok, gelu);
        HIPC_LAUNCHED(ctx);
        return HIPC_OK;
    };
    if (gelu.on == GELU_SQRT2) return launch(std::integral_constant<int, GELU_SQRT2>{});
    if (gelu.on == GELU_ANY) return launch(std::integral_constant<int, GELU_ANY>{});
    return launch(std::integral_constant<int, GELU_OFF>{});
}

int gelu_params(hipc_ctx *ctx, float divisor, float offset, float factor, int factor_first, GeluParams *out) {
    HIPC_REQUIRE(ctx, divisor == divisor && offset == offset && factor == factor && divisor != 0.f, "DecomposedGelu: bad constants");
    *out = GeluParams{divisor == 1.41421356f ? GELU_SQRT2 : GELU_ANY, divisor, offset, factor, factor_first != 0};
    return HIPC_OK;
}

}  // namespace

extern "C" {

int hipc_dynamic_quantize_linear(hipc_ctx *ctx, const void *X, int64_t n, void *Y, void *scale_out, void *zp_out,
                                 void *range, int range_ready) {
    return entry(ctx, [&]() -> int {
        return dql_launch(ctx, X, n, Y, scale_out, zp_out, range, range_ready, GeluParams{});
    });
}

int hipc_dynamic_quantize_linear_static(hipc_ctx *ctx, const void *X, int64_t n, void *Y, void *scale_out, void *zp_out) {
    return entry(ctx, [&]() -> int {
        HIPC_REQUIRE(ctx, n <= HIPC_DQL_STATIC_MAX_N, "DynamicQuantizeLinear (static): %ld elements exceed the limit of %ld", (long)n,
                     (long)HIPC_DQL_STATIC_MAX_N);
        HIPC_REQUIRE(ctx, ctx->dql_static, "DynamicQuantizeLinear (static): the static array was not found on this device");
        // every pair the second pass reads is written by the first pass of this same call, so
        // what an earlier (larger) call left in the array is never seen and nothing needs clearing
        return dql_launch(ctx, X, n, Y, scale_out, zp_out, nullptr, 0, GeluParams{},
                          static_cast<uint32_t *>(ctx->dql_static));
    });
}

int hipc_dynamic_quantize_linear_gelu(hipc_ctx *ctx, const void *X, int64_t n, float divisor, float offset, float factor,
                                      int factor_first, void *Y, void *scale_out, void *zp_out, void *range) {
    return entry(ctx, [&]() -> int {
        GeluParams gp;
        if (int rc = gelu_params(ctx, divisor, offset, factor, factor_first, &gp)) return rc;
        return dql_launch(ctx, X, n, Y, scale_out, zp_out, range, 0, gp);
    });
}

int hipc_decomposed_gelu(hipc_ctx *ctx, const void *X, int64_t n, float divisor, float offset, float factor,
                         int factor_first, void *Y) {
    return entry(ctx, [&]() -> int {
        HIPC_REQUIRE(ctx, n >= 0, "DecomposedGelu: negative length");
        GeluParams gp;
        if (int rc = gelu_params(ctx, divisor, offset, factor, factor_first, &gp)) return rc;
        if (n == 0) return HIPC_OK;
        HIPC_REQUIRE(ctx, X && Y && aligned(X, 4) && aligned(Y, 4), "DecomposedGelu: null or unaligned tensor");
        HIPC_REQUIRE(ctx, ceil_div(n, 256) < (int64_t(1) << 31), "DecomposedGelu: tensor too large");
        if (gp.on == GELU_SQRT2)
            hipLaunchKernelGGL((decomposed_gelu_kernel<GELU_SQRT2>), (unsigned)ceil_div(n, 256), 256, 0, ctx->stream, static_cast<const float *>(X), (long)n, gp, static_cast<float *>(Y));
        else
            hipLaunchKernelGGL((decomposed_gelu_kernel<GELU_ANY>), (unsigned)ceil_div(n, 256), 256, 0, ctx->stream, static_cast<const float *>(X), (long)n, gp, static_cast<float *>(Y));
        HIPC_LAUNCHED(ctx);
        return HIPC_OK;
    });
}

}  // extern "C"
