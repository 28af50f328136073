// Memory-bound uint8 operators for gfx950: add, n-ary eltwise, relu, pooling, quantize, dequantize,
// layout conversion.  Each is a grid-stride wavefront kernel moving 128 bits per lane per access so that
// a wave touches 1 KiB of contiguous HBM per instruction; the integer arithmetic is the reference's
// fixed-point arithmetic, statement for statement (files under art/modules/quant/src/op/).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "common.h"

namespace hipq {

static inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// RN(1 / alpha): the double quotient rounded to fp32 can be one ulp off the correctly rounded reciprocal (double
// rounding); alpha * candidate is exact in a double, so the candidate with the smallest |1 - alpha * y| is it
static float rounded_reciprocal(float alpha)
{
    float rcp = (float)(1.0 / (double)alpha);
    for (float c : {nextafterf(rcp, 0.f), nextafterf(rcp, INFINITY)})
        if (fabs(1.0 - (double)alpha * (double)c) < fabs(1.0 - (double)alpha * (double)rcp))
            rcp = c;
    return rcp;
}

static inline unsigned grid_for(size_t work_items, int per_block = 256)
{
    const size_t b = (work_items + per_block - 1) / per_block;
    return (unsigned)std::min<size_t>(std::max<size_t>(b, 1), 256 * 16);
}

// ---- add (add.c:83-148); arithmetic in common.h ------------------------------------------------
struct AddArgs {
    const uint8_t *a, *b;
    uint8_t *y;
    size_t count;
    AddParams q;
};

template <bool FAST>
__global__ __launch_bounds__(256) void add_u8_kernel(const AddArgs p)
{
    const size_t nvec = p.count / 16;
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x, nthr = (size_t)gridDim.x * blockDim.x;
    for (size_t i = tid; i < nvec; i += nthr) {
        const u32x4 va = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p.a) + i);
        const u32x4 vb = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p.b) + i);
        reinterpret_cast<u32x4 *>(p.y)[i] = add_16<FAST>(va, vb, p.q);
    }
    for (size_t i = nvec * 16 + tid; i < p.count; i += nthr)
        p.y[i] = (uint8_t)add_one_generic(p.a[i], p.b[i], p.q);
}

// ---- n-ary eltwise (eltwise.c:137-271) ---------------------------------------------------------
struct EltArgs {
    const uint8_t *in[HIPQ_MAX_ELTWISE_INPUTS];
    uint32_t mult[HIPQ_MAX_ELTWISE_INPUTS];
    int shift[HIPQ_MAX_ELTWISE_INPUTS]; // shift[n] - s0
    int zp[HIPQ_MAX_ELTWISE_INPUTS];
    int cfast[HIPQ_MAX_ELTWISE_INPUTS]; // fast form: 2^(shift-1) - zp * mult
    int n_in, s0, oz, hi, is_max, fast, cadd;
    uint8_t *y;
    size_t count;
};

// one partial term: input byte x of input n
template <bool FAST>
__device__ static inline int32_t eltwise_term(uint32_t x, int n, const EltArgs &p)
{
    if (FAST) // |mult * (x - zp)| < 2^30 and shift <= 30: 32-bit arithmetic is exact
        return (__mul24((int)x, (int)p.mult[n]) + p.cfast[n]) >> p.shift[n];
    return (int32_t)rshift_rn((int32_t)((uint32_t)((int32_t)x - p.zp[n]) * p.mult[n]), p.shift[n]);
}

template <bool FAST>
__device__ static inline uint32_t eltwise_finish(int32_t t, const EltArgs &p)
{
    if (FAST)
        return (uint32_t)sat_hi((t + p.cadd) >> p.s0, p.hi);
    return (uint32_t)sat_hi((int32_t)(rshift_rn(t, p.s0) + p.oz), p.hi);
}

// NIN inputs and the operation known at compile time (register arrays stay in registers), 16 bytes per thread and input
template <int NIN, bool FAST, bool IS_MAX>
__global__ __launch_bounds__(256) void eltwise_u8_kernel(const EltArgs p)
{
    const size_t nvec = p.count / 16;
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x, nthr = (size_t)gridDim.x * blockDim.x;
    for (size_t i = tid; i < nvec; i += nthr) {
        u32x4 v[NIN];
#pragma unroll
        for (int n = 0; n < NIN; n++)
            v[n] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p.in[n]) + i);
        u32x4 o;
#pragma unroll
        for (int d = 0; d < 4; d++) {
            uint32_t w = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                int32_t t = IS_MAX ? -1 : 0; // the reference's running maximum starts at 0xffffffff (eltwise.c:198)
#pragma unroll
                for (int n = 0; n < NIN; n++) {
                    const int32_t r = eltwise_term<FAST>((v[n][d] >> (8 * e)) & 255, n, p);
                    t = IS_MAX ? (t < r ? r : t) : (int32_t)((uint32_t)t + (uint32_t)r);
                }
                w |= eltwise_finish<FAST>(t, p) << (8 * e);
            }
            o[d] = w;
        }
        reinterpret_cast<u32x4 *>(p.y)[i] = o;
    }
    for (size_t i = nvec * 16 + tid; i < p.count; i += nthr) {
        int32_t t = IS_MAX ? -1 : 0;
#pragma unroll
        for (int n = 0; n < NIN; n++) {
            const int32_t r = eltwise_term<false>(p.in[n][i], n, p);
            t = IS_MAX ? (t < r ? r : t) : (int32_t)((uint32_t)t + (uint32_t)r);
        }
        p.y[i] = (uint8_t)eltwise_finish<false>(t, p);
    }
}

// any number of inputs: one byte position at a time per input, no register arrays
__global__ __launch_bounds__(256) void eltwise_u8_generic_kernel(const EltArgs p)
{
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x, nthr = (size_t)gridDim.x * blockDim.x;
    for (size_t i = tid; i < p.count; i += nthr) {
        int32_t t = p.is_max ? -1 : 0;
        for (int n = 0; n < p.n_in; n++) {
            const int32_t r = eltwise_term<false>(p.in[n][i], n, p);
            t = p.is_max ? (t < r ? r : t) : (int32_t)((uint32_t)t + (uint32_t)r);
        }
        p.y[i] = (uint8_t)eltwise_finish<false>(t, p);
    }
}

// ---- relu (relu.c:76-115) ----------------------------------------------------------------------
struct ReluArgs {
    const uint8_t *x;
    uint8_t *y;
    size_t count;
    uint32_t mult;
    int shift, iz, oz, hi;
};

__device__ static inline uint32_t relu_one(uint32_t x, const ReluArgs &p)
{
    const int32_t v = (int32_t)x >= p.iz ? (int32_t)x : p.iz;
    const uint32_t pr = (uint32_t)(v - p.iz) * p.mult; // evaluated unsigned, widened without sign
    return (uint32_t)sat_hi((int32_t)(rshift_rn((int64_t)pr, p.shift) + p.oz), p.hi);
}

// WORD: shift <= 31.  The multiplier has 23 bits, so difference * mult + 2^(shift - 1) stays below 2^32: one 24-bit
// multiply-add and a shift per byte instead of a 64-bit product (3 instead of 11 vector instructions).  Bytes in and out, 64-bit ->
// 24-bit form: 2 x 1 MB 2.03 -> 1.97 us (a launch), 2 x 10.2 MB 5.55 -> 4.76, 2 x 51.4 MB 19.4 -> 16.6 (6.2 TB/s).
template <bool WORD>
__global__ __launch_bounds__(256) void relu_u8_kernel(const ReluArgs p)
{
    const size_t nvec = p.count / 16;
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x, nthr = (size_t)gridDim.x * blockDim.x;
    const uint32_t radd = WORD ? 1u << (p.shift - 1) : 0;
    for (size_t i = tid; i < nvec; i += nthr) {
        const u32x4 v = reinterpret_cast<const u32x4 *>(p.x)[i];
        u32x4 o;
#pragma unroll
        for (int d = 0; d < 4; d++) {
            uint32_t w = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t x = (v[d] >> (8 * e)) & 255;
                if (WORD) {
                    const uint32_t dx = (uint32_t)(max((int)x, p.iz) - p.iz);
                    w |= (uint32_t)min((int)((__umul24(dx, p.mult) + radd) >> p.shift) + p.oz, p.hi) << (8 * e);
                } else {
                    w |= relu_one(x, p) << (8 * e);
                }
            }
            o[d] = w;
        }
        reinterpret_cast<u32x4 *>(p.y)[i] = o;
    }
    for (size_t i = nvec * 16 + tid; i < p.count; i += nthr)
        p.y[i] = (uint8_t)relu_one(p.x[i], p);
}

// ---- pooling (pool.c:96-249), NHWC: one thread = 4 channels of one output pixel ------------------
struct PoolArgs {
    const uint8_t *x;
    uint8_t *y;
    int N, H, W, OH, OW, cs, kh, kw, ph, pw, sh, sw;
    int is_avg, iz, oz, hi;
    float ia_over_oa; // fp32 ialpha / oalpha, as the reference forms it before dividing by the pool size
    uint32_t mult;    // max pooling: uint16 multiplier
    int shift;
};

// get_quant_scale(x, 16) evaluated on the device with the same fp32 operations (quant_helper.h:98-118)
__device__ static inline void quant_scale16(float x, uint32_t &mult, int &shift)
{
    int s = 0;
    mult = 0;
    shift = 0;
    if (fabs((double)x) < 1e-10)
        return;
    while (x >= 1.0f) {
        x /= 2;
        s -= 1;
    }
    while (x < 0.5f) {
        x *= 2;
        s += 1;
    }
    mult = (uint32_t)(x * 32768.0f);
    shift = s + 15;
}

__global__ __launch_bounds__(256) void pool_u8_kernel(const PoolArgs p)
{
    const int cq = p.cs >> 2;
    const size_t total = (size_t)p.N * p.OH * p.OW * cq;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (size_t)gridDim.x * blockDim.x) {
        const size_t m = idx / cq;
        const int c0 = (int)(idx - m * cq) * 4;
        const int n = (int)(m / ((size_t)p.OH * p.OW)), rem = (int)(m - (size_t)n * p.OH * p.OW);
        const int oh = rem / p.OW, ow = rem - oh * p.OW;
        int hs = oh * p.sh - p.ph, ws = ow * p.sw - p.pw;
        uint32_t o = 0;
        if (!p.is_avg) {
            const int he = min(hs + p.kh, p.H), we = min(ws + p.kw, p.W);
            hs = max(hs, 0), ws = max(ws, 0);
            uint32_t mx[4] = {0, 0, 0, 0};
            for (int i = hs; i < he; i++)
                for (int j = ws; j < we; j++) {
                    const uint32_t v = *reinterpret_cast<const uint32_t *>(
                        p.x + ((size_t)(n * p.H + i) * p.W + j) * p.cs + c0);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        mx[e] = max(mx[e], (v >> (8 * e)) & 255);
                }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int32_t pr = (int32_t)p.mult * ((int32_t)mx[e] - p.iz);
                o |= (uint32_t)sat_hi((int32_t)(rshift_rn(pr, p.shift) + p.oz), p.hi) << (8 * e);
            }
        } else {
            int he = min(hs + p.kh, p.H + p.ph), we = min(ws + p.kw, p.W + p.pw);
            const uint32_t pool_size = (uint32_t)((he - hs) * (we - ws)); // padding counts (pool.c:211-213)
            uint32_t mult;
            int shift;
            quant_scale16(p.ia_over_oa / (float)pool_size, mult, shift);
            hs = max(hs, 0), ws = max(ws, 0), he = min(he, p.H), we = min(we, p.W);
            int32_t sum[4] = {0, 0, 0, 0};
            for (int i = hs; i < he; i++)
                for (int j = ws; j < we; j++) {
                    const uint32_t v = *reinterpret_cast<const uint32_t *>(
                        p.x + ((size_t)(n * p.H + i) * p.W + j) * p.cs + c0);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        sum[e] += (int32_t)((v >> (8 * e)) & 255) - p.iz;
                }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int32_t pr = (int32_t)(mult * (uint32_t)sum[e]);
                o |= (uint32_t)sat_hi((int32_t)(rshift_rn(pr, shift) + p.oz), p.hi) << (8 * e);
            }
        }
        *reinterpret_cast<uint32_t *>(p.y + m * p.cs + c0) = o;
    }
}

// Pooling with a channel stride that is a multiple of 16: a thread owns 16 channels of one output pixel (128-bit
// loads, one 128-bit store), 32-bit index arithmetic.  Maxima and sums are taken on the packed dwords (sums: bytes 0, 2 and
// bytes 1, 3 as two 16-bit halves each; the host guarantees windows of at most 128 pixels).  Average pooling of 8 x 35 x 35 x 192,
// 3x3 / stride 1: 6.75 us with four channels per thread -> 3.64.
// K: windows of 2x2 or 3x3, whose loads are all under way before the first is used (a position outside the image reads a clamped
// one and counts as zeros, which change neither a maximum of bytes nor a sum): maximum at stride 2 5.1 -> 3.2 us, average at stride 1
// 4.8 -> 3.7 at that size; 0: any window, a load's latency after the other.
template <bool AVG, int K>
__global__ __launch_bounds__(256) void pool16_u8_kernel(const PoolArgs p, double inv_c16, double inv_ow, double inv_oh)
{
    const int c16n = p.cs >> 4;
    const int total = p.N * p.OH * p.OW * c16n; // the host guarantees 31 bits
    const bool same = !AVG && p.mult == (1u << p.shift) && p.iz == p.oz && p.hi == 255;
    // work-groups go to the 8 XCDs in turn: renumbered so that each XCD works on a contiguous eighth of the (image-major)
    // index space, the eighth whose pixels its convolution tiles read (the grid is a multiple of 8)
    const int L = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    for (int idx = L * 256 + threadIdx.x; idx < total; idx += gridDim.x * 256) {
        const int m = (int)((double)idx * inv_c16);
        const int mm = m - (m * c16n > idx) + ((m + 1) * c16n <= idx), c0 = (idx - mm * c16n) * 16;
        int row = (int)((double)mm * inv_ow);
        row += ((row + 1) * p.OW <= mm) - (row * p.OW > mm);
        const int ow = mm - row * p.OW;
        int n = (int)((double)row * inv_oh);
        n += ((n + 1) * p.OH <= row) - (n * p.OH > row);
        const int oh = row - n * p.OH;
        const int h0 = oh * p.sh - p.ph, w0 = ow * p.sw - p.pw;
        const int hs = max(h0, 0), ws = max(w0, 0);
        const int he = min(h0 + p.kh, p.H), we = min(w0 + p.kw, p.W);
        u32x4 ev = {0, 0, 0, 0}, od = {0, 0, 0, 0}; // max: the maxima in ev; average: even bytes' and odd bytes' sums
        auto take = [&](const u32x4 &v) {
#pragma unroll
            for (int d = 0; d < 4; d++) {
                if (AVG) {
                    ev[d] += v[d] & 0x00ff00ffu;
                    od[d] += (v[d] >> 8) & 0x00ff00ffu;
                } else {
                    ev[d] = max_u8x4(ev[d], v[d]);
                }
            }
        };
        auto at = [&](int i, int j) { return *reinterpret_cast<const u32x4 *>(p.x + (size_t)((n * p.H + i) * p.W + j) * p.cs + c0); };
        if constexpr (K > 0) {
            u32x4 v[K * K];
#pragma unroll
            for (int i = 0; i < K; i++)
#pragma unroll
                for (int j = 0; j < K; j++)
                    v[i * K + j] = at(min(max(h0 + i, 0), p.H - 1), min(max(w0 + j, 0), p.W - 1));
#pragma unroll
            for (int i = 0; i < K; i++)
#pragma unroll
                for (int j = 0; j < K; j++)
                    take((unsigned)(h0 + i) < (unsigned)p.H && (unsigned)(w0 + j) < (unsigned)p.W ? v[i * K + j] : u32x4{0, 0, 0, 0});
        } else {
            for (int i = hs; i < he; i++)
                for (int j = ws; j < we; j++)
                    take(at(i, j));
        }
        u32x4 o = ev;
        if (!same) { // else equal scales (a multiplier of exactly 2^shift), equal zero points, 8 bits: the maximum is the result
            uint32_t mult = p.mult;
            int shift = p.shift, zsum = p.iz;
            if (AVG) {
                // the divisor counts padding but not what a window hangs over it (pool.c:211-213): one value for all windows
                // but those at the far edges in ceil mode
                const int size = (min(h0 + p.kh, p.H + p.ph) - h0) * (min(w0 + p.kw, p.W + p.pw) - w0);
                if (size != p.kh * p.kw)
                    quant_scale16(p.ia_over_oa / (float)(uint32_t)size, mult, shift);
                zsum = max(he - hs, 0) * max(we - ws, 0) * p.iz;
            }
            const int radd = (1 << (shift - 1)) + (p.oz << shift);
            const int phi = ((p.hi + 1) << shift) - 1; // the largest value that the shift takes to hi
#pragma unroll
            for (int d = 0; d < 4; d++) {
                int32_t v[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t t = !AVG ? (ev[d] >> (8 * e)) & 255 : (((e & 1) ? od[d] : ev[d]) >> (8 * (e & 2))) & 0xffff;
                    // max: mult < 2^16 and 9 bits; average: 15 and 15 bits plus a sign; shift <= 22 (host): 32-bit arithmetic
                    // is exact; the upper clamp in front of the shift, the lower one is the pack's saturation
                    v[e] = min(__mul24((int)mult, (int)t - zsum) + radd, phi);
                }
                o[d] = AVG ? ashr_sat_u8x4_lanes(v[0], v[1], v[2], v[3], shift) : ashr_sat_u8x4(v[0], v[1], v[2], v[3], p.shift);
            }
        }
        *reinterpret_cast<u32x4 *>(p.y + (size_t)mm * p.cs + c0) = o;
    }
}

// Global average pooling (one window = the whole image, no padding) with a channel stride that is a multiple of 16.  A
// work-group of NT threads covers `cpb` (a power of two, 4..64) groups of 16 channels of one image and deals the pixels to its
// NT / cpb thread groups; a thread sums its pixels on packed 16-bit lanes, unpacked every 256 of them, and the partial sums meet in
// LDS in two steps.  What bounds it is one thread's list of pixels (a load latency per four), so the host takes the largest cpb
// that still makes 1024 work-groups and 1024 threads where 256 would leave lists of more than four.  8 x 35 x 35 x 192:
// 150 us with one thread per four channels and image -> 7.2 with 256 threads -> 4.1.  The sums in LDS are loops of a fixed length, so
// that their reads are under way together (ResNet-18 at batch 1, whose last kernels these are: 97.5 -> 96.1 us).
template <int NT>
__global__ __launch_bounds__(NT) void pool_gavg16_u8_kernel(const PoolArgs p, uint32_t mult, int shift, int cpb_log2)
{
    __shared__ int32_t part[NT][17];
    const int c16n = p.cs >> 4, hw = p.H * p.W, tid = threadIdx.x, cpb = 1 << cpb_log2, PG = NT >> cpb_log2;
    const int n = blockIdx.y, chunk = blockIdx.x * cpb + (tid & (cpb - 1)), pg = tid >> cpb_log2;
    int32_t sum[16];
#pragma unroll
    for (int e = 0; e < 16; e++)
        sum[e] = 0;
    if (chunk < c16n) {
        const uint8_t *src = p.x + (size_t)n * hw * p.cs + chunk * 16;
        for (int i0 = pg; i0 < hw; i0 += PG * 256) {
            uint32_t ev[4] = {0, 0, 0, 0}, od[4] = {0, 0, 0, 0};
            const int iend = min(hw, i0 + PG * 256);
#pragma unroll 4
            for (int i = i0; i < iend; i += PG) {
                const u32x4 v = *reinterpret_cast<const u32x4 *>(src + (size_t)i * p.cs);
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    ev[d] += v[d] & 0x00ff00ffu;
                    od[d] += (v[d] >> 8) & 0x00ff00ffu;
                }
            }
#pragma unroll
            for (int d = 0; d < 4; d++) {
                sum[4 * d + 0] += ev[d] & 0xffff, sum[4 * d + 1] += od[d] & 0xffff;
                sum[4 * d + 2] += ev[d] >> 16, sum[4 * d + 3] += od[d] >> 16;
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 16; e++)
        part[tid][e] = sum[e]; // row tid = pg * cpb + chunk
    __syncthreads();
    const int items = cpb * 16; // (chunk, channel) pairs of this work-group
    const int parts = items < NT ? NT / items : 1;
    constexpr int PER = 1024 / NT; // items <= 1024
    int32_t t[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
        t[k] = 0;
        const int it = (tid & (items - 1)) + NT * k;
        const int32_t *from = &part[(tid / items) * cpb + (it >> 4)][it & 15];
        if (items <= NT) { // PG / parts = NT / cpb * items / NT
#pragma unroll
            for (int g = 0; g < 16; g++)
                t[k] += k == 0 ? from[g * parts * cpb * 17] : 0;
        } else if (k * NT < items) {
            for (int g = 0; g < PG; g++)
                t[k] += from[g * cpb * 17];
        }
    }
    if (parts > 1) {
        __syncthreads();
        part[tid >> 4][tid & 15] = t[0];
        __syncthreads();
        t[0] = 0;
        if (tid < items) { // parts: 2 (NT / 128, at the least) to 16
            const int32_t *from = &part[tid >> 4][tid & 15];
#pragma unroll
            for (int g = 0; g < NT / 64; g++)
                t[0] += g < parts ? from[g * cpb * 17] : 0;
        }
    }
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int it = tid + NT * k, c = blockIdx.x * cpb * 16 + it;
        if (it < items && c < p.cs) {
            const int32_t pr = (int32_t)(mult * (uint32_t)(t[k] - hw * p.iz));
            p.y[(size_t)n * p.cs + c] = (uint8_t)sat_hi((int32_t)(rshift_rn(pr, shift) + p.oz), p.hi);
        }
    }
}

// ---- concat along the channels (op_quant_concat_run, concat.c:82-124) ----------------------------------------------
// Output pixel p, channel c comes from input j with off[j] <= c < off[j+1]; every input has its own rescale
// y = sat(rrn(mult_j * (x - zp_j), shift_j) + oz) with a 16-bit multiplier.
// concat16_u8_kernel: a work-group copies one input (blockIdx.y), a thread 16 of its channels: aligned 128-bit loads, stores at
// whatever byte offset the input has in the output, the last piece of a pixel in 8 / 4 / 2 / 1 bytes; parameters are uniform.
// concat_u8_kernel (an input or an output of at most 4 channels, shifts beyond 22): one thread per output dword.
struct ConcatArgs {
    const uint8_t *in[HIPQ_MAX_ELTWISE_INPUTS];
    int off[HIPQ_MAX_ELTWISE_INPUTS + 1]; // first output channel of each input; off[n_in] = total channels
    int cs[HIPQ_MAX_ELTWISE_INPUTS];      // channel stride of each input
    uint32_t mult[HIPQ_MAX_ELTWISE_INPUTS];
    int shift[HIPQ_MAX_ELTWISE_INPUTS];
    int zp[HIPQ_MAX_ELTWISE_INPUTS];
    int n_in, oz, hi, cs_out;
    uint8_t *y;
    size_t npix;
};

__device__ static inline uint32_t concat_one(uint32_t x, int j, const ConcatArgs &p)
{
    const int32_t pr = (int32_t)p.mult[j] * ((int32_t)x - p.zp[j]); // 16-bit * 9-bit
    return (uint32_t)sat_hi((int32_t)(rshift_rn(pr, p.shift[j]) + p.oz), p.hi);
}

__global__ __launch_bounds__(256) void concat_u8_kernel(const ConcatArgs p)
{
    const int cq = p.cs_out >> 2;
    const size_t total = p.npix * cq;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (size_t)gridDim.x * blockDim.x) {
        const size_t pix = idx / cq;
        const int c0 = (int)(idx - pix * cq) * 4;
        uint32_t o = 0;
        int j = 0;
        while (j + 1 < p.n_in && c0 >= p.off[j + 1])
            j++;
        if (c0 + 3 < p.off[j + 1] && ((c0 - p.off[j]) & 3) == 0) {
            const uint32_t v = *reinterpret_cast<const uint32_t *>(p.in[j] + pix * p.cs[j] + (c0 - p.off[j]));
#pragma unroll
            for (int e = 0; e < 4; e++)
                o |= concat_one((v >> (8 * e)) & 255, j, p) << (8 * e);
        } else {
            for (int e = 0; e < 4; e++) {
                const int c = c0 + e;
                if (c >= p.off[p.n_in])
                    break; // pad channels of the output stay zero
                while (c >= p.off[j + 1])
                    j++;
                o |= concat_one(p.in[j][pix * p.cs[j] + (c - p.off[j])], j, p) << (8 * e);
            }
        }
        *reinterpret_cast<uint32_t *>(p.y + pix * p.cs_out + c0) = o;
    }
}

template <class T>
struct __attribute__((packed)) unaligned_t { T v; };
template <class T>
__device__ static inline void store_unaligned(uint8_t *p, T v) { reinterpret_cast<unaligned_t<T> *>(p)->v = v; }

// 8 x 35 x 35, 192 + 100 channels: 4.98 us with a thread per output dword -> 3.08
__global__ __launch_bounds__(256) void concat16_u8_kernel(const ConcatArgs p)
{
    const int j = blockIdx.y, ch = p.off[j + 1] - p.off[j], n16 = p.cs[j] >> 4, tail = ch & 15;
    const int shift = p.shift[j], mult = (int)p.mult[j];
    const int radd = (1 << (shift - 1)) + (p.oz << shift) - p.zp[j] * mult, phi = ((p.hi + 1) << shift) - 1;
    const int pad = j == p.n_in - 1 ? p.cs_out - p.off[p.n_in] : 0; // pad channels of the output are zeros
    const size_t total = p.npix * n16;
    for (size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (size_t)gridDim.x * 256) {
        const size_t pix = (uint32_t)n16 == 1 ? idx : (total >> 32 ? idx / n16 : (uint32_t)idx / (uint32_t)n16);
        const int g = (int)(idx - pix * n16);
        const u32x4 v = *reinterpret_cast<const u32x4 *>(p.in[j] + idx * 16);
        u32x4 o;
#pragma unroll
        for (int d = 0; d < 4; d++) {
            int32_t r[4];
#pragma unroll
            for (int e = 0; e < 4; e++) // 16-bit multiplier * byte and the folded constants below 2^31: exact (shift <= 22)
                r[e] = min(__mul24((int)((v[d] >> (8 * e)) & 255), mult) + radd, phi);
            o[d] = ashr_sat_u8x4(r[0], r[1], r[2], r[3], shift);
        }
        uint8_t *y = p.y + pix * p.cs_out + p.off[j] + g * 16;
        if (tail == 0 || g < n16 - 1) {
            store_unaligned(y, o);
        } else {
            uint32_t w0 = o[0], w1 = o[1]; // the dwords of the piece not stored yet
            if (tail & 8) {
                store_unaligned(y, (uint64_t)w0 | (uint64_t)w1 << 32);
                y += 8, w0 = o[2], w1 = o[3];
            }
            if (tail & 4) {
                store_unaligned(y, w0);
                y += 4, w0 = w1;
            }
            if (tail & 2) {
                store_unaligned(y, (uint16_t)w0);
                y += 2, w0 >>= 16;
            }
            if (tail & 1)
                *y = (uint8_t)w0;
        }
        if (g == n16 - 1)
            for (int c = 0; c < pad; c++)
                p.y[pix * p.cs_out + p.off[p.n_in] + c] = 0;
    }
}

// ---- softmax over the channels (op_quant_softmax_run, softmax.c:89-122) -------------------------------------------
// e(x) = fp32(exp(double(fp32(ialpha * (x - izp))))) takes 256 values: the host tabulates them with the C library's
// exp, the very call the reference makes.  The sum of a pixel is fp32 in channel order (the reference's order), then
// y = saturate_float_by_bits(e / sum / oalpha + ozp) with IEEE fp32 divisions.
// A work-group stages the bytes of `rows` pixels in LDS (coalesced both ways), one thread per pixel walks its channels for the sum -
// that order leaves no other parallelism - and all threads share the divisions, four channels at a time, writing the bytes back in
// place.  A thread per pixel for everything took 31.0 us for 9800 pixels of 81 channels, this 4.6.
struct SoftmaxArgs {
    const uint8_t *x;
    uint8_t *y;
    size_t npix;
    int C, cs;
    float oalpha, ozp, hi;
    float rcp; // RN(1 / oalpha)
    float table[256];
};

static const int SOFTMAX_LDS = 40960; // bytes of staged pixels: three work-groups per CU

// RN(a / b) from rcp = RN(1 / b): once within an ulp, the second correction rounds correctly (Markstein's theorem), where nothing
// underflows or overflows
__device__ static inline float div_by(float a, float b, float rcp)
{
    float q = __fmul_rn(a, rcp);
    q = __fmaf_rn(__fmaf_rn(-b, q, a), rcp, q);
    return __fmaf_rn(__fmaf_rn(-b, q, a), rcp, q);
}

// FAST: the host has checked that every quotient of table values and their sums stays far inside the range of fp32: ten
// multiply-adds instead of two IEEE division sequences of a dozen instructions each.
template <bool FAST>
__device__ static inline uint32_t softmax_byte(float e, float sum, float rsum, const SoftmaxArgs &p)
{
    const float r = FAST ? div_by(div_by(e, sum, rsum), p.oalpha, p.rcp) : __fdiv_rn(__fdiv_rn(e, sum), p.oalpha);
    const float q = __fadd_rn(r, p.ozp);
    // q > hi -> hi; q < 0 -> 0; else trunc(double(q) + 0.5): the integer part plus one if the (exact) fraction is at least a half
    const float c = fminf(fmaxf(q, 0.f), p.hi); // a NaN (0 / 0) becomes 0, as its conversion does
    return (uint32_t)c + (uint32_t)(__builtin_amdgcn_fractf(c) >= 0.5f);
}

// NDW: dwords of a piece (4; 1 for the channel stride of 4)
template <bool FAST, int NDW>
__global__ __launch_bounds__(256) void softmax_u8_kernel(const SoftmaxArgs p, int rows)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ float tab[256], sums[64];
    const int stride = p.cs + 4; // row stride in LDS: the pixels of a wave's lanes fall on different banks
    typedef uint32_t vec_t __attribute__((ext_vector_type(NDW)));
    const int pieces = p.cs / (4 * NDW), tid = threadIdx.x; // of a pixel
    tab[tid] = p.table[tid];
    for (size_t first = (size_t)blockIdx.x * rows; first < p.npix; first += (size_t)gridDim.x * rows) {
        const int live = (int)min((size_t)rows, p.npix - first);
        const int n = live * pieces;
        const vec_t *src = reinterpret_cast<const vec_t *>(p.x + first * p.cs);
        for (int i0 = tid; i0 < n; i0 += 1024) { // four loads in flight per thread
            vec_t v[4];
#pragma unroll
            for (int u = 0; u < 4; u++)
                v[u] = src[min(i0 + 256 * u, n - 1)];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int i = i0 + 256 * u;
                const int r = (int)((unsigned)i / (unsigned)pieces);
                if (i < n)
#pragma unroll
                    for (int d = 0; d < NDW; d++)
                        *reinterpret_cast<uint32_t *>(lds + r * stride + (i - r * pieces) * (4 * NDW) + 4 * d) = v[u][d];
            }
        }
        __syncthreads();
        if (tid < live) {
            const uint8_t *row = lds + tid * stride;
            float sum = 0.f;
            const int whole = p.C & ~15; // in pieces of 16: the next piece's table entries are on their way while this one's are added
            float e[16], f[16];
            auto look_up = [&](int c, float (&t)[16]) {
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const uint32_t v = *reinterpret_cast<const uint32_t *>(row + c + 4 * d);
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        t[4 * d + k] = tab[(v >> (8 * k)) & 255];
                }
            };
            auto add_up = [&](const float (&t)[16]) {
#pragma unroll
                for (int k = 0; k < 16; k++)
                    sum = __fadd_rn(sum, t[k]);
            };
            if (whole)
                look_up(0, e);
            for (int c = 0; c < whole; c += 32) {
                if (c + 16 < whole)
                    look_up(c + 16, f);
                add_up(e);
                if (c + 16 < whole) {
                    if (c + 32 < whole)
                        look_up(c + 32, e);
                    add_up(f);
                }
            }
            for (int c = whole; c < p.C; c++)
                sum = __fadd_rn(sum, tab[row[c]]);
            sums[tid] = sum;
        }
        __syncthreads();
        vec_t *dst = reinterpret_cast<vec_t *>(p.y + first * p.cs);
        for (int i = tid; i < n; i += 256) {
            const int r = (int)((unsigned)i / (unsigned)pieces), c = (i - r * pieces) * (4 * NDW);
            const float sum = sums[r], rsum = FAST ? __fdiv_rn(1.f, sum) : 0.f;
            vec_t o;
#pragma unroll
            for (int d = 0; d < NDW; d++) {
                const uint32_t v = *reinterpret_cast<const uint32_t *>(lds + r * stride + c + 4 * d);
                uint32_t w = 0;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t b = softmax_byte<FAST>(tab[(v >> (8 * k)) & 255], sum, rsum, p);
                    w |= (c + 4 * d + k < p.C ? b : 0u) << (8 * k); // pad channels are zeros
                }
                o[d] = w;
            }
            dst[i] = o;
        }
        __syncthreads();
    }
}

// pixels that do not fit the LDS: a thread per pixel
__global__ __launch_bounds__(256) void softmax_u8_wide_kernel(const SoftmaxArgs p)
{
    __shared__ float tab[256];
    tab[threadIdx.x] = p.table[threadIdx.x];
    __syncthreads();
    for (size_t pix = (size_t)blockIdx.x * blockDim.x + threadIdx.x; pix < p.npix; pix += (size_t)gridDim.x * blockDim.x) {
        const uint8_t *xr = p.x + pix * p.cs;
        uint8_t *yr = p.y + pix * p.cs;
        float sum = 0.f;
        for (int c = 0; c < p.C; c++)
            sum = __fadd_rn(sum, tab[xr[c]]);
        for (int c = 0; c < p.C; c++)
            yr[c] = (uint8_t)softmax_byte<false>(tab[xr[c]], sum, 0.f, p);
        for (int c = p.C; c < p.cs; c++)
            yr[c] = 0;
    }
}

// ---- quantize (quantize.c:145-157): fp32 NCHW -> uint8 NHWC --------------------------------------
// One thread produces the 4 channels of one dword of the output; reads are coalesced along W per
// channel plane, writes along the pixel index.
struct QuantArgs {
    const float *x;
    uint8_t *y;
    int N, C, H, W, cs;
    float alpha, beta, hi;
    float rcp, xlo, xhi; // uint8 variant: RN(1 / alpha) and the clamp of x - beta, [-alpha, (hi + 1) * alpha]
    int lim; // int8 variant: alpha holds fp32(1 / oalpha), the result is clipped to +-lim
};

// The reference: q = fp32((x - beta) / alpha); q > hi -> hi; q < 0 -> 0 (NaN too: the x86 conversion of NaN is 0 in
// the low byte); else trunc(double(q) + 0.5).  Here, value for value the same byte with a third of the instructions of
// the IEEE division sequence:
//   * x - beta is clamped to [-alpha, (hi + 1) * alpha] first: outside that range the quotient is below 0 or above hi
//     anyway, inside it nothing changes, and no infinity reaches the steps below (a NaN leaves v_med3_f32 as the
//     smallest of the other two operands, i.e. as a negative quotient: 0, like the reference);
//   * the correctly rounded quotient from the correctly rounded reciprocal rcp = RN(1 / alpha) (the host computes it):
//     q0 = RN(a * rcp), then twice r = a - alpha * q (exact in an FMA), q = RN(q + r * rcp).  After the first
//     correction q is within an ulp of a / alpha, and then the second yields RN(a / alpha) (Markstein's theorem on
//     division with a correctly rounded reciprocal; no overflow by the clamp, and an underflowing residual belongs to
//     a quotient far below 0.5, whose byte is 0 whatever its last bits are);
//   * trunc(q + 0.5) for 0 <= q <= hi + 1 without the double: the integer part plus one if the fraction (exact in
//     fp32) is at least a half.
__device__ static inline uint32_t quantize_one(float x, const QuantArgs &p)
{
    float a = __fsub_rn(x, p.beta);
    asm("v_med3_f32 %0, %1, %2, %3" : "=v"(a) : "v"(a), "v"(p.xlo), "v"(p.xhi));
    float q = __fmul_rn(a, p.rcp);
    q = __fmaf_rn(__fmaf_rn(-p.alpha, q, a), p.rcp, q);
    q = __fmaf_rn(__fmaf_rn(-p.alpha, q, a), p.rcp, q);
    q = fmaxf(q, 0.f);
    const uint32_t r = (uint32_t)q + (uint32_t)(__builtin_amdgcn_fractf(q) >= 0.5f);
    return min(r, (uint32_t)p.hi);
}

// op_quantize_run_i8 (quantize.c:159-185): clip(round(x * fp32(1 / oalpha)), -lim, lim).  The product is fp32, round()
// is the C library's on a double (half away from zero), and clip() takes an int: the reference's x86-64 conversion
// turns everything outside int32 (and NaN) into INT32_MIN, which then clips to -lim.
__device__ static inline uint32_t quantize_one_i8(float x, const QuantArgs &p)
{
    const double r = round((double)__fmul_rn(x, p.alpha));
    const int v = (r >= -2147483648.0 && r < 2147483648.0) ? (int)r : INT32_MIN;
    return (uint32_t)min(max(v, -p.lim), p.lim) & 255u;
}

template <bool SIGNED>
__device__ static inline uint32_t quantize_any(float x, const QuantArgs &p)
{
    return SIGNED ? quantize_one_i8(x, p) : quantize_one(x, p);
}

template <bool SIGNED>
__global__ __launch_bounds__(256) void quantize_u8_kernel(const QuantArgs p)
{
    const int cq = p.cs >> 2;
    const size_t hw = (size_t)p.H * p.W, total = (size_t)p.N * hw * cq;
    // pixel index fastest across threads: each channel plane is read with unit stride
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (size_t)gridDim.x * blockDim.x) {
        const size_t pix = idx % hw, rest = idx / hw;
        const int q4 = (int)(rest % cq), n = (int)(rest / cq);
        uint32_t o = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int c = q4 * 4 + e;
            if (c < p.C)
                o |= quantize_any<SIGNED>(p.x[((size_t)n * p.C + c) * hw + pix], p) << (8 * e);
        }
        *reinterpret_cast<uint32_t *>(p.y + ((size_t)n * hw + pix) * p.cs + q4 * 4) = o;
    }
}

// Network inputs (C <= 4, channel stride 4): a thread converts 4 consecutive pixels, i.e. one 128-bit load per
// channel plane and one 128-bit store; blockIdx.y is the image, so no 64-bit index arithmetic is needed.  The vectors are
// only 4-byte aligned - that is where the planes of an image with an odd number of pixels begin, and aligned addresses pay
// nothing for it - and the last 1..3 pixels of such an image go one by one.
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

template <bool SIGNED>
__global__ __launch_bounds__(256) void quantize_u8_c4_kernel(const QuantArgs p)
{
    const int hw = p.H * p.W, hw4 = hw >> 2;
    const int n = blockIdx.y;
    const float *xn = p.x + (size_t)n * p.C * hw;
    uint32_t *yn = reinterpret_cast<uint32_t *>(p.y) + (size_t)n * hw;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < hw4; i += gridDim.x * 256) {
        u32x4 o = {0, 0, 0, 0};
        for (int c = 0; c < p.C; c++) { // one plane at a time: with every plane's load issued first the kernel is a third slower
            const f32x4_a4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4_a4 *>(xn + (size_t)c * hw) + i);
#pragma unroll
            for (int e = 0; e < 4; e++)
                o[e] |= quantize_any<SIGNED>(v[e], p) << (8 * c);
        }
        *(reinterpret_cast<u32x4_a4 *>(yn) + i) = o;
    }
    const int last = hw4 * 4 + threadIdx.x;
    if (blockIdx.x == 0 && last < hw) {
        uint32_t o = 0;
        for (int c = 0; c < p.C; c++)
            o |= quantize_any<SIGNED>(xn[(size_t)c * hw + last], p) << (8 * c);
        yn[last] = o;
    }
}

// More channels (stride a multiple of 16): a thread converts 16 channels (blockIdx.z) of one pixel; the 64 lanes of a wave read
// 64 consecutive pixels of a plane per load and every lane writes one 128-bit piece.  The grid covers the whole stride: pieces of
// pad channels alone are written as zeros.
template <bool SIGNED>
__global__ __launch_bounds__(256) void quantize_u8_c16_kernel(const QuantArgs p)
{
    const int hw = p.H * p.W, n = blockIdx.y, c0 = blockIdx.z * 16;
    const int last = p.C - 1 - c0; // channels beyond it read plane C - 1 again and store zeros: no load waits for a branch
    const float *xn = p.x + (size_t)n * p.C * hw;
    uint8_t *yn = p.y + (size_t)n * hw * p.cs + c0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < hw; i += gridDim.x * 256) {
        float v[16];
#pragma unroll
        for (int c = 0; c < 16; c++)
            v[c] = xn[(size_t)min(c0 + c, p.C - 1) * hw + i];
        u32x4 o = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 16; c++)
            o[c >> 2] |= (c <= last ? quantize_any<SIGNED>(v[c], p) : 0u) << (8 * (c & 3));
        *reinterpret_cast<u32x4 *>(yn + (size_t)i * p.cs) = o;
    }
}

// ---- dequantize (dequantize.c:111-123): uint8 NHWC -> fp32 NCHW ----------------------------------
struct DequantArgs {
    const uint8_t *x;
    float *y;
    int N, C, H, W, cs;
    float alpha;
    int zp;
    int sgn; // 1: the bytes are int8 and there is no zero point (op_dequantize_run_i8, dequantize.c:125-136)
};

__global__ __launch_bounds__(256) void dequantize_u8_kernel(const DequantArgs p)
{
    const size_t hw = (size_t)p.H * p.W, total = (size_t)p.N * p.C * hw;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (size_t)gridDim.x * blockDim.x) {
        const size_t pix = idx % hw, rest = idx / hw;
        const int c = (int)(rest % p.C), n = (int)(rest / p.C);
        const uint8_t b = p.x[((size_t)n * hw + pix) * p.cs + c];
        const int v = p.sgn ? (int)(int8_t)b : (int)b - p.zp;
        p.y[idx] = __fmul_rn((float)v, p.alpha);
    }
}

// Images: a thread converts VEC channels (16, or the 4 of a network input; blockIdx.z) of one pixel with one load; the 64 lanes
// of a wave write 64 consecutive pixels of a plane per store.  The loop over single bytes above reads every line VEC
// times over and divides twice per value: 64 x 21 x 56 x 56 took 11.8 us, this 4.6.
template <int VEC>
__global__ __launch_bounds__(256) void dequantize_planes_kernel(const DequantArgs p)
{
    typedef uint32_t vec_t __attribute__((ext_vector_type(VEC / 4)));
    const int hw = p.H * p.W, n = blockIdx.y, c0 = blockIdx.z * VEC;
    const uint8_t *xn = p.x + (size_t)n * hw * p.cs + c0;
    float *yn = p.y + ((size_t)n * p.C + c0) * hw;
    const int flip = p.sgn ? 0x80 : 0; // int8: byte ^ 0x80 minus 128 is its value
    const float zp = (float)(p.sgn ? 128 : p.zp);
    for (int i = blockIdx.x * 256 + threadIdx.x; i < hw; i += gridDim.x * 256) {
        const vec_t v = *reinterpret_cast<const vec_t *>(xn + (size_t)i * p.cs) ^ (uint32_t)(flip * 0x01010101);
#pragma unroll
        for (int c = 0; c < VEC; c++)
            if (c0 + c < p.C) // small whole numbers: their difference is exact in fp32, the product is the one rounding
                yn[(size_t)c * hw + i] = __fmul_rn(__fsub_rn((float)((v[c >> 2] >> (8 * (c & 3))) & 255), zp), p.alpha);
    }
}

// int32 accumulators (NHWC, as hipq_conv2d_run's acc_out writes them) -> fp32 dense NCHW: (float)acc * alpha
struct DequantI32Args {
    const int32_t *x;
    float *y;
    int N, C, H, W, cs;
    float alpha;
};

__global__ __launch_bounds__(256) void dequantize_i32_kernel(const DequantI32Args p)
{
    const size_t hw = (size_t)p.H * p.W, total = (size_t)p.N * p.C * hw;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (size_t)gridDim.x * blockDim.x) {
        const size_t pix = idx % hw, rest = idx / hw;
        const int c = (int)(rest % p.C), n = (int)(rest / p.C);
        p.y[idx] = __fmul_rn(__int2float_rn(p.x[((size_t)n * hw + pix) * p.cs + c]), p.alpha);
    }
}

// ---- layout conversion ---------------------------------------------------------------------------
struct LayoutArgs {
    const uint8_t *src;
    uint8_t *dst;
    int N, C, H, W, cs;
};

__global__ __launch_bounds__(256) void nchw_to_nhwc_kernel(const LayoutArgs p)
{
    const int cq = p.cs >> 2;
    const size_t hw = (size_t)p.H * p.W, total = (size_t)p.N * hw * cq;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (size_t)gridDim.x * blockDim.x) {
        const size_t pix = idx % hw, rest = idx / hw;
        const int q4 = (int)(rest % cq), n = (int)(rest / cq);
        uint32_t o = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int c = q4 * 4 + e;
            if (c < p.C)
                o |= (uint32_t)p.src[((size_t)n * p.C + c) * hw + pix] << (8 * e);
        }
        *reinterpret_cast<uint32_t *>(p.dst + ((size_t)n * hw + pix) * p.cs + q4 * 4) = o;
    }
}

// Network inputs (C <= 4, channel stride 4): a thread converts 4 consecutive pixels - one dword per plane, a byte transpose,
// one 128-bit store - and the last 1..3 pixels of an image go one by one; the planes are read at any alignment.
struct __attribute__((packed)) u32_a1 { uint32_t v; };

__global__ __launch_bounds__(256) void nchw_to_nhwc_c4_kernel(const LayoutArgs p)
{
    const int hw = p.H * p.W, hw4 = hw >> 2, n = blockIdx.y;
    const uint8_t *src = p.src + (size_t)n * p.C * hw;
    uint32_t *dst = reinterpret_cast<uint32_t *>(p.dst) + (size_t)n * hw;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < hw4; i += gridDim.x * 256) {
        uint32_t v[4] = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (c < p.C)
                v[c] = reinterpret_cast<const u32_a1 *>(src + (size_t)c * hw + i * 4)->v;
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++)
            o[e] = ((v[0] >> (8 * e)) & 255) | ((v[1] >> (8 * e)) & 255) << 8 | ((v[2] >> (8 * e)) & 255) << 16 | (v[3] >> (8 * e)) << 24;
        *(reinterpret_cast<u32x4_a4 *>(dst) + i) = o;
    }
    const int last = hw4 * 4 + threadIdx.x;
    if (blockIdx.x == 0 && last < hw) {
        uint32_t o = 0;
        for (int c = 0; c < p.C; c++)
            o |= (uint32_t)src[(size_t)c * hw + last] << (8 * c);
        dst[last] = o;
    }
}

__global__ __launch_bounds__(256) void nhwc_to_nchw_kernel(const LayoutArgs p)
{
    const size_t hw = (size_t)p.H * p.W, total = (size_t)p.N * p.C * hw;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (size_t)gridDim.x * blockDim.x) {
        const size_t pix = idx % hw, rest = idx / hw;
        const int c = (int)(rest % p.C), n = (int)(rest / p.C);
        p.dst[idx] = p.src[((size_t)n * hw + pix) * p.cs + c];
    }
}

__global__ __launch_bounds__(256) void copy_bytes_kernel(const u32x4 *src, u32x4 *dst, size_t nvec)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nvec; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

} // namespace hipq

// =================================================================================================
using namespace hipq;

extern "C" int hipq_add_u8(const void *a, const void *b, void *y, size_t count, float ia0, int iz0, float ia1,
                           int iz1, float oa, int oz, int obits, void *stream)
{
    clear_error();
    HIPQ_REQUIRE(a && b && y, "hipq_add_u8: null pointer");
    HIPQ_REQUIRE(aligned16(a) && aligned16(b) && aligned16(y), "hipq_add_u8: buffers must be 16-byte aligned");
    if (count == 0)
        return 0;
    AddArgs p;
    HIPQ_REQUIRE(make_add_params(ia0, iz0, ia1, iz1, oa, oz, obits, &p.q),
                 "hipq_add_u8: scales out of the fixed-point range");
    p.a = static_cast<const uint8_t *>(a), p.b = static_cast<const uint8_t *>(b), p.y = static_cast<uint8_t *>(y);
    p.count = count;
    const dim3 grid(grid_for(count / 16)), block(256);
    if (p.q.fast)
        hipLaunchKernelGGL(add_u8_kernel<true>, grid, block, 0, static_cast<hipStream_t>(stream), p);
    else
        hipLaunchKernelGGL(add_u8_kernel<false>, grid, block, 0, static_cast<hipStream_t>(stream), p);
    return launch_status("add_u8_kernel");
}

extern "C" int hipq_eltwise_u8(const void *const *in, int n_in, const float *coeff, const float *ialpha,
                               const uint8_t *izp, void *y, size_t count, int operation, float oa, int oz,
                               int obits, void *stream)
{
    clear_error();
    HIPQ_REQUIRE(in && ialpha && izp && y && aligned16(y), "hipq_eltwise_u8: null pointer or output not 16-byte aligned");
    HIPQ_REQUIRE(n_in >= 2 && n_in <= HIPQ_MAX_ELTWISE_INPUTS, "hipq_eltwise_u8: %d inputs (2..%d supported)", n_in,
                 HIPQ_MAX_ELTWISE_INPUTS);
    HIPQ_REQUIRE(operation == HIPQ_ELTWISE_SUM || operation == HIPQ_ELTWISE_MAX,
                 "hipq_eltwise_u8: operation %d is not implemented (PROD is rejected by the reference too)", operation);
    if (count == 0)
        return 0;
    EltArgs p;
    memset(&p, 0, sizeof p);
    int smin = 127, sh[HIPQ_MAX_ELTWISE_INPUTS];
    for (int n = 0; n < n_in; n++) {
        HIPQ_REQUIRE(in[n] && aligned16(in[n]), "hipq_eltwise_u8: input %d is null or not 16-byte aligned", n);
        hipq_quant_scale((coeff ? coeff[n] : 1.0f) * ialpha[n] / oa, 23, &p.mult[n], &sh[n]);
        smin = std::min(smin, sh[n]);
        p.in[n] = static_cast<const uint8_t *>(in[n]);
        p.zp[n] = izp[n];
    }
    p.s0 = smin - 1;
    HIPQ_REQUIRE(valid_shift(p.s0), "hipq_eltwise_u8: scales out of the fixed-point range");
    for (int n = 0; n < n_in; n++) {
        p.shift[n] = sh[n] - p.s0;
        HIPQ_REQUIRE(valid_shift(p.shift[n]), "hipq_eltwise_u8: scales out of the fixed-point range");
    }
    p.n_in = n_in, p.oz = oz, p.hi = (1 << obits) - 1, p.is_max = operation == HIPQ_ELTWISE_MAX;
    p.y = static_cast<uint8_t *>(y), p.count = count;
    // 32-bit form: every product below 2^30 (22-bit multipliers), shifts within a word, the sum of n terms and
    // the folded rounding / zero-point constant without overflow
    p.fast = p.s0 <= 20 && n_in <= 4;
    for (int n = 0; n < n_in; n++) {
        p.fast = p.fast && p.shift[n] <= 30 && p.mult[n] < (1u << 23) && (reinterpret_cast<uintptr_t>(in[n]) & 15) == 0;
        p.cfast[n] = p.fast ? (1 << (p.shift[n] - 1)) - p.zp[n] * (int32_t)p.mult[n] : 0;
    }
    p.fast = p.fast && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
    p.cadd = p.fast ? (1 << (p.s0 - 1)) + (oz << p.s0) : 0;
    const dim3 grid(grid_for(count / 16 + 1)), block(256);
    hipStream_t st = static_cast<hipStream_t>(stream);
#define HIPQ_ELT(NIN)                                                                          \
    if (p.fast && p.is_max)                                                                    \
        hipLaunchKernelGGL((eltwise_u8_kernel<NIN, true, true>), grid, block, 0, st, p);       \
    else if (p.fast)                                                                           \
        hipLaunchKernelGGL((eltwise_u8_kernel<NIN, true, false>), grid, block, 0, st, p);      \
    else if (p.is_max)                                                                         \
        hipLaunchKernelGGL((eltwise_u8_kernel<NIN, false, true>), grid, block, 0, st, p);      \
    else                                                                                       \
        hipLaunchKernelGGL((eltwise_u8_kernel<NIN, false, false>), grid, block, 0, st, p)
    if (n_in == 2) {
        HIPQ_ELT(2);
    } else if (n_in == 3) {
        HIPQ_ELT(3);
    } else if (n_in == 4) {
        HIPQ_ELT(4);
    } else {
        hipLaunchKernelGGL(eltwise_u8_generic_kernel, dim3(grid_for(count)), block, 0, st, p);
    }
#undef HIPQ_ELT
    return launch_status("eltwise_u8_kernel");
}

extern "C" int hipq_relu_u8(const void *x, void *y, size_t count, float ia, int iz, float oa, int oz, int obits,
                            void *stream)
{
    clear_error();
    HIPQ_REQUIRE(x && y && aligned16(x) && aligned16(y), "hipq_relu_u8: null or unaligned pointer");
    if (count == 0)
        return 0;
    ReluArgs p;
    hipq_quant_scale(ia / oa, 24, &p.mult, &p.shift);
    HIPQ_REQUIRE(valid_shift(p.shift), "hipq_relu_u8: scale out of the fixed-point range");
    p.x = static_cast<const uint8_t *>(x), p.y = static_cast<uint8_t *>(y), p.count = count;
    p.iz = iz, p.oz = oz, p.hi = (1 << obits) - 1;
    if (p.shift <= 31)
        hipLaunchKernelGGL(relu_u8_kernel<true>, dim3(grid_for(count / 16)), dim3(256), 0, static_cast<hipStream_t>(stream), p);
    else
        hipLaunchKernelGGL(relu_u8_kernel<false>, dim3(grid_for(count / 16)), dim3(256), 0, static_cast<hipStream_t>(stream), p);
    return launch_status("relu_u8_kernel");
}

extern "C" int hipq_concat_u8(const void *const *in, int n_in, const int *channels, const float *ialpha, const uint8_t *izp,
                              void *y, size_t npix, float oa, int oz, int obits, void *stream)
{
    clear_error();
    HIPQ_REQUIRE(in && channels && ialpha && izp && y, "hipq_concat_u8: null pointer");
    HIPQ_REQUIRE(n_in >= 2 && n_in <= HIPQ_MAX_ELTWISE_INPUTS, "hipq_concat_u8: %d inputs (2..%d supported)", n_in,
                 HIPQ_MAX_ELTWISE_INPUTS);
    HIPQ_REQUIRE(obits >= 1 && obits <= 8, "hipq_concat_u8: obits must be in 1..8");
    if (npix == 0)
        return 0;
    ConcatArgs p;
    memset(&p, 0, sizeof p);
    for (int j = 0; j < n_in; j++) {
        HIPQ_REQUIRE(in[j] && channels[j] > 0, "hipq_concat_u8: input %d is null or has no channels", j);
        p.in[j] = static_cast<const uint8_t *>(in[j]);
        p.off[j + 1] = p.off[j] + channels[j];
        p.cs[j] = hipq_channel_stride(channels[j]);
        hipq_quant_scale(ialpha[j] / oa, 16, &p.mult[j], &p.shift[j]); // concat.c:104-108
        p.mult[j] &= 0xffff;
        HIPQ_REQUIRE(valid_shift(p.shift[j]), "hipq_concat_u8: scale of input %d out of the fixed-point range", j);
        p.zp[j] = izp[j];
    }
    p.n_in = n_in, p.oz = oz, p.hi = (1 << obits) - 1, p.cs_out = hipq_channel_stride(p.off[n_in]);
    p.y = static_cast<uint8_t *>(y), p.npix = npix;
    bool vec16 = p.cs_out % 16 == 0;
    size_t most = 0;
    for (int j = 0; j < n_in; j++) {
        vec16 = vec16 && p.cs[j] % 16 == 0 && p.shift[j] <= 22 && aligned16(in[j]);
        most = std::max(most, npix * (p.cs[j] / 16));
    }
    if (vec16) {
        hipLaunchKernelGGL(concat16_u8_kernel, dim3(grid_for(most), n_in), dim3(256), 0, static_cast<hipStream_t>(stream), p);
        return launch_status("concat16_u8_kernel");
    }
    hipLaunchKernelGGL(concat_u8_kernel, dim3(grid_for(npix * (p.cs_out / 4))), dim3(256), 0, static_cast<hipStream_t>(stream), p);
    return launch_status("concat_u8_kernel");
}

extern "C" int hipq_softmax_u8(const void *x, void *y, size_t npix, int C, int cs, float ia, int iz, float oa, int oz, int obits,
                               void *stream)
{
    clear_error();
    HIPQ_REQUIRE(x && y && C > 0 && cs >= C, "hipq_softmax_u8: bad argument");
    HIPQ_REQUIRE(obits >= 1 && obits <= 8, "hipq_softmax_u8: obits must be in 1..8");
    if (npix == 0)
        return 0;
    SoftmaxArgs p;
    p.x = static_cast<const uint8_t *>(x), p.y = static_cast<uint8_t *>(y), p.npix = npix, p.C = C, p.cs = cs;
    p.oalpha = oa, p.ozp = (float)oz, p.hi = (float)((1 << obits) - 1);
    // The table follows from the operator's scale and zero point alone.  256 calls of exp are 3 us of a 4 us launch: each
    // thread keeps the table of the last pair it saw (1 KB).
    static thread_local struct { float ia; int iz; bool set; float table[256], least, most; } last;
    if (!last.set || last.ia != ia || last.iz != iz) {
        for (int v = 0; v < 256; v++) {
            const float arg = ia * (float)(v - iz);        // softmax.c:112: an fp32 product ...
            last.table[v] = (float)std::exp((double)arg);  // ... passed to the double exp, stored as fp32
        }
        last.least = *std::min_element(last.table, last.table + 256), last.most = *std::max_element(last.table, last.table + 256);
        last.ia = ia, last.iz = iz, last.set = true;
    }
    memcpy(p.table, last.table, sizeof p.table);
    // pixels per work-group: as many as a wave can sum at once, fewer where the LDS or the number of pixels asks for it (four
    // work-groups per CU before a work-group takes more pixels)
    const int rows = (int)std::min<size_t>(std::min(64, SOFTMAX_LDS / (cs + 4)), std::max<size_t>(4, (npix + 1023) / 1024));
    const uintptr_t both = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y);
    if (rows >= 1 && ((cs % 16 == 0 && both % 16 == 0) || (cs == 4 && both % 4 == 0))) {
        const dim3 grid((unsigned)std::min<size_t>((npix + rows - 1) / rows, 256 * 16)), block(256);
        const size_t bytes = (size_t)rows * (cs + 4);
        const hipStream_t st = static_cast<hipStream_t>(stream);
        const bool fast = last.least >= 1e-20f && last.most <= 1e20f && (double)last.most * C / last.least <= 1e25 && oa >= 1e-10f
            && oa <= 1e10f;
        p.rcp = rounded_reciprocal(oa);
        if (cs == 4)
            hipLaunchKernelGGL((softmax_u8_kernel<false, 1>), grid, block, bytes, st, p, rows);
        else if (fast)
            hipLaunchKernelGGL((softmax_u8_kernel<true, 4>), grid, block, bytes, st, p, rows);
        else
            hipLaunchKernelGGL((softmax_u8_kernel<false, 4>), grid, block, bytes, st, p, rows);
        return launch_status("softmax_u8_kernel");
    }
    hipLaunchKernelGGL(softmax_u8_wide_kernel, dim3(grid_for(npix)), dim3(256), 0, static_cast<hipStream_t>(stream), p);
    return launch_status("softmax_u8_wide_kernel");
}

template <bool AVG>
static void launch_pool16(const PoolArgs &p, unsigned grid, hipStream_t st)
{
    const double c16 = 1.0 / (p.cs / 16), ow = 1.0 / p.OW, oh = 1.0 / p.OH;
    if (p.kh == 3 && p.kw == 3)
        hipLaunchKernelGGL((pool16_u8_kernel<AVG, 3>), dim3(grid), dim3(256), 0, st, p, c16, ow, oh);
    else if (p.kh == 2 && p.kw == 2)
        hipLaunchKernelGGL((pool16_u8_kernel<AVG, 2>), dim3(grid), dim3(256), 0, st, p, c16, ow, oh);
    else
        hipLaunchKernelGGL((pool16_u8_kernel<AVG, 0>), dim3(grid), dim3(256), 0, st, p, c16, ow, oh);
}

extern "C" int hipq_pool_u8(const void *x, void *y, int N, int C, int H, int W, int OH, int OW, int cs, int kh, int kw,
                            int ph, int pw, int sh, int sw, int method, float ia, int iz, float oa, int oz, int obits,
                            void *stream)
{
    clear_error();
    HIPQ_REQUIRE(x && y, "hipq_pool_u8: null pointer");
    HIPQ_REQUIRE(N > 0 && C > 0 && H > 0 && W > 0 && OH > 0 && OW > 0 && cs >= C && cs % 4 == 0, "hipq_pool_u8: bad shape");
    HIPQ_REQUIRE(kh > 0 && kw > 0 && sh > 0 && sw > 0 && ph >= 0 && pw >= 0, "hipq_pool_u8: bad window");
    // every window must overlap the padded image, otherwise the reference divides by a pool size <= 0
    HIPQ_REQUIRE((OH - 1) * sh - ph < H + ph && (OW - 1) * sw - pw < W + pw, "hipq_pool_u8: a window lies outside the image");
    PoolArgs p;
    p.x = static_cast<const uint8_t *>(x), p.y = static_cast<uint8_t *>(y);
    p.N = N, p.H = H, p.W = W, p.OH = OH, p.OW = OW, p.cs = cs, p.kh = kh, p.kw = kw, p.ph = ph, p.pw = pw, p.sh = sh, p.sw = sw;
    p.is_avg = method != HIPQ_POOL_MAX, p.iz = iz, p.oz = oz, p.hi = (1 << obits) - 1;
    p.ia_over_oa = ia / oa;
    hipq_quant_scale(ia / oa, 16, &p.mult, &p.shift);
    p.mult &= 0xffff; // get_quant_scale_int16 stores the multiplier in a uint16_t
    HIPQ_REQUIRE(valid_shift(p.shift), "hipq_pool_u8: scale out of the fixed-point range");
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const bool vec16 = cs % 16 == 0 && aligned16(x) && aligned16(y);
    if (p.is_avg && OH == 1 && OW == 1 && ph == 0 && pw == 0 && kh >= H && kw >= W && vec16 && N <= 65535) {
        uint32_t mult;
        int shift;
        hipq_quant_scale(p.ia_over_oa / (float)(uint32_t)(H * W), 16, &mult, &shift); // pool.c:211-216
        if (valid_shift(shift)) {
            int lg = 6;
            while (lg > 2 && (long long)N * ((cs / 16 + (1 << lg) - 1) >> lg) < 1024)
                lg--;
            const dim3 grid((cs / 16 + (1 << lg) - 1) >> lg, N);
            if ((long long)H * W > 4 * (256 >> lg))
                hipLaunchKernelGGL(pool_gavg16_u8_kernel<1024>, grid, dim3(1024), 0, st, p, mult, shift, lg);
            else
                hipLaunchKernelGGL(pool_gavg16_u8_kernel<256>, grid, dim3(256), 0, st, p, mult, shift, lg);
            return launch_status("pool_gavg16_u8_kernel");
        }
    }
    if (vec16 && (long long)N * OH * OW * (cs / 16) < (1ll << 31) && (long long)N * H * W < (1ll << 31)) {
        const unsigned grid = (grid_for((size_t)N * OH * OW * (cs / 16)) + 7) / 8 * 8;
        if (!p.is_avg && p.shift <= 22) {
            launch_pool16<false>(p, grid, st);
            return launch_status("pool16_u8_kernel");
        }
        PoolArgs q = p; // average: the multiplier of a whole window; p.shift is that of the smallest one, a single pixel
        hipq_quant_scale(p.ia_over_oa / (float)(uint32_t)(kh * kw), 16, &q.mult, &q.shift);
        if (p.is_avg && (long long)kh * kw <= 128 && p.shift >= 1 && q.shift >= 1 && q.shift <= 22) {
            launch_pool16<true>(q, grid, st);
            return launch_status("pool16_u8_kernel");
        }
    }
    const size_t total = (size_t)N * OH * OW * (cs / 4);
    hipLaunchKernelGGL(pool_u8_kernel, dim3(grid_for(total)), dim3(256), 0, st, p);
    return launch_status("pool_u8_kernel");
}

// Is a conversion between planes and pixels worth a wave per 64 pixels?  Below half a wave of pixels the kernels that walk the
// channels fastest read and write better (a classifier's [N, C, 1, 1] is the same order on both sides).
static bool image16(size_t hw, int N, int cs)
{
    return cs % 16 == 0 && hw >= 32 && hw < (1u << 30) && N <= 65535 && cs / 16 <= 65535;
}

static int launch_quantize(const char *who, bool sgn, const float *x, void *y, int N, int C, int H, int W, int cs, float oa,
                           int oz, int obits, void *stream)
{
    clear_error();
    HIPQ_REQUIRE(x && y && N > 0 && C > 0 && H > 0 && W > 0 && cs >= C && cs % 4 == 0, "%s: bad argument", who);
    HIPQ_REQUIRE(obits >= 1 && obits <= 8, "%s: obits must be in 1..8", who);
    HIPQ_REQUIRE(oa >= 1e-30f && oa <= 1e30f, "%s: the scale must be a positive number between 1e-30 and 1e30", who);
    QuantArgs p;
    p.x = x, p.y = static_cast<uint8_t *>(y), p.N = N, p.C = C, p.H = H, p.W = W, p.cs = cs;
    p.alpha = sgn ? (float)(1. / (double)oa) : oa; // quantize.c:166: a double division, rounded to fp32
    p.beta = -(oa * (float)oz);                    // quantize.c:152
    p.hi = (float)((1 << obits) - 1);
    p.lim = (1 << (obits - 1)) - 1;
    p.rcp = rounded_reciprocal(oa);
    p.xlo = -oa, p.xhi = (p.hi + 1.f) * oa;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const size_t hw = (size_t)H * W;
    if (cs == 4 && hw < (1u << 30) && N <= 65535) {
        const unsigned bx = (unsigned)std::min<size_t>((hw / 4 + 255) / 256 + (hw < 4), 1024);
        if (sgn)
            hipLaunchKernelGGL(quantize_u8_c4_kernel<true>, dim3(bx, N), dim3(256), 0, st, p);
        else
            hipLaunchKernelGGL(quantize_u8_c4_kernel<false>, dim3(bx, N), dim3(256), 0, st, p);
        return launch_status(sgn ? "quantize_i8_c4_kernel" : "quantize_u8_c4_kernel");
    }
    if (image16(hw, N, cs) && aligned16(y)) {
        const dim3 grid((unsigned)std::min<size_t>((hw + 255) / 256, 1024), N, cs / 16);
        if (sgn)
            hipLaunchKernelGGL(quantize_u8_c16_kernel<true>, grid, dim3(256), 0, st, p);
        else
            hipLaunchKernelGGL(quantize_u8_c16_kernel<false>, grid, dim3(256), 0, st, p);
        return launch_status(sgn ? "quantize_i8_c16_kernel" : "quantize_u8_c16_kernel");
    }
    const size_t total = (size_t)N * H * W * (cs / 4);
    if (sgn)
        hipLaunchKernelGGL(quantize_u8_kernel<true>, dim3(grid_for(total)), dim3(256), 0, st, p);
    else
        hipLaunchKernelGGL(quantize_u8_kernel<false>, dim3(grid_for(total)), dim3(256), 0, st, p);
    return launch_status(sgn ? "quantize_i8_kernel" : "quantize_u8_kernel");
}

extern "C" int hipq_quantize_u8(const float *x, void *y, int N, int C, int H, int W, int cs, float oa, int oz, int obits,
                                void *stream)
{
    return launch_quantize("hipq_quantize_u8", false, x, y, N, C, H, W, cs, oa, oz, obits, stream);
}

extern "C" int hipq_quantize_i8(const float *x, void *y, int N, int C, int H, int W, int cs, float oa, int obits, void *stream)
{
    return launch_quantize("hipq_quantize_i8", true, x, y, N, C, H, W, cs, oa, 0, obits, stream);
}

static int launch_dequantize(const char *who, int sgn, const void *x, float *y, int N, int C, int H, int W, int cs, float ia,
                             int iz, void *stream)
{
    clear_error();
    HIPQ_REQUIRE(x && y && N > 0 && C > 0 && H > 0 && W > 0 && cs >= C, "%s: bad argument", who);
    DequantArgs p;
    p.x = static_cast<const uint8_t *>(x), p.y = y, p.N = N, p.C = C, p.H = H, p.W = W, p.cs = cs, p.alpha = ia, p.zp = iz;
    p.sgn = sgn;
    const size_t hw = (size_t)H * W;
    if (image16(hw, N, cs) && aligned16(x)) {
        hipLaunchKernelGGL(dequantize_planes_kernel<16>, dim3((unsigned)std::min<size_t>((hw + 255) / 256, 1024), N, (C + 15) / 16), dim3(256),
                           0, static_cast<hipStream_t>(stream), p);
        return launch_status("dequantize_planes_kernel");
    }
    if (cs == 4 && hw >= 32 && hw < (1u << 30) && N <= 65535 && (reinterpret_cast<uintptr_t>(x) & 3) == 0) {
        hipLaunchKernelGGL(dequantize_planes_kernel<4>, dim3((unsigned)std::min<size_t>((hw + 255) / 256, 1024), N), dim3(256), 0,
                           static_cast<hipStream_t>(stream), p);
        return launch_status("dequantize_planes_kernel");
    }
    hipLaunchKernelGGL(dequantize_u8_kernel, dim3(grid_for((size_t)N * C * H * W)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), p);
    return launch_status(sgn ? "dequantize_i8_kernel" : "dequantize_u8_kernel");
}

extern "C" int hipq_dequantize_u8(const void *x, float *y, int N, int C, int H, int W, int cs, float ia, int iz,
                                  void *stream)
{
    return launch_dequantize("hipq_dequantize_u8", 0, x, y, N, C, H, W, cs, ia, iz, stream);
}

extern "C" int hipq_dequantize_i8(const void *x, float *y, int N, int C, int H, int W, int cs, float ia, void *stream)
{
    return launch_dequantize("hipq_dequantize_i8", 1, x, y, N, C, H, W, cs, ia, 0, stream);
}

extern "C" int hipq_dequantize_i32(const int32_t *x, float *y, int N, int C, int H, int W, int cs, float alpha, void *stream)
{
    clear_error();
    HIPQ_REQUIRE(x && y && N > 0 && C > 0 && H > 0 && W > 0 && cs >= C, "hipq_dequantize_i32: bad argument");
    DequantI32Args p;
    p.x = x, p.y = y, p.N = N, p.C = C, p.H = H, p.W = W, p.cs = cs, p.alpha = alpha;
    hipLaunchKernelGGL(dequantize_i32_kernel, dim3(grid_for((size_t)N * C * H * W)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), p);
    return launch_status("dequantize_i32_kernel");
}

static int layout_args(LayoutArgs &p, const void *src, void *dst, int N, int C, int H, int W, int cs)
{
    HIPQ_REQUIRE(src && dst && N > 0 && C > 0 && H > 0 && W > 0 && cs >= C && cs % 4 == 0, "layout conversion: bad argument");
    p.src = static_cast<const uint8_t *>(src), p.dst = static_cast<uint8_t *>(dst);
    p.N = N, p.C = C, p.H = H, p.W = W, p.cs = cs;
    return 0;
}

extern "C" int hipq_nchw_to_nhwc_u8(const void *src, void *dst, int N, int C, int H, int W, int cs, void *stream)
{
    clear_error();
    LayoutArgs p;
    if (int rc = layout_args(p, src, dst, N, C, H, W, cs))
        return rc;
    const size_t hw = (size_t)H * W;
    if (cs == 4 && hw < (1u << 30) && N <= 65535) {
        hipLaunchKernelGGL(nchw_to_nhwc_c4_kernel, dim3((unsigned)std::min<size_t>((hw / 4 + 255) / 256 + (hw < 4), 1024), N), dim3(256), 0,
                           static_cast<hipStream_t>(stream), p);
        return launch_status("nchw_to_nhwc_c4_kernel");
    }
    hipLaunchKernelGGL(nchw_to_nhwc_kernel, dim3(grid_for((size_t)N * H * W * (cs / 4))), dim3(256), 0,
                       static_cast<hipStream_t>(stream), p);
    return launch_status("nchw_to_nhwc_kernel");
}

extern "C" int hipq_nhwc_to_nchw_u8(const void *src, void *dst, int N, int C, int H, int W, int cs, void *stream)
{
    clear_error();
    LayoutArgs p;
    if (int rc = layout_args(p, src, dst, N, C, H, W, cs))
        return rc;
    hipLaunchKernelGGL(nhwc_to_nchw_kernel, dim3(grid_for((size_t)N * C * H * W)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), p);
    return launch_status("nhwc_to_nchw_kernel");
}

extern "C" int hipq_copy_bytes(const void *src, void *dst, size_t count, void *stream)
{
    clear_error();
    HIPQ_REQUIRE(src && dst && aligned16(src) && aligned16(dst) && count % 16 == 0, "hipq_copy_bytes: need 16-byte granularity");
    hipLaunchKernelGGL(copy_bytes_kernel, dim3(grid_for(count / 16)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const u32x4 *>(src), static_cast<u32x4 *>(dst), count / 16);
    return launch_status("copy_bytes_kernel");
}
