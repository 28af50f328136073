// A depthwise 3x3 convolution, the 1x1 convolution that reads it and, where there is one, the residual add in ONE kernel: what is
// left of an inverted residual block that has no expanding layer (the first of a mobile network) or whose expanding layer has too
// much to do to be computed again at every patch's border (the last ones, 576 to 960 channels on 7x7).  gfx950 only.
//
// Reproduces, bit for bit, op_conv_2d_u8xu8_run (art/modules/quant/src/op/conv_2d_uint8_impl.c:39-165) twice and op_quant_add_run
// (art/modules/quant/src/op/add.c:83-148): the depthwise output is requantised and clamped exactly as if it had travelled through
// memory.
//
// Why: the tensor in between is written and read once, and on small images either layer is a launch that waits for memory once and
// computes next to nothing.  A wave takes a slice of 32 channels of a patch of output pixels: its input region -> LDS, re-centred; the
// depthwise layer as nine diagonal matrices (conv_dw_frag.h); its requantised sums are, as they lie in the lanes, one k-step of
// the 1x1 layer.  The next slice's region is on its way meanwhile.
// The waves of a work-group split the channels of one patch and add their partial sums up in LDS, or, where there are many patches and
// one slice, every wave has patches of its own.  Output channel tiles are divided into groups: each group computes the depthwise
// layer again, which costs less than idle CUs, and spreads a 7x7 image over more CUs.
// What bounds it: many patches of few channels - memory and vector issue (the requantisations: 45 % of a CU's busy time at 4 clocks an
// instruction, matrix cores 14 %); few pixels of many channels - the chain launch, region, slices, sum, in which a CU's vector units (28
// to 34 %) and matrix cores (7 to 8 %) take turns and mostly wait.
// Measured, the two launches -> this one (back to back, three sets of tensors in turn): 32 -> 16 channels at 112x112, 64 images: 24.6 -> 15.7
// us (38 MB of input and output), 1 image: 5.6 -> 3.4; 64 -> 128 at 56x56, stride 2, 1 image: 6.5 -> 3.8; 192 -> 64 at 28x28, stride 2,
// 6 images: 5.8 -> 4.3; 960 -> 160 at 7x7, 64 images: 10.0 -> 8.3, 1 image: 6.0 -> 6.3 (the rule takes it for a tie).  A shared patch's
// biases, residual and the place where its sums meet are ready before them: 1.1 to 1.4 times as fast as with the three in the chain (960 ->
// 320, 64 images, 11.2 -> 9.4).
// Requirements (checked by the host): uint8 tensors, weight zero points 128, per-tensor scales, one-multiply requantisations.
#include "conv_dwpoint.h"

#include <algorithm>
#include <cmath>

#include "conv_dw_frag.h"

namespace hipq {

using namespace frag;

namespace {

// S: stride, PH x 8: output pixels of a patch; rows, columns and positions of the input region; PT: pixel tiles of 32 outputs; NR: pieces
// of 16 bytes of a slice's region that a lane brings
template <int S, int PH_>
struct PairPatch {
    static constexpr int PH = PH_, PW = 8, RH = S * (PH - 1) + 3, RW = S * (PW - 1) + 3, NP = RH * RW, PT = PH / 4, NR = (2 * NP + 63) / 64;
    static constexpr int BYTES = NR * 1024; // a wave's buffer
};

// waves of a work-group that shares a patch: as many as the accumulators leave registers for
constexpr int max_waves(int PT, int CT) { return PT * CT == 1 ? 16 : PT * CT <= 3 ? 12 : 8; }

struct PairGeom {
    int PY, PX; // patches per image
    int nT;     // slices of 32 channels
    int ct;     // tiles of 32 output channels
    int groups; // of output channel tiles, a work-group each
    int nw;     // waves
    int red;    // where a shared patch's sums lie in LDS
    int ppi, items, per_xcd;         // patches of an image, work-groups, those of an XCD
    uint32_t m_groups, m_ppi, m_px;  // x / groups, x / ppi and x / PX (hipq_div_magic)
    int s_groups, s_ppi, s_px;
};

// x / d for any x below 2^31 (hipq_div_magic)
__device__ static __forceinline__ int quot(int x, uint32_t m, int s) { return m ? (int)(__umulhi((uint32_t)x, m) >> s) : x; }

} // namespace

template <int S, int PH, int CT>
__global__ __launch_bounds__(64 * max_waves(PH / 4, CT)) void conv_dwpoint_kernel(const ConvArgs d, const ConvArgs pr, const PairGeom geo)
{
    using G = PairPatch<S, PH>;
    constexpr int PW = G::PW, RW = G::RW, NP = G::NP, PT = G::PT, NR = G::NR;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = geo.nw;
    const int p = lane & 31, h = lane >> 5;
    const int ch = slice_channel(p);
    // work-groups go to the 8 XCDs in turn: XCD x takes the x-th contiguous eighth of the work, the groups of a patch side by side.
    // (Eighths of the patches with all their groups left XCDs idle where patches are few: 18 patches in 13 groups took 7.0 us, two
    // rounds of work-groups on six XCDs, against 4.5.)
    const int item = (int)(blockIdx.x % 8) * geo.per_xcd + (int)(blockIdx.x / 8);
    if (item >= geo.items)
        return;
    const int gid = quot(item, geo.m_groups, geo.s_groups);
    const int n = quot(gid, geo.m_ppi, geo.s_ppi), pi = gid - n * geo.ppi, py = quot(pi, geo.m_px, geo.s_px);
    const int oy0 = py * PH, ox0 = (pi - py * geo.PX) * PW;
    const int iy0 = S * oy0 - 1, ix0 = S * ox0 - 1; // the region's first row and column
    const int ct0 = (item - gid * geo.groups) * CT;
    uint8_t *const buf = lds + wave * G::BYTES;

    // ---- the pieces of a region that this lane brings: 16 channels of a position each, where in the image (clamped), and whether it is in it
    uint32_t from[NR];
    uint32_t valid = 0;
    const int epad = (int)(d.padword ^ 0x80808080u);
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const int pos = min((lane + 64 * i) >> 1, NP - 1), ry = pos / RW, iy = iy0 + ry, ix = ix0 + pos - ry * RW;
        const bool in = ((unsigned)iy < (unsigned)d.H) & ((unsigned)ix < (unsigned)d.W);
        valid |= in ? 1u << i : 0u;
        from[i] = (uint32_t)(((n * d.H + min(max(iy, 0), d.H - 1)) * d.W + min(max(ix, 0), d.W - 1)) * d.in_cs);
    }

    // ---- a slice's pixels, weights and constants, each loaded as soon as the slice before has used its own
    v4i x[NR], wp[CT];
    v16i dbias; // the folded biases of the lane's 16 consecutive channels
    int wd[3];  // the depthwise weights of the channel that this lane's row stands for, a kernel row each
    auto load_x = [&](int T) {
        const int c = min(32 * T + 16 * (lane & 1), d.in_cs - 16); // the last slice may be half empty; its products meet zero weights
#pragma unroll
        for (int i = 0; i < NR; i++)
            x[i] = ldg128(d.x + (from[i] + (uint32_t)c));
    };
    auto load_d = [&](int T) {
        init_acc(dbias, d.bias2 + min(32 * T + 16 * h, d.in_cs - 16), false);
        const int *wt = reinterpret_cast<const int *>(d.wpack) + min(32 * T + ch, d.in_cs - 1);
#pragma unroll
        for (int r = 0; r < 3; r++)
            wd[r] = wt[r * 2 * d.in_cs];
    };
    auto load_p = [&](int T) {
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
            wp[ct] = ldg128(pr.wfrag1 + ((size_t)((T >> 1) * (pr.kout_pad >> 5) + min(ct0 + ct, geo.ct - 1)) * 2 + (T & 1)) * 1024 + lane * 16);
    };
    int T = wave; // never more waves than slices
    load_x(T);
    load_d(T);
    load_p(T);
    // the sums, from the folded bias of the lane's 16 consecutive channels in the first wave; what is here does not wait for the loads
    v16i acc[CT][PT];
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int t = 0; t < PT; t++) {
            if (wave == 0)
                init_acc(acc[ct][t], pr.bias2 + 32 * min(ct0 + ct, geo.ct - 1) + 16 * h, false);
            else
                acc[ct][t] = v16i{};
        }
    int32_t *const red = reinterpret_cast<int32_t *>(lds + geo.red);
    for (int i = threadIdx.x; i < CT * PT * 256; i += 64 * nw)
        reinterpret_cast<v4i *>(red)[i] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NR; i++)
        if (!(valid >> i & 1)) // the same byte in every slice
            *reinterpret_cast<v4i *>(buf + (lane + 64 * i) * 16) = v4i{epad, epad, epad, epad};
    const DiagonalTap taps(lane);
    int first[PT]; // the lane's outputs 32 t + p: their first tap in the region
#pragma unroll
    for (int t = 0; t < PT; t++)
        first[t] = (S * (4 * t + (p >> 3)) * RW + S * (p & 7)) * 32 + 16 * h;
    // The sums have to be zero before the first is added to.  Up to six waves wait for that here, where their loads are under way; more
    // reach this point one prologue after the other, and wait behind their slices, where they meet anyway (16 slices at stride 2, one image,
    // 6.8 us here and 6.4 there; 12 slices 5.9 and 5.6; 5 slices 5.0 and 5.1)
    const bool early = nw <= 6;
    auto sums_ready = [&]() {
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
    };
    if (early)
        sums_ready();

    while (true) {
        const bool more = T + nw < geo.nT;
        T += nw;
#pragma unroll
        for (int i = 0; i < NR; i++)
            if (valid >> i & 1)
                *reinterpret_cast<v4i *>(buf + (lane + 64 * i) * 16) = x[i] ^ (int)0x80808080;
        if (more)
            load_x(T);
        lds_order();
        v16i o[PT];
#pragma unroll
        for (int t = 0; t < PT; t++)
            o[t] = dbias;
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int s = 0; s < 3; s++) {
                const v4i m = taps.matrix(wd[r], s);
#pragma unroll
                for (int t = 0; t < PT; t++)
                    o[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(m, *reinterpret_cast<const v4i *>(buf + first[t] + (r * RW + s) * 32), o[t], 0, 0, 0);
            }
        if (more)
            load_d(T);
#pragma unroll
        for (int t = 0; t < PT; t++) {
            const v4i b = requant_centred(d, o[t]);
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
                acc[ct][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wp[ct], b, acc[ct][t], 0, 0, 0);
        }
        if (!more)
            break;
        load_p(T);
        lds_order();
    }

    // ---- the waves' partial sums meet in LDS; a wave's output tile, i, is the one it takes first: its residual is under way meanwhile
    auto place = [&](int i, uint32_t *at) { // of the lane's 16 channels of its pixel
        const int ct = i / PT, oy = oy0 + 4 * (i - ct * PT) + (p >> 3), ox = ox0 + (p & 7), c0 = 32 * (ct0 + ct) + 16 * h;
        *at = (uint32_t)(((n * pr.OH + oy) * pr.OW + ox) * pr.out_cs + c0); // below 2^31
        return (i < CT * PT) & (oy < pr.OH) & (ox < pr.OW) & (c0 < pr.out_cs);
    };
    uint32_t at;
    bool in = place(wave, &at);
    v4i res = {0, 0, 0, 0};
    if (in && pr.res != nullptr)
        res = ldg128(pr.res + at);
    if (!early)
        sums_ready();
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int t = 0; t < PT; t++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                atomicAdd(&red[((ct * PT + t) * 16 + r) * 64 + lane], acc[ct][t][r]);
    __syncthreads();
    for (int i = wave; i < CT * PT; i += nw) {
        if (i != wave) {
            in = place(i, &at);
            if (in && pr.res != nullptr)
                res = ldg128(pr.res + at);
        }
        v16i s;
#pragma unroll
        for (int r = 0; r < 16; r++)
            s[r] = red[(i * 16 + r) * 64 + lane];
        if (in)
            *reinterpret_cast<v4i *>(pr.y + at) = pr.res != nullptr ? requant_add16(pr, s, res) : requant16(pr, s, 0);
    }
}

// The same for one slice of channels: a wave takes patch after patch, with all weights in registers (the nine diagonal matrices too)
// and the next patch's region on its way.  PACK: 16 output channels would leave half of a multiply's rows empty; the second half of
// the patch takes them, so that one accumulator holds 64 pixels.
template <int S, int PH, int CT, bool PACK>
__global__ __launch_bounds__(256) void conv_dwpoint_narrow_kernel(const ConvArgs d, const ConvArgs pr, const PairGeom geo)
{
    using G = PairPatch<S, PH>;
    constexpr int PW = G::PW, RH = G::RH, RW = G::RW, NP = G::NP, PT = G::PT, NR = G::NR;
    static_assert(!PACK || (PT == 2 && CT == 1));
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p = lane & 31, h = lane >> 5;
    const int ct0 = blockIdx.y * CT;
    uint8_t *const buf = lds + wave * G::BYTES + lane * 16;

    // work-groups go to the 8 XCDs in turn: XCD x takes the x-th contiguous eighth of the patches, its waves side by side
    const int ppi = geo.PY * geo.PX, all = ppi * d.N, part = (all + 7) / 8, xcd = (int)(blockIdx.x % 8);
    int at = xcd * part + (int)(blockIdx.x / 8) * 4 + wave;
    const int end = min(all, (xcd + 1) * part);
    if (at >= end)
        return;
    int n = at / ppi, py = (at - n * ppi) / geo.PX, px = at - n * ppi - py * geo.PX;
    const int step = (int)(gridDim.x / 8) * 4;

    // ---- the pieces of a region that this lane brings: 16 channels of a position each
    int piece[NR], row[NR], col[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const int pos = min((lane + 64 * i) >> 1, NP - 1);
        row[i] = pos / RW, col[i] = pos - row[i] * RW;
        piece[i] = (row[i] * d.W + col[i]) * d.in_cs + min(16 * (lane & 1), d.in_cs - 16);
    }
    const int epad = (int)(d.padword ^ 0x80808080u);
    v4i x[NR];
    uint32_t valid; // bit i: piece i lies in the image
    auto load_x = [&]() {
        const int iy0 = S * PH * py - 1, ix0 = S * PW * px - 1; // the region's first row and column
        const int base = ((n * d.H + iy0) * d.W + ix0) * d.in_cs;
        valid = ~0u;
        if (iy0 >= 0 && ix0 >= 0 && iy0 + RH <= d.H && ix0 + RW <= d.W) {
#pragma unroll
            for (int i = 0; i < NR; i++)
                x[i] = ldg128(d.x + base + (uint32_t)piece[i]);
        } else {
            valid = 0;
#pragma unroll
            for (int i = 0; i < NR; i++) {
                const bool in = (unsigned)(iy0 + row[i]) < (unsigned)d.H && (unsigned)(ix0 + col[i]) < (unsigned)d.W;
                valid |= in ? 1u << i : 0u;
                x[i] = ldg128(d.x + (uint32_t)(in ? base + piece[i] : 0));
            }
        }
    };
    load_x();

    v16i dbias, pbias[CT]; // folded biases of the lane's 16 consecutive channels
    v4i diag[9], wp[CT];
    {
        const int *wt = reinterpret_cast<const int *>(d.wpack) + min(slice_channel(p), d.in_cs - 1);
        const DiagonalTap taps(lane);
#pragma unroll
        for (int r = 0; r < 3; r++) {
            const int w = wt[r * 2 * d.in_cs];
#pragma unroll
            for (int s = 0; s < 3; s++)
                diag[3 * r + s] = taps.matrix(w, s);
        }
    }
    init_acc(dbias, d.bias2 + min(16 * h, d.in_cs - 16), false);
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int c = min(ct0 + ct, geo.ct - 1);
        init_acc(pbias[ct], pr.bias2 + 32 * c + (PACK ? 0 : 16 * h), false);
        wp[ct] = ldg128(pr.wfrag1 + (size_t)c * 2048 + lane * 16);
    }
    v4i wq = {}; // PACK: the rows' other half
    if (PACK)
        wq = ldg128(pr.wfrag1 + (lane ^ 4) * 16);
    uint8_t *const rows = lds + wave * G::BYTES + (S * (p >> 3) * RW + S * (p & 7)) * 32 + 16 * h;
    int to[CT]; // where the lane's first output lies from the patch's
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
        to[ct] = ((p >> 3) * pr.OW + (p & 7)) * pr.out_cs + (PACK ? 4 * h * pr.OW * pr.out_cs : 32 * (ct0 + ct) + 16 * h);

    while (true) {
        const int m = n, oy0 = py * PH, ox0 = px * PW;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            v4i v = x[i] ^ (int)0x80808080;
            if (valid != ~0u && !(valid >> i & 1))
                v = v4i{epad, epad, epad, epad};
            *reinterpret_cast<v4i *>(buf + i * 1024) = v;
        }
        at += step;
        if (at < end) {
            px += step; // the next patch of this wave
            if (px >= geo.PX) {
                const int rows_on = px / geo.PX;
                px -= rows_on * geo.PX, py += rows_on;
                if (py >= geo.PY) {
                    const int images_on = py / geo.PY;
                    py -= images_on * geo.PY, n += images_on;
                }
            }
            load_x();
        }
        lds_order();
        v16i o[PT];
#pragma unroll
        for (int t = 0; t < PT; t++)
            o[t] = dbias;
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int s = 0; s < 3; s++)
#pragma unroll
                for (int t = 0; t < PT; t++)
                    o[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(diag[3 * r + s], *reinterpret_cast<const v4i *>(rows + ((S * 4 * t + r) * RW + s) * 32),
                                                                 o[t], 0, 0, 0);
        v4i b[PT];
#pragma unroll
        for (int t = 0; t < PT; t++)
            b[t] = requant_centred(d, o[t]);
        uint8_t *const y = pr.y + (size_t)((m * pr.OH + oy0) * pr.OW + ox0) * pr.out_cs;
        const uint8_t *const res = pr.res != nullptr ? pr.res + (y - pr.y) : nullptr;
        const bool in_x = ox0 + (p & 7) < pr.OW;
        auto store = [&](const v16i &s, int oy, bool keep, int where) {
            if (!keep || !in_x || oy >= pr.OH)
                return;
            const v4i v = res != nullptr ? requant_add16(pr, s, ldg128(res + where)) : requant16(pr, s, 0);
            *reinterpret_cast<v4i *>(y + where) = v;
        };
        if constexpr (PACK) {
            v16i a = __builtin_amdgcn_mfma_i32_32x32x32_i8(wp[0], b[0], pbias[0], 0, 0, 0);
            a = __builtin_amdgcn_mfma_i32_32x32x32_i8(wq, b[1], a, 0, 0, 0);
            store(a, oy0 + 4 * h + (p >> 3), true, to[0]);
        } else {
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
#pragma unroll
                for (int t = 0; t < PT; t++)
                    store(__builtin_amdgcn_mfma_i32_32x32x32_i8(wp[ct], b[t], pbias[ct], 0, 0, 0), oy0 + 4 * t + (p >> 3),
                          32 * (ct0 + ct) + 16 * h < pr.out_cs, to[ct] + 4 * t * pr.OW * pr.out_cs);
        }
        if (at >= end)
            break;
        lds_order();
    }
}

namespace {

struct PairShape {
    int ph, ct;
    bool narrow;
};
constexpr PairShape kShapes[] = {{4, 1, false}, {4, 2, false}, {4, 3, false}, {4, 5, false}, {8, 1, false}, {8, 2, false}, {8, 3, false},
                                 {4, 1, true},  {4, 2, true},  {8, 1, true},  {8, 2, true}};
constexpr int kCount = sizeof kShapes / sizeof *kShapes;

// how a launch divides the work
struct PairDivision {
    PairGeom geo;
    int nw, rounds; // waves of a work-group; slices (narrow: patches) that one of them takes one after the other
    int held;       // narrow: work-groups that a CU holds
    unsigned lds;
    int groups;
    long long patches, wgs;
};

PairDivision divide(const ConvArgs &d, const ConvArgs &p, const PairShape &s)
{
    const int st = d.stride_h, np = (st * (s.ph - 1) + 3) * (st * 7 + 3), bytes = (2 * np + 63) / 64 * 1024; // as in PairPatch
    PairDivision v;
    v.geo.PY = (p.OH + s.ph - 1) / s.ph, v.geo.PX = (p.OW + 7) / 8, v.geo.nT = (d.in_cs + 31) / 32, v.geo.ct = (p.out_cs + 31) / 32;
    v.groups = v.geo.groups = (v.geo.ct + s.ct - 1) / s.ct;
    v.patches = (long long)d.N * v.geo.PY * v.geo.PX;
    v.geo.red = 0, v.geo.ppi = v.geo.PY * v.geo.PX, v.geo.items = (int)v.patches * v.groups, v.geo.per_xcd = (v.geo.items + 7) / 8;
    hipq_div_magic((uint32_t)v.groups, &v.geo.m_groups, &v.geo.s_groups);
    hipq_div_magic((uint32_t)v.geo.ppi, &v.geo.m_ppi, &v.geo.s_ppi);
    hipq_div_magic((uint32_t)v.geo.PX, &v.geo.m_px, &v.geo.s_px);
    if (s.narrow) {
        const bool three = s.ph == 8 ? s.ct == 1 && p.out_cs == 16 : st == 1 || s.ct == 1; // waves per SIMD that the registers allow, or two
        v.held = three ? 3 : 2;
        v.nw = 4, v.wgs = std::min((v.patches + 3) / 4, 256ll * v.held);
        v.rounds = (int)((v.patches + 4 * v.wgs - 1) / (4 * v.wgs));
        v.lds = (unsigned)(4 * bytes);
    } else {
        v.nw = std::min(v.geo.nT, max_waves(s.ph / 4, s.ct));
        v.rounds = (v.geo.nT + v.nw - 1) / v.nw;
        v.nw = (v.geo.nT + v.rounds - 1) / v.rounds; // the same rounds with fewer waves
        v.wgs = v.patches;
        v.geo.red = v.nw * bytes, v.lds = (unsigned)(v.geo.red + s.ct * (s.ph / 4) * 4096);
    }
    v.geo.nw = v.nw;
    return v;
}

template <int S, int PH, int CT, bool NARROW>
void launch_shape(const ConvArgs &d, const ConvArgs &p, const PairShape &s, hipStream_t st)
{
    const PairDivision v = divide(d, p, s);
    const dim3 block(64 * v.nw), grid(NARROW ? (unsigned)((v.wgs + 7) / 8 * 8) : (unsigned)((v.wgs * v.groups + 7) / 8 * 8), NARROW ? (unsigned)v.groups : 1u);
    if constexpr (!NARROW)
        hipLaunchKernelGGL((conv_dwpoint_kernel<S, PH, CT>), grid, block, v.lds, st, d, p, v.geo);
    else if (PH == 8 && CT == 1 && p.out_cs == 16)
        hipLaunchKernelGGL((conv_dwpoint_narrow_kernel<S, PH, CT, PH == 8 && CT == 1>), grid, block, v.lds, st, d, p, v.geo);
    else
        hipLaunchKernelGGL((conv_dwpoint_narrow_kernel<S, PH, CT, false>), grid, block, v.lds, st, d, p, v.geo);
}

// Time by shape, in us, fitted to 3600 pairs of layers (1 to 128 images of 3x3 to 128x128, 16 to 1024 channels to 12 to 400; nine in
// ten within 15 % of the fit; the shape it picks takes 0.8 % more than the best one on average), narrow ones to 900.  Shared patches: a
// launch; per generation of resident work-groups its start; the slices per SIMD of the chip; per generation the output tiles that a wave finishes and
// the multiplies of its slices; per CU the sums that meet in LDS, and the slices.  Narrow ones: a launch; per patch that a wave takes its
// chain, alone and per wave on its SIMD; the patches, and their channel tiles, per SIMD of the chip; generations.
double shape_cost(const ConvArgs &d, const ConvArgs &p, int shape)
{
    static const double kShared[3][7] = {{2.932, 0.471, 0.142, 0.235, 0.117, 0.636, 0.280}, // 4x8, stride 1
                                         {2.321, 1.496, 0.190, 0.256, 0.086, 0.429, 0.551}, // 8x8
                                         {2.086, 1.572, 0.252, 0.219, 0.133, 0.468, 0.374}}; // 4x8, stride 2
    static const double kNarrow[3][6] = {{2.370, 0, 0.132, 0, 0.435, 0.557}, {2.379, 0.569, 0, 0, 0.794, 0.660}, {3.016, 0, 0.103, 0, 0.695, 0.155}};
    const PairShape &s = kShapes[shape];
    if ((d.stride_h == 2 && s.ph == 8) || (s.narrow && d.in_cs > 32))
        return 1e30; // not built
    const PairDivision v = divide(d, p, s);
    const int row = d.stride_h == 2 ? 2 : s.ph == 8, pt = s.ph / 4, tiles = std::min(s.ct, v.geo.ct);
    const double groups = (double)v.wgs * v.groups, work = (double)v.patches * v.groups / 1024;
    // work-groups that a CU holds
    const int held = s.narrow ? v.held : std::max(1, std::min((int)(160 * 1024 / v.lds), max_waves(pt, s.ct) / v.nw));
    const double gens = std::ceil(groups / (256 * held)), act = std::min((double)held, std::ceil(groups / 256)), steps = gens * v.rounds;
    const double cu = std::ceil(groups / 256);
    const double shared[7] = {1, gens, work * v.geo.nT, gens * ((s.ct * pt + v.nw - 1) / v.nw), gens * v.rounds * s.ct * pt, cu * tiles * pt * v.nw / 16,
                              cu * v.geo.nT / 4};
    const double narrow[6] = {1, steps, steps * act, work, work * tiles, gens};
    double t = 0;
    for (int i = 0; i < (s.narrow ? 6 : 7); i++)
        t += s.narrow ? kNarrow[row][i] * narrow[i] : kShared[row][i] * shared[i];
    return t;
}

int choose_shape(const ConvArgs &d, const ConvArgs &p, int wanted, double *us)
{
    if (wanted >= 0 && wanted < kCount && shape_cost(d, p, wanted) < 1e30) {
        *us = shape_cost(d, p, wanted);
        return wanted;
    }
    int best = 0;
    *us = shape_cost(d, p, best);
    for (int i = 1; i < kCount; i++)
        if (const double t = shape_cost(d, p, i); t < *us)
            *us = t, best = i;
    return best;
}

template <int S>
void launch_stride(const ConvArgs &d, const ConvArgs &p, int shape, hipStream_t st)
{
    const PairShape &s = kShapes[shape];
    if constexpr (S == 1)
        switch (shape) {
        case 4: return launch_shape<S, 8, 1, false>(d, p, s, st);
        case 5: return launch_shape<S, 8, 2, false>(d, p, s, st);
        case 6: return launch_shape<S, 8, 3, false>(d, p, s, st);
        case 9: return launch_shape<S, 8, 1, true>(d, p, s, st);
        case 10: return launch_shape<S, 8, 2, true>(d, p, s, st);
        }
    switch (shape) {
    case 0: return launch_shape<S, 4, 1, false>(d, p, s, st);
    case 1: return launch_shape<S, 4, 2, false>(d, p, s, st);
    case 2: return launch_shape<S, 4, 3, false>(d, p, s, st);
    case 3: return launch_shape<S, 4, 5, false>(d, p, s, st);
    case 7: return launch_shape<S, 4, 1, true>(d, p, s, st);
    case 8: return launch_shape<S, 4, 2, true>(d, p, s, st);
    }
}

bool plain(const ConvArgs &a) { return a.bwz == 0 && a.xmask != 0 && a.lo >= 0 && a.fastq && a.qmult == nullptr; }

} // namespace

bool conv_dwpoint_applies(const ConvArgs &d, const ConvArgs &p)
{
    return plain(d) && d.group == d.C && d.R == 3 && d.S == 3 && d.pad_h == 1 && d.pad_w == 1 && d.stride_h == d.stride_w
        && (d.stride_h == 1 || d.stride_h == 2) && d.in_cs == d.out_cs && d.in_cs % 16 == 0 && (long long)d.N * d.H * d.W * d.in_cs < (1ll << 31)
        && plain(p) && p.group == 1 && p.R == 1 && p.S == 1 && p.pad_h == 0 && p.pad_w == 0 && p.stride_h == 1 && p.stride_w == 1
        && p.wfrag1 != nullptr && p.out_cs % 16 == 0 && p.in_cs == d.in_cs && p.N == d.N && p.H == d.OH && p.W == d.OW
        && (long long)p.P * p.out_cs < (1ll << 31) && (p.res == nullptr || (p.addq.fast && p.addq.hi == 255));
}

double conv_dwpoint_us(const ConvArgs &d, const ConvArgs &p)
{
    double us;
    choose_shape(d, p, -1, &us);
    return us;
}

// The two launches: their latencies, the bytes of the tensor between them, the products of the second, its output, channels and weights,
// and what the tile kernel's two groups of waves add where they keep a 1x1 layer with a partial last slab (an even number of at least 8);
// fitted to 2200 further pairs (nine in ten within 10 %), by 6 % more: the fit above is 8 % above what these measure, and a tie stays apart.
// Of the 2200 this fuses 1796, 20 of them more than 3 % longer (1.3 times at most), and leaves 18 apart that are more than 3 % faster
// as one, where the fit before, which did not tell the partial slabs, left 80 (878 -> 14 channels on five images of 5x4: 8.4 us, 6.1);
// it takes 0.5 % more than the better of the two would each time, before 1.0.
double conv_dwpoint_apart_us(const ConvArgs &d, const ConvArgs &p)
{
    const double mid = (double)p.P * d.in_cs * 1e-6, out = (double)p.P * p.out_cs * 1e-6;
    const double channels = d.in_cs * 1e-3, weights = (double)d.in_cs * p.out_cs * 1e-6;
    const bool partial = d.in_cs % 64 != 0 && p.nslab >= 8 && p.nslab % 2 == 0;
    return d.stride_h == 1 ? 5.92 + 0.669 * mid + 0.00187 * mid * p.out_cs + 0.237 * out + 0.263 * channels + 2.75 * weights + (partial ? 0.172 + 0.1425 * p.nslab : 0)
                           : 6.33 + 1.05 * mid + 0.00243 * mid * p.out_cs + 0.205 * out + 0.158 * channels + 1.62 * weights + (partial ? 0.305 + 0.14 * p.nslab : 0);
}

const char *conv_dwpoint_name(const ConvArgs &d, const ConvArgs &p, int wanted)
{
    static thread_local char nm[48];
    double us;
    const PairShape &s = kShapes[choose_shape(d, p, wanted, &us)];
    snprintf(nm, sizeof nm, "conv_dwpoint_s%d_%s%dx8_n%d", d.stride_h, s.narrow ? "narrow" : "", s.ph, s.ct);
    return nm;
}

void launch_conv_dwpoint(const ConvArgs &d, const ConvArgs &p, int wanted, hipStream_t st)
{
    double us;
    const int shape = choose_shape(d, p, wanted, &us);
    d.stride_h == 1 ? launch_stride<1>(d, p, shape, st) : launch_stride<2>(d, p, shape, st);
}

int conv_dwpoint_shapes() { return kCount; }

} // namespace hipq
