// An inverted residual block of a mobile network in ONE kernel: the 1x1 convolution that widens the channels, the depthwise
// 3x3 convolution, the 1x1 convolution that narrows them again and, where there is one, the residual add.  gfx950 only.
//
// Reproduces, bit for bit, op_conv_2d_u8xu8_run (art/modules/quant/src/op/conv_2d_uint8_impl.c:39-165) three times and
// op_quant_add_run (art/modules/quant/src/op/add.c:83-148): every intermediate value is requantised, clamped and re-read exactly
// as if it had travelled through memory.
//
// Why: the hidden tensor is six times as wide as the block's input and output, is written and read twice, and the three layers
// are three launches.  Here a work-group owns a patch of output pixels of ONE image, and its waves take the hidden channels in
// slices of 32.  A wave takes a slice through all three layers on its own, without a barrier:
//   * expand: the slice's weights, channels as the ROWS of the multiply, times the patch's input region, which lies re-centred in
//     LDS: the 16 accumulators of a lane are 16 consecutive channels of one position, requantised to 16 bytes of its row in LDS;
//   * depthwise, also on the matrix cores: for each of the nine taps a diagonal matrix of the slice's 32 weights, made from a dword by
//     a byte permutation and four ANDs, times the rows at that tap.  31 of 32 products are with zeros, and still nine matrix
//     instructions and 45 others replace the 130 dot products, byte alignments and LDS reads of 32 outputs of 32 channels: the
//     matrix cores idle, and vector instructions are the largest part of a wave's chain;
//   * the requantised sums are, as they lie in the lanes, one k-step of the last layer's pixel operand.  Where the waves split one patch
//     they put them into LDS, and after the only barrier the last layer's output tiles go to the waves instead of the slices (its
//     first weights wait in LDS by then); where a wave has a patch it multiplies them at once.
// Patches of 2x4 outputs do not fill a multiply's 32 columns.  Theirs keeps the expanded pixels as rows (a lane has four runs of four
// consecutive pixels of ONE channel), takes dot products of such a run with {w0, w1, w2, 0} and {0, w0, w1, w2} (two neighbouring
// outputs; one at stride 2), and puts the result into LDS byte by byte.
// Positions outside the image hold the depthwise layer's pad byte; the border of a patch is expanded again by its neighbours,
// which costs vector instructions (the requantisation), not memory.
// Two divisions of the work.  Few patches: the waves of a work-group split the slices of one patch, then its output tiles.  (Partial sums
// of every output in every wave, added up in LDS, took the registers of eight waves instead of twelve or sixteen and 64 atomic
// additions a wave: 64 -> 384 -> 64 at 14x14, batch 64, 11.8 us, this way 9.4; 64 -> 384 -> 96 12.6 and 9.5; 96 -> 576 -> 96 16.1 and
// 12.8; 32 -> 192 -> 64 from 28x28, stride 2, 12.3 and 9.0; 64 -> 384 -> 64 on one image 6.5 and 5.9.)  Many patches and few slices: every
// wave has a patch of its own and takes all slices through it, so that no barrier ties it to others - with shared patches each wave of
// a 24 -> 144 -> 24 block has one slice between two barriers, 46 us at 56x56, batch 64, against 27.
// Patches are 2x4 outputs where even so the chip is nearly empty (a slice's chain of
// instructions is then a third as long as for 4x8), 4x8, 8x8 or 7x7 otherwise: fewer positions expanded twice, and 7x7 fills three of a
// multiply's tiles with its region where 8x8 fills three and an eighth, and divides images of 14x14 and 28x28 (64 -> 384 -> 64
// 10.4 and 9.4 us).  But a wave of 8x8 outputs
// with a patch of its own holds 168 registers where one of 4x8 holds 110: 29.2 us against 26.8 for 24 -> 144 -> 24, 14.2 against 12.2 for
// 32 -> 192 -> 32 at 28x28.
// A work-group's first instructions count: its pixels, its waves' weights and biases of all layers are under way before the first wait,
// with quotients from the host (0.6 us of each block; until then the weights followed the pixels).
// What bounds it, at batch 64: with a patch per wave vector issue first (the requantisations; 57 to 60 % of a CU's busy time at 4 clocks an
// instruction, matrix cores 9 to 10 %).  With a shared patch the chain of a wave, region - expand - LDS - depthwise - LDS -
// project, a slice after the other, with three waves a SIMD (vector issue 32 to 38 %, matrix cores 4 to 9 %).
// Measured, the three launches -> this one (batch 64, launches back to back, random bytes): 24 -> 144 -> 24 at 56x56: 39.5 -> 26.8 us;
// 32 -> 192 -> 32 at 28x28: 18.4 -> 12.2; 64 -> 384 -> 64 at 14x14: 14.7 -> 9.4; 96 -> 576 -> 96: 18.1 -> 12.8; 160 -> 960 -> 160 at 7x7: 15.1 -> 14.0;
// batch 1, 24 -> 144 -> 24: 10.4 -> 5.8.
// Requirements (checked by the host): uint8 tensors, weight zero points 128, per-tensor scales, one-multiply
// requantisations, at most 160 input and output channels; with the add stride 1 and as many output as input channels.
#include "conv_invres.h"

#include <algorithm>

#include "conv_dw_frag.h"
#include "conv_dwpoint.h"

namespace hipq {

using namespace frag;

namespace {

constexpr int kStaged = 6; // k-steps of the last layer's weights that wait in LDS, at most

// waves of a work-group: four per SIMD leave each 128 registers, three 168
constexpr int max_waves(bool MATRIX, int TILES, int NK) { return NK <= (MATRIX ? 1 : 2) && TILES <= (MATRIX ? 4 : 1) ? 16 : 12; }

struct InvresGeom {
    int ppi, PX, patches, per_xcd; // patches of an image, of a row of it, all; work-groups of an XCD
    uint32_t m_ppi, m_px;          // x / ppi and x / PX (hipq_div_magic)
    int s_ppi, s_px;
    int nw;               // waves
    int pieces, m_pieces; // 16-byte pieces of an input pixel; id / pieces == (id * m_pieces) >> 16, id < 4096
    int nT;     // slices of 32 hidden channels
    int nk, ct; // k-steps of the expanding layer, channel tiles of the projecting one
    int xrow;   // bytes of a pixel row of the input region in LDS
    int region; // bytes of an input region with its masks in LDS
    int wave_bytes; // bytes of a wave's own buffers
    int hidden;     // bytes of the patch's depthwise results in LDS
    int ks, per;    // waves that share a tile of the last layer, k-steps of one
    int slab;       // bytes of two k-steps of all its channel tiles
    int weights;    // where the first weights of the last layer lie in LDS
    int depth;      // k-steps of them, for each wave
    int bias;       // where the last layer's biases lie
    int m_tiles;    // i / tiles == (i * m_tiles) >> 16, i below 16
};

// S: stride, PH x PW: output pixels of a patch.  Rows and columns of the input region; tiles of 32 positions; pixel tiles of 32
// outputs.
// MATRIX: the depthwise layer as diagonal matrices, for patches that fill a multiply's 32 columns; otherwise as dot products, with the
// region's rows in whole runs of four columns.
template <int S, int PH_, int PW_>
struct Patch {
    static constexpr int PH = PH_, PW = PW_;
    static constexpr bool MATRIX = PH * PW >= 32;
    static constexpr int QW = (S * (PW - 1) + 3 + 3) / 4, RH = S * (PH - 1) + 3, RW = MATRIX ? S * (PW - 1) + 3 : 4 * QW, NP = RH * RW;
    static constexpr int TILES = (NP + 31) / 32, PT = (PH * PW + 31) / 32;
    static constexpr int E_BYTES = TILES * 1024, MASK_BYTES = MATRIX ? 0 : TILES * 32;
};

__device__ static __forceinline__ int32_t dot4(uint32_t a, int b, int32_t c)
{
    return __builtin_amdgcn_sdot4((int)a, b, c, false);
}

// dot(a, b) + c into a new register: the compiler's own choice for this is a copy of c followed by the accumulating form
__device__ static __forceinline__ int32_t dot4_from(uint32_t a, int32_t b, int32_t c)
{
    int32_t d;
    asm("v_dot4_i32_i8 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}

// x / d for any x below 2^31 (hipq_div_magic)
__device__ static __forceinline__ int quot(int x, uint32_t m, int s) { return m ? (int)(__umulhi((uint32_t)x, m) >> s) : x; }

} // namespace

// NK: k-steps of 32 input channels (may be more than the layer has: the weights are zeros there).  OWN: every wave has a patch of its
// own and takes all slices through it, over the accumulators of CT tiles of 32 output channels; otherwise the waves of a work-group split
// the slices of one patch and then the output tiles.
template <int S, int PH, int PW, int NK, int CT, bool OWN>
__global__ __launch_bounds__(OWN ? 256 : 64 * max_waves(Patch<S, PH, PW>::MATRIX, Patch<S, PH, PW>::TILES, NK)) void conv_invres_kernel(const ConvArgs e, const ConvArgs d, const ConvArgs pr,
                                                                                const InvresGeom geo)
{
    using G = Patch<S, PH, PW>;
    constexpr int RH = G::RH, RW = G::RW, NP = G::NP, TILES = G::TILES, PT = G::PT, QW = G::QW;
    constexpr bool MATRIX = G::MATRIX;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = geo.nw;
    const int p = lane & 31, h = lane >> 5;
    const int ch = slice_channel(p); // the channel of a slice that this lane's column stands for
    // work-groups go to the 8 XCDs in turn: XCD x takes the x-th contiguous eighth of the patches
    int gid = (int)(blockIdx.x % 8) * geo.per_xcd + (int)(blockIdx.x / 8);
    if (OWN)
        gid = gid * nw + wave;
    if (gid >= geo.patches)
        return;
    const int n = quot(gid, geo.m_ppi, geo.s_ppi), pi = gid - n * geo.ppi, py = quot(pi, geo.m_px, geo.s_px);
    const int oy0 = py * PH, ox0 = (pi - py * geo.PX) * PW;
    const int iy0 = S * oy0 - 1, ix0 = S * ox0 - 1; // the region's first row and column
    const bool inside = iy0 >= 0 && ix0 >= 0 && iy0 + RH <= e.H && ix0 + RW <= e.W; // no position to replace
    uint8_t *const xbuf = lds + (OWN ? wave * (geo.region + geo.wave_bytes) : geo.hidden);
    uint32_t *const masks = reinterpret_cast<uint32_t *>(xbuf + geo.region - G::MASK_BYTES); // dot products: which bytes of a run lie inside the image
    uint8_t *const ebuf = xbuf + geo.region + (OWN ? 0 : wave * geo.wave_bytes);

    // ---- a slice's weights and constants, each loaded as soon as the slice before has used its own
    v4i we[NK], wp[OWN ? CT : 1];
    // MATRIX: the folded biases of the lane's 16 consecutive channels, and the depthwise weights of the channel that its row of a multiply
    // stands for, a kernel row each; otherwise biases and weights of the channel that its column stands for, the weights in both
    // alignments
    v16i ebias, dbias;
    int ebias1, dbias1, wd[3], wb[3];
    auto load_e = [&](int T) {
        if constexpr (MATRIX)
            init_acc(ebias, e.bias2 + 32 * T + 16 * h, false);
        else
            ebias1 = e.bias2[32 * T + ch];
#pragma unroll
        for (int kk = 0; kk < NK; kk++)
            we[kk] = kk == 0 || kk < geo.nk ? ldg128(e.wfrag1 + ((size_t)((kk >> 1) * (e.kout_pad >> 5) + T) * 2 + (kk & 1)) * 1024 + lane * 16)
                                            : v4i{0, 0, 0, 0};
    };
    const DiagonalTap taps(lane);
    auto load_d = [&](int T) {
        const int c0 = min(32 * T + 16 * h, d.in_cs - 16), cd = min(32 * T + ch, d.in_cs - 1); // the last slice may be half empty; its products meet zero weights
        if constexpr (MATRIX)
            init_acc(dbias, d.bias2 + c0, false);
        else
            dbias1 = d.bias2[cd];
        const int *wt = reinterpret_cast<const int *>(d.wpack) + cd;
#pragma unroll
        for (int r = 0; r < 3; r++) {
            wd[r] = wt[(r * 2 + 0) * d.in_cs];
            if (!MATRIX && S == 1)
                wb[r] = wt[(r * 2 + 1) * d.in_cs];
        }
    };
    auto load_p = [&](int T) {
#pragma unroll
        for (int ct = 0; OWN && ct < CT; ct++)
            wp[ct] = ct == 0 || ct < geo.ct ? ldg128(pr.wfrag1 + ((size_t)((T >> 1) * (pr.kout_pad >> 5) + ct) * 2 + (T & 1)) * 1024 + lane * 16)
                                            : v4i{0, 0, 0, 0};
    };

    // ---- the input region -> LDS, re-centred.  Positions outside the image are never used (the mask below) and hold the bytes of one inside.
    // A thread's first pieces are under way before the weights
    constexpr int AHEAD = OWN ? (NP <= 64 ? 2 : 4) : PT;
    const int tid = OWN ? lane : (int)threadIdx.x, nthr = OWN ? 64 : nw * 64, total = NP * geo.pieces;
    v4i piece[AHEAD];
    auto load_pieces = [&](int id0) {
#pragma unroll
        for (int j = 0; j < AHEAD; j++) {
            const int id = min(id0 + j * nthr, total - 1), px = (id * geo.m_pieces) >> 16, ry = px / RW;
            const int iy = min(max(iy0 + ry, 0), e.H - 1), ix = min(max(ix0 + px - ry * RW, 0), e.W - 1);
            piece[j] = ldg128(e.x + (uint32_t)(((n * e.H + iy) * e.W + ix) * e.in_cs + (id - px * geo.pieces) * 16));
        }
    };
    auto store_pieces = [&](int id0) {
#pragma unroll
        for (int j = 0; j < AHEAD; j++) {
            const int id = min(id0 + j * nthr, total - 1), px = (id * geo.m_pieces) >> 16;
            *reinterpret_cast<v4i *>(xbuf + px * geo.xrow + (id - px * geo.pieces) * 16) = piece[j] ^ (int)0x80808080;
        }
    };
    load_pieces(tid);
    load_e(OWN ? 0 : wave); // never more waves than slices
    load_d(OWN ? 0 : wave);
    load_p(0);
    // otherwise: a wave's tile of the last layer, 32 channels by 32 pixels, or its share of the tile's k-steps with ks waves a tile.  The
    // first steps' weights wait in LDS while the slices are computed, and so do the folded biases
    const int tiles = geo.ct * PT, items = tiles * geo.ks;
    uint8_t *const wbuf = lds + geo.weights + wave * geo.depth * 1024;
    auto step = [&](int ct, int k) { // the lane's weights; k-steps lie in pairs, a pair of every channel tile after the other
        k = min(k, geo.nT - 1);
        return pr.wfrag1 + ((uint32_t)((k >> 1) * geo.slab + (2 * ct + (k & 1)) * 1024) + lane * 16);
    };
    if constexpr (!OWN) {
        const int share = wave * geo.m_tiles >> 16, ct = (wave - share * tiles) / PT;
        const int k0 = share * geo.per;
#pragma unroll
        for (int j = 0; j < kStaged; j++)
            if (j < geo.depth && wave < items)
                __builtin_amdgcn_global_load_lds((gptr_t)step(ct, k0 + j), (lptr_t)(wbuf + j * 1024), 16, 0, 0);
        for (int c = wave; 2 * c < geo.ct; c += nw)
            __builtin_amdgcn_global_load_lds((gptr_t)(pr.bias2 + min(64 * c + lane, 32 * geo.ct - 1)), (lptr_t)(lds + geo.bias + 256 * c), 4, 0, 0);
    }
    store_pieces(tid);
    for (int id = tid + AHEAD * nthr; id < total; id += AHEAD * nthr) {
        load_pieces(id);
        store_pieces(id);
    }
    if (!MATRIX && !inside)
        for (int q = (OWN ? lane : (int)threadIdx.x); q < TILES * 8; q += nthr) {
            const int ry = q / QW, rx = (q - ry * QW) * 4, iy = iy0 + ry;
            uint32_t m = 0;
            if (q < RH * QW && (unsigned)iy < (unsigned)e.H)
                for (int b = 0; b < 4; b++)
                    m |= (unsigned)(ix0 + rx + b) < (unsigned)e.W ? 0xffu << (8 * b) : 0u;
            masks[q] = m;
        }
    uint32_t outside = 0; // bit t: the lane's position of tile t lies outside the image
    if (MATRIX && !inside)
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            const int pos = 32 * t + p, ry = pos / RW;
            outside |= (int)((unsigned)(iy0 + ry) >= (unsigned)e.H) | (int)((unsigned)(ix0 + pos - ry * RW) >= (unsigned)e.W) ? 1u << t : 0u;
        }
    int first[PT]; // the lane's outputs 32 t + p: their first tap in the expanded region
#pragma unroll
    for (int t = 0; t < PT; t++) {
        const int m = min(32 * t + p, PH * PW - 1);
        first[t] = (S * (m / PW) * RW + S * (m % PW)) * 32 + 16 * h;
    }
    v16i acc[OWN ? CT : 1][PT]; // from the folded bias of the lane's 16 consecutive channels
    if constexpr (OWN)
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
#pragma unroll
            for (int t = 0; t < PT; t++)
                init_acc(acc[ct][t], pr.bias2 + 32 * (ct < geo.ct ? ct : 0) + 16 * h, false);
    const int epad = (int)(d.padword ^ 0x80808080u);
    if (OWN)
        lds_order();
    else {
        wait_vmcnt<0>();
        __syncthreads(); // the region, the masks and the last layer's first weights are in LDS
    }

    auto slice = [&](int T, int Tn) { // Tn: the wave's next one, past the end a harmless load
        v4i b[PT]; // the depthwise layer's bytes, as the last layer's pixel operand
        if constexpr (MATRIX) {
            // ---- expand: a lane's 16 channels of a position are 16 bytes of the position's row
            auto expand = [&](auto whole) {
#pragma unroll (TILES <= 4 ? TILES : 2)
                for (int t = 0; t < TILES; t++) {
                    v16i a = ebias;
                    const uint8_t *row = xbuf + (32 * t + p) * geo.xrow + 16 * h;
#pragma unroll
                    for (int kk = 0; kk < NK; kk++)
                        a = __builtin_amdgcn_mfma_i32_32x32x32_i8(we[kk], *reinterpret_cast<const v4i *>(row + 32 * kk), a, 0, 0, 0);
                    v4i v = requant_centred(e, a);
                    if (!decltype(whole)::value && (outside >> t & 1))
                        v = v4i{epad, epad, epad, epad};
                    *reinterpret_cast<v4i *>(ebuf + (32 * t + p) * 32 + 16 * h) = v;
                }
            };
            if (inside)
                expand(std::true_type{});
            else
                expand(std::false_type{});
            load_e(Tn);
            lds_order();
            // ---- depthwise, on the matrix cores: tap by tap a diagonal matrix times the region's rows at that tap.  The requantised sums
            // are the pixel operand of the last layer as they are
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
                        o[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(m, *reinterpret_cast<const v4i *>(ebuf + first[t] + (r * RW + s) * 32), o[t], 0, 0, 0);
                }
            load_d(Tn);
#pragma unroll
            for (int t = 0; t < PT; t++)
                b[t] = requant_centred(d, o[t]);
        } else {
            // ---- expand, pixels as the rows of the multiply: a lane's accumulators are four runs of four consecutive pixels of its channel
            auto expand = [&](auto whole) {
#pragma unroll
                for (int t = 0; t < TILES; t++) {
                    v16i a;
                    const uint8_t *row = xbuf + (32 * t + p) * geo.xrow + 16 * h;
#pragma unroll
                    for (int i = 0; i < 16; i++)
                        a[i] = ebias1;
#pragma unroll
                    for (int kk = 0; kk < NK; kk++)
                        a = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const v4i *>(row + 32 * kk), we[kk], a, 0, 0, 0);
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        const int q = 8 * t + 2 * g + h;
                        uint32_t v = conv_requant4<false>(e, a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]) ^ 0x80808080u;
                        if (!decltype(whole)::value) {
                            const uint32_t m = masks[q];
                            v = (v & m) | ((uint32_t)epad & ~m);
                        }
                        *reinterpret_cast<uint32_t *>(ebuf + (q * 32 + p) * 4) = v;
                    }
                }
            };
            if (inside)
                expand(std::true_type{});
            else
                expand(std::false_type{});
            load_e(Tn);
            lds_order();
            // ---- depthwise: half h of the wave takes PH / 2 output rows of this lane's channel
            constexpr int HR = PH / 2, IR = S * (HR - 1) + 3;
            int32_t o[HR][PW];
#pragma unroll
            for (int ir = 0; ir < IR; ir++) {
                const uint8_t *er = ebuf + ((S * HR * h + ir) * QW * 32 + p) * 4;
                uint32_t q[QW];
#pragma unroll
                for (int i = 0; i < QW; i++)
                    q[i] = *reinterpret_cast<const uint32_t *>(er + i * 128);
                uint32_t mid[QW - 1]; // bytes 2, 3 of run i and 0, 1 of run i + 1
#pragma unroll
                for (int i = 0; i + 1 < QW; i++)
                    mid[i] = __builtin_amdgcn_alignbyte(q[i + 1], q[i], 2);
#pragma unroll
                for (int r = 0; r < HR; r++) {
                    const int kr = ir - S * r;
                    if (kr < 0 || kr > 2)
                        continue;
#pragma unroll
                    for (int x = 0; x < PW; x++) {
                        const uint32_t v = S == 1 ? ((x & 2) ? mid[x >> 2] : q[x >> 2]) : ((x & 1) ? mid[x >> 1] : q[x >> 1]);
                        const int w = S == 1 && (x & 1) ? wb[kr] : wd[kr];
                        o[r][x] = kr == 0 ? dot4_from(v, w, dbias1) : dot4(v, w, o[r][x]);
                    }
                }
            }
            load_d(Tn);
            // this lane's channel of its outputs, as bytes of the operand that the last layer multiplies
#pragma unroll
            for (int r = 0; r < HR; r++)
#pragma unroll
                for (int x4 = 0; x4 < PW; x4 += 4) {
                    const uint32_t v = conv_requant4<false>(d, o[r][x4], o[r][x4 + 1], o[r][x4 + 2], o[r][x4 + 3]) ^ 0x80808080u;
                    uint8_t *to = lds + T * 1024 + ((ch >> 4) * 32 + (HR * h + r) * PW + x4) * 16 + (ch & 15);
                    to[0] = (uint8_t)v, to[16] = (uint8_t)(v >> 8), to[32] = (uint8_t)(v >> 16), to[48] = (uint8_t)(v >> 24);
                }
        }
        // ---- project: one k-step of every channel tile (rows past the patch, where it has fewer than 32 pixels, are never stored)
        if constexpr (OWN) {
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
#pragma unroll
                for (int t = 0; t < PT; t++)
                    acc[ct][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wp[ct], b[t], acc[ct][t], 0, 0, 0);
            load_p(Tn);
        } else if constexpr (MATRIX) {
#pragma unroll
            for (int t = 0; t < PT; t++)
                *reinterpret_cast<v4i *>(lds + (T * PT + t) * 1024 + lane * 16) = b[t];
        }
        lds_order();
    };

    auto place = [&](int ct, int t, uint32_t *at) { // of the lane's 16 channels of its pixel
        const int m = 32 * t + p, oy = oy0 + m / PW, ox = ox0 + m % PW, c0 = 32 * ct + 16 * h;
        *at = (uint32_t)(((n * pr.OH + oy) * pr.OW + ox) * pr.out_cs + c0); // below 2^31
        return (m < PH * PW) & (oy < pr.OH) & (ox < pr.OW) & (c0 < pr.out_cs);
    };
    if constexpr (OWN) {
        for (int T = 0; T < geo.nT; T++)
            slice(T, min(T + 1, geo.nT - 1));
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
#pragma unroll
            for (int t = 0; t < PT; t++) {
                uint32_t at;
                if (place(ct, t, &at))
                    *reinterpret_cast<v4i *>(pr.y + at) = pr.res != nullptr ? requant_add16(pr, acc[ct][t], ldg128(pr.res + at)) : requant16(pr, acc[ct][t], 0);
            }
    } else {
        for (int T = wave; T < geo.nT; T += nw)
            slice(T, min(T + nw, geo.nT - 1));
        // ---- project, from the whole patch's depthwise results
        constexpr int D = 4; // k-steps of weights ahead
        for (int i = wave; i == wave || i < items; i += nw) {
            asm("" : "+s"(i)); // what hangs on it is computed here, not kept in registers from the front
            const bool work = i < items;
            const int share = work ? i * geo.m_tiles >> 16 : 0, tile = work ? i - share * tiles : 0, ct = tile / PT, t = tile - ct * PT;
            const int k0 = min(share * geo.per, geo.nT), k1 = work ? min(k0 + geo.per, geo.nT) : k0;
            uint32_t at;
            const bool store = place(ct, t, &at) && work && share == 0;
            const v4i *const bias = reinterpret_cast<const v4i *>(lds + geo.bias + 128 * ct + 64 * h);
            v4i res = {0, 0, 0, 0};
            if (S == 1 && store && pr.res != nullptr) { // the residual is the block's input
                const int m = 32 * t + p;
                res = *reinterpret_cast<const v4i *>(xbuf + ((m / PW + 1) * RW + m % PW + 1) * geo.xrow + 32 * ct + 16 * h) ^ (int)0x80808080;
            }
            v16i sum;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4i q = share > 0 ? v4i{0, 0, 0, 0} : bias[j];
                sum[4 * j] = q[0], sum[4 * j + 1] = q[1], sum[4 * j + 2] = q[2], sum[4 * j + 3] = q[3];
            }
            const int kr = i == wave ? min(k0 + geo.depth, k1) : k0;
            v4i w[D];
            if (kr < k1)
#pragma unroll
                for (int j = 0; j < D; j++)
                    w[j] = ldg128(step(ct, kr + j));
            if (i == wave)
                __syncthreads(); // the slices are there
            constexpr int GROUP = MATRIX && NK == 1 ? 3 : kStaged; // as many as the registers hold
            for (int k = k0; k < kr; k += GROUP) {
                v4i ws[GROUP], xs[GROUP];
#pragma unroll
                for (int j = 0; j < GROUP; j++) {
                    const int kj = min(k + j, kr - 1);
                    ws[j] = *reinterpret_cast<const v4i *>(wbuf + (kj - k0) * 1024 + lane * 16);
                    xs[j] = *reinterpret_cast<const v4i *>(lds + (kj * PT + t) * 1024 + lane * 16);
                }
#pragma unroll
                for (int j = 0; j < GROUP; j++)
                    if (k + j < kr)
                        sum = __builtin_amdgcn_mfma_i32_32x32x32_i8(ws[j], xs[j], sum, 0, 0, 0);
            }
            for (int k = kr; k < k1; k += D)
#pragma unroll
                for (int j = 0; j < D; j++) {
                    if (k + j < k1)
                        sum = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[j], *reinterpret_cast<const v4i *>(lds + ((k + j) * PT + t) * 1024 + lane * 16), sum, 0, 0, 0);
                    if (k + D < k1)
                        w[j] = ldg128(step(ct, k + j + D));
                }
            if (geo.ks > 1) { // the shares meet where the region was (no wave has two items then)
                v4i *const red = reinterpret_cast<v4i *>(xbuf) + tile * 256 + lane;
                if (share > 0)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        red[(share - 1) * tiles * 256 + j * 64] = v4i{sum[4 * j], sum[4 * j + 1], sum[4 * j + 2], sum[4 * j + 3]};
                __syncthreads();
                if (work && share == 0)
                    for (int s = 0; s + 1 < geo.ks; s++)
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const v4i q = red[s * tiles * 256 + j * 64];
                            sum[4 * j] += q[0], sum[4 * j + 1] += q[1], sum[4 * j + 2] += q[2], sum[4 * j + 3] += q[3];
                        }
            }
            if (store)
                *reinterpret_cast<v4i *>(pr.y + at) = pr.res != nullptr ? requant_add16(pr, sum, res) : requant16(pr, sum, 0);
        }
    }
}

namespace {

// the channel counts that are built: k-steps of the expanding layer and channel tiles of the projecting one, each at least what the
// layers have
struct Channels {
    int nk, ct;
};

Channels channels_of(const ConvArgs &e, const ConvArgs &p)
{
    const int nk = (e.in_cs + 31) / 32, ct = (p.out_cs + 31) / 32;
    if (nk == 1 && ct <= 2)
        return {1, ct};
    if (nk <= 2 && ct <= 3)
        return {2, ct <= 2 ? 2 : 3};
    if (nk <= 3)
        return {3, ct <= 3 ? 3 : 5};
    return {5, 5};
}

// kOwn: a patch per wave, 8x8 outputs at stride 1, 4x8 at stride 2; kOwn4: 4x8 at stride 1
enum Shape { k2x4, k4x8, k8x8, kOwn, kOwn4, k7x7, kShapes };

bool own(int shape) { return shape == kOwn || shape == kOwn4; }

// how a launch divides the work
struct Division {
    int PY, PX, nT, xrow, region, wave_bytes, hidden, ks, weights, depth, bias;
    int nw, rounds; // waves of a work-group; slices that one of them takes one after the other
    int waves;      // of a SIMD that the registers allow
    int tiles;      // of the last layer
    unsigned lds;
    long long wgs;
};

Division divide(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, int shape)
{
    const Channels c = channels_of(e, p);
    const int S = d.stride_h, ph = shape == k2x4 ? 2 : shape == k7x7 ? 7 : shape == k8x8 || (shape == kOwn && S == 1) ? 8 : 4;
    const int pw = shape == k2x4 ? 4 : shape == k7x7 ? 7 : 8;
    const bool matrix = ph * pw >= 32; // these as in Patch
    const int tiles = ((S * (ph - 1) + 3) * (matrix ? S * (pw - 1) + 3 : (S * (pw - 1) + 6) / 4 * 4) + 31) / 32, pt = (ph * pw + 31) / 32;
    Division v;
    v.PY = (p.OH + ph - 1) / ph, v.PX = (p.OW + pw - 1) / pw;
    v.nT = (d.in_cs + 31) / 32;
    // rows of 16 bytes (the other half of a k-step meets zero weights) and of 32 read without bank conflicts as they are, longer
    // ones 16 bytes apart
    v.xrow = e.in_cs == 16 ? 16 : c.nk == 1 ? 32 : 32 * c.nk + 16;
    v.region = (tiles * 32 * v.xrow + 16 + (matrix ? 0 : tiles * 32) + 15) / 16 * 16;
    v.wave_bytes = tiles * 1024;
    const long long patches = (long long)d.N * v.PY * v.PX;
    if (own(shape)) {
        v.nw = 4, v.rounds = v.nT, v.wgs = (patches + 3) / 4;
        v.lds = (unsigned)(4 * (v.region + v.wave_bytes)), v.hidden = v.weights = v.depth = v.bias = 0, v.ks = 1, v.tiles = c.ct * pt;
        v.waves = shape == kOwn4 || S == 2 ? (c.ct == 1 ? 4 : 3) : c.ct == 1 ? 3 : 2;
    } else {
        const int out = v.tiles = (p.out_cs + 31) / 32 * pt;
        v.nw = std::min(v.nT, max_waves(matrix, tiles, c.nk)), v.rounds = (v.nT + v.nw - 1) / v.nw;
        v.nw = (v.nT + v.rounds - 1) / v.rounds; // the same rounds with fewer waves
        v.ks = std::max(1, std::min(v.nw / out, v.nT / 6)); // shares of six k-steps: a shorter one takes longer to add up than to multiply
        const int rest = std::max(v.region + v.nw * v.wave_bytes, (v.ks - 1) * out * 4096), holders = std::min(v.nw, out * v.ks);
        v.hidden = v.nT * pt * 1024, v.bias = v.hidden + rest, v.weights = v.bias + (p.out_cs + 63) / 64 * 256;
        v.depth = std::min((v.nT + v.ks - 1) / v.ks, kStaged);
        while (v.depth > 0 && v.weights + holders * v.depth * 1024 > 160 * 1024)
            v.depth--;
        v.wgs = patches;
        v.lds = (unsigned)(v.weights + holders * v.depth * 1024), v.waves = max_waves(matrix, tiles, c.nk) / 4;
    }
    return v;
}

template <int S, int PH, int PW, int NK, int CT, bool OWN>
void launch_shape(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, int shape, hipStream_t st)
{
    using G = Patch<S, PH, PW>;
    const Division v = divide(e, d, p, shape);
    InvresGeom geo;
    geo.nk = (e.in_cs + 31) / 32, geo.ct = (p.out_cs + 31) / 32;
    geo.ppi = v.PY * v.PX, geo.PX = v.PX, geo.patches = d.N * geo.ppi, geo.per_xcd = (int)((v.wgs + 7) / 8), geo.nw = v.nw;
    hipq_div_magic((uint32_t)geo.ppi, &geo.m_ppi, &geo.s_ppi);
    hipq_div_magic((uint32_t)geo.PX, &geo.m_px, &geo.s_px);
    geo.pieces = e.in_cs / 16, geo.m_pieces = 65536 / geo.pieces + 1, geo.slab = p.kout_pad / 32 * 2048;
    geo.nT = v.nT, geo.xrow = v.xrow, geo.region = v.region, geo.wave_bytes = v.wave_bytes, geo.hidden = v.hidden;
    geo.ks = v.ks, geo.per = (v.nT + v.ks - 1) / v.ks, geo.m_tiles = 65536 / (geo.ct * G::PT) + 1;
    geo.weights = v.weights, geo.depth = v.depth, geo.bias = v.bias;
    static_assert(G::E_BYTES == G::TILES * 1024, "divide()");
    hipLaunchKernelGGL((conv_invres_kernel<S, PH, PW, NK, CT, OWN>), dim3((unsigned)((v.wgs + 7) / 8 * 8)), dim3(64 * v.nw), v.lds, st, e, d, p, geo);
}

// ---- the shapes, and what each takes

// Time by shape, in us, fitted to 2400 blocks (1 to 128 images of 3x3 to 128x128, 16 to 160 channels widened 1 to 6 times; nine in ten
// within 15 % of the fit).  A launch; for every generation of resident work-groups its start and end, and the k-steps of the last layer
// that a wave takes, or a slice's channel tiles where each wave has a patch; per SIMD of the chip the slices, and their output channel tiles;
// per SIMD of a CU the slices, and their k-steps; the input's MB.  Chosen by this the blocks take 0.5 % more than the best shape would on
// average, one in twenty more than 5 %.
double shape_cost(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, int shape)
{
    // launch, generation, k-steps of the last layer, slices per SIMD, x channel tiles, slices of a CU's SIMD, x k-steps, MB
    static const double kCost[2][kShapes][8] = {
        {{3.871, 0.308, 0.029, 0.014, 0.084, 0.204, 0.059, 0.058}, {3.880, 0.462, 0.045, 0.111, 0.085, 0.446, 0.082, 0.142},
         {4.348, 0.870, 0.000, 0.000, 0.335, 0.695, 0.165, 0.147}, {3.345, 0.960, 0.289, 0.000, 0.164, 0.839, 0.000, 0.189},
         {3.049, 0.595, 0.219, 0.000, 0.052, 0.470, 0.000, 0.295}, {4.469, 0.556, 0.000, 0.027, 0.266, 0.667, 0.161, 0.054}},
        {{4.046, 0.309, 0.028, 0.025, 0.060, 0.201, 0.096, 0.177}, {4.210, 0.527, 0.052, 0.015, 0.133, 0.535, 0.173, 0.238},
         {}, {3.089, 0.703, 0.321, 0.000, 0.083, 0.833, 0.000, 0.169}, {}, {}}};
    const int s = d.stride_h;
    const Channels c = channels_of(e, p);
    if ((own(shape) && (c.nk > 2 || c.ct > 2)) || (shape == kOwn4 && s == 2) || ((shape == k8x8 || shape == k7x7) && (s == 2 || c.ct > 3)))
        return 1e30; // not built: the accumulators or the region would be too much for a wave
    const Division v = divide(e, d, p, shape);
    if (v.lds > 160 * 1024) // 8x8 and 7x7 patches of 1450 hidden channels and more; the smaller patches hold the 2048 that a layer can have here
        return 1e30;
    const int held = std::max(1, std::min((int)(160 * 1024 / v.lds), v.waves / ((v.nw + 3) / 4))); // work-groups of a CU, the first wave of each on the first SIMD
    const double gens = (double)((v.wgs + 256 * held - 1) / (256 * held)), steps = gens * v.rounds;
    const double work = (double)d.N * v.PY * v.PX * v.nT / 1024, slices = (double)((v.wgs + 255) / 256) * v.rounds * v.nw / 4;
    const double last = own(shape) ? steps * c.ct : gens * ((v.tiles * v.ks + v.nw - 1) / v.nw) * ((v.nT + v.ks - 1) / v.ks);
    const double f[8] = {1, gens, last, work, work * ((p.out_cs + 31) / 32), slices, slices * c.nk, (double)e.P * e.in_cs * 1e-6};
    double t = 0;
    for (int i = 0; i < 8; i++)
        t += kCost[s - 1][shape][i] * f[i];
    return t;
}

// wanted: the caller's choice, where that shape is built for these channels; -1: the cheapest
int choose_shape(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, int wanted, double *us)
{
    if (wanted >= 0 && wanted < kShapes && shape_cost(e, d, p, wanted) < 1e30) {
        *us = shape_cost(e, d, p, wanted);
        return wanted;
    }
    int best = k2x4;
    *us = shape_cost(e, d, p, best);
    for (int sh = k4x8; sh < kShapes; sh++)
        if (const double t = shape_cost(e, d, p, sh); t < *us)
            *us = t, best = sh;
    return best;
}

template <int S, int NK, int CT>
void launch_tiles(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, int shape, hipStream_t st)
{
    if constexpr (NK <= 2 && CT <= 2) {
        if (shape == kOwn)
            return launch_shape<S, S == 1 ? 8 : 4, 8, NK, CT, true>(e, d, p, shape, st);
        if constexpr (S == 1)
            if (shape == kOwn4)
                return launch_shape<1, 4, 8, NK, CT, true>(e, d, p, shape, st);
    }
    if constexpr (S == 1 && CT <= 3) {
        if (shape == k8x8)
            return launch_shape<S, 8, 8, NK, 0, false>(e, d, p, shape, st);
        if (shape == k7x7)
            return launch_shape<S, 7, 7, NK, 0, false>(e, d, p, shape, st);
    }
    if (shape == k4x8)
        return launch_shape<S, 4, 8, NK, 0, false>(e, d, p, shape, st);
    launch_shape<S, 2, 4, NK, 0, false>(e, d, p, k2x4, st);
}

template <int S>
void launch_stride(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, int shape, hipStream_t st)
{
    const Channels c = channels_of(e, p);
    switch (c.nk * 10 + c.ct) {
    case 11: launch_tiles<S, 1, 1>(e, d, p, shape, st); break;
    case 12: launch_tiles<S, 1, 2>(e, d, p, shape, st); break;
    case 22: launch_tiles<S, 2, 2>(e, d, p, shape, st); break;
    case 23: launch_tiles<S, 2, 3>(e, d, p, shape, st); break;
    case 33: launch_tiles<S, 3, 3>(e, d, p, shape, st); break;
    case 35: launch_tiles<S, 3, 5>(e, d, p, shape, st); break;
    default: launch_tiles<S, 5, 5>(e, d, p, shape, st); break;
    }
}

bool plain(const ConvArgs &a) { return a.bwz == 0 && a.xmask != 0 && a.lo >= 0 && a.fastq && a.qmult == nullptr; }

bool point(const ConvArgs &a)
{
    return plain(a) && a.group == 1 && a.R == 1 && a.S == 1 && a.pad_h == 0 && a.pad_w == 0 && a.stride_h == 1 && a.stride_w == 1
        && a.wfrag1 != nullptr && a.in_cs % 16 == 0 && a.out_cs % 16 == 0;
}

} // namespace

bool conv_invres_applies(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p)
{
    // the residual is the block's input, which the kernel reads with the output's geometry: it has to be a tensor of that shape
    const bool same = d.stride_h == 1 && e.C == p.K && e.in_cs == p.out_cs;
    return plain(d) && d.group == d.C && d.R == 3 && d.S == 3 && d.pad_h == 1 && d.pad_w == 1 && d.stride_h == d.stride_w
        && (d.stride_h == 1 || d.stride_h == 2) && d.in_cs == d.out_cs && d.in_cs % 16 == 0 && point(p) && p.in_cs == d.in_cs && p.N == d.N
        && p.H == d.OH && p.W == d.OW && (long long)p.P * p.out_cs < (1ll << 31) && p.out_cs <= 160
        && (p.res == nullptr || (p.addq.fast && p.addq.hi == 255 && same)) && point(e) && e.out_cs == d.in_cs && e.in_cs <= 160
        && e.N == d.N && e.OH == d.H && e.OW == d.W && (long long)e.P * e.in_cs < (1ll << 31);
}

// The layers apart: the first one's latency, the last two by their own estimate (one launch where that is faster), the hidden tensor's
// bytes, the products of both 1x1 layers, fitted to the same blocks (nine in ten within 11 %).  (A fit to the three launches, less what the
// last two gain as one by the estimates of conv_dwpoint.hip, was 5 % low in the middle and 21 % at the ends: 64 -> 192 -> 16 on
// 22 images of 31x28 went apart, 10.4 -> 12.7 us.)  Less 4 %: of 900 blocks that no fit has seen 852 go the one launch's way, 8 of
// them more than 3 % slower than apart; 12 of the others would be more than 3 % faster; on average a block takes 0.3 % more than the best
// choice would.
bool conv_invres_preferred(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p)
{
    const double wide = (double)e.P * d.in_cs * 1e-6, narrow = (double)p.P * d.in_cs * 1e-6;
    double two = conv_dwpoint_apart_us(d, p);
    if (conv_dwpoint_applies(d, p))
        two = std::min(two, conv_dwpoint_us(d, p));
    const double apart = d.stride_h == 1 ? 2.991 + 0.970 * two + 0.191 * wide + 0.00277 * wide * e.in_cs + 0.00083 * narrow * p.out_cs
                                         : 2.875 + 0.993 * two + 0.195 * wide + 0.00315 * wide * e.in_cs + 0.00102 * narrow * p.out_cs;
    double us;
    choose_shape(e, d, p, -1, &us);
    return us < 0.96 * apart;
}

const char *conv_invres_name(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, int wanted)
{
    static const char *const kPatch[kShapes] = {"2x4", "4x8", "8x8", "own", "own4x8", "7x7"};
    static thread_local char nm[48];
    double us;
    const int shape = choose_shape(e, d, p, wanted, &us);
    const Channels c = channels_of(e, p);
    snprintf(nm, sizeof nm, "conv_invres_s%d_%s_k%d_n%d", d.stride_h, kPatch[shape], c.nk, c.ct);
    return nm;
}

void launch_conv_invres(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, int wanted, hipStream_t st)
{
    double us;
    const int shape = choose_shape(e, d, p, wanted, &us);
    d.stride_h == 1 ? launch_stride<1>(e, d, p, shape, st) : launch_stride<2>(e, d, p, shape, st);
}

} // namespace hipq
