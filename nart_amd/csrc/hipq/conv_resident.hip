// Convolutions whose input pixels stay in LDS while the weights go straight into registers: any stride, channel count and data type, and
// windows of up to 29 taps with less than half of the window as padding (conv_resident_applies), for the layers that have no kernel of
// their own.  gfx950 only.
//
// Reproduces op_conv_2d_u8xu8_run (art/modules/quant/src/op/conv_2d_uint8_impl.c:39-165), op_quant_ip_u8xu8_run (ip.cpp:133-209),
// their int8 variants and, with a residual, op_quant_add_run (add.c:83-148) bit for bit, like the tile kernels of conv.hip.
//
// The tile kernels walk a reduction in 64-byte steps with a barrier each and form every step's addresses anew, tap by tap; the streaming
// kernel pulls every pixel through its CU once per tap.  Both spend most of a small layer's time in instructions: a SIMD with one wave
// issues a vector instruction every 8 clocks (two waves share 4 clocks each), so a chain of 650 is 2.3 us whatever it computes.  Here
//   * a work-group owns 16 MB consecutive output pixels of the flattened (image, row, column) space and 16 NB nwc output channels.
//     The input pixels that its taps touch are one run of the flattened input, from the first tap of the first pixel to the last of the
//     last: they go to LDS once, by the load unit, without an address to form but the run's own;
//   * a tap of a pixel is then its first tap's LDS address plus a step that all lanes share, and a bit of a mask per lane sends taps
//     outside the image to a row of pad bytes: one vector instruction per operand where channels come in whole slabs;
//   * weights are loaded from the packed order into the registers of the wave that multiplies them, D slabs ahead, no barrier in
//     the loop; ks waves share every reduction (a wave's chain is an eighth as long, and all of a layer's weights are under way at
//     once), or none, where there are waves enough without;
//   * a lane's accumulators are 4 NB consecutive channels of one pixel, which leave as one store.
// What bounds it: few pixels, the weight bytes that a CU pulls from beyond its L2 (512 -> 512, 3x3, at 7x7: 73 KB, 2 us of 4.9);
// many, vector issue.  Measured on rotating weights and tensors, batch 1 unless said: 64 -> 128, 3x3 / stride 2, to 28x28 4.8 -> 3.9 us (tile
// kernel); 128 -> 128, 3x3, at 28x28 4.6 -> 4.1; 256 -> 256 at 14x14 4.6 -> 3.9; 512 -> 512 at 7x7 6.5 -> 4.9 (streaming kernel);
// 2048 -> 512, 1x1, 11 images of 7x7 8.8 -> 7.0; int8 with a scale per channel, 96 -> 200, 3x3, five images of 75x67 18.2 -> 12.3;
// 242 -> 394, 5x5 / stride 2, six images of 47x54 35 -> 20.
//
// Layers with work for every SIMD go through the same LDS rows in 32 x 32 tiles (conv_resident_wide_kernel), a launch of several
// layers in one list of work-groups (conv_resident_pair_kernel).
#include "conv_resident.h"

#include <algorithm>
#include <cmath>

#include "conv_frag.h"

namespace hipq {

namespace {

// What the waves need before their loads are under way, together at the front of the kernel's arguments
struct ResidentGeom {
    const uint8_t *x, *wpack;
    const int32_t *bias2;
    uint32_t wslab, kout_pad, padword, xmask;
    int h, w, ohw, ow, sh_w, stride_w; // sh_w: stride_h * W
    int pads;                          // pad_h * W + pad_w
    int last;                          // the tensor's last 16-byte piece
    int mtiles, ntiles, total, per_xcd;
    uint32_t m_tile;    // x / mtiles (ntiles where pixel tiles are the outer loop), x below the number of work-groups
    int mt_inner;       // 1: neighbouring work-groups share channels, 0: pixels
    int nload;          // 1 KB loads per wave
    int cpr, lpr, rb;   // 16-byte pieces of a pixel row; of its LDS row, an odd number; bytes of that
    uint32_t m_cpr, m_lpr, m_s, m_ks; // x / cpr, x / lpr, tap / S, wave / ks
    uint32_t m_ohw, m_ow1;            // m0 / (OH OW) and / OW, any m0
    int s_ohw, s_ow1;
    int ks, nwaves, nwc, per; // waves that share a reduction, waves, groups of them, slabs of a wave
    int nslab;
    uint32_t m_ow, m_oh; // x / OW and / OH, small x
    int oh, pad_h, pad_w, stride_h, P, R, S;
    uint32_t taprows; // bit S i: the first tap of row i
};

typedef const __attribute__((address_space(1))) uint8_t *gbytes_t;
typedef const __attribute__((address_space(1))) v4i *gv4i_t;

// x / d for x d < 2^31 with m from magic(d)
__device__ static inline uint32_t quot(uint32_t x, uint32_t m) { return __umulhi(x << 1, m); }

// x / d for any x below 2^31 (hipq_div_magic)
__device__ static inline uint32_t quot_any(uint32_t x, uint32_t m, int s) { return m ? __umulhi(x, m) >> s : x; }

// How a slab of the reduction finds its pixels.  kPoint: 1x1 / stride 1, one row for all; kWhole: channel strides that are multiples of
// 64, where a slab lies in one tap; kPieces: any multiple of 16, where each of a slab's four pieces has a tap of its own.
enum Gather { kPoint, kWhole, kPieces };

// What becomes of the sums.  kTensor: uint8, one scale, one-multiply requantisation to a range within [0, 255]; kChannels: one-multiply
// requantisation with a scale per channel or to a signed range; kAny: every option, among them weight zero points other than 128,
// accumulators and floats to write.
enum Finish { kTensor, kChannels, kAny };

} // namespace

// The tile gid of a layer.  SPLIT: several waves share a reduction
template <int MB, int NB, bool SPLIT, int GATHER, int FINISH>
__device__ static __forceinline__ void resident_tile(const ResidentGeom &geo, const ConvArgs &a, const int gid, uint8_t *const lds)
{
    constexpr int D = NB == 1 ? (MB == 1 ? 9 : 8) : NB == 2 && MB < 8 ? 6 : FINISH == kTensor || MB < 8 ? 4 : 2; // slabs of weights ahead
    constexpr int XD = MB == 1 ? 3 : 2; // slabs of pixel operands, the present one among them
    constexpr bool CENTRE = GATHER != kPoint && !SPLIT; // re-centre the region in LDS, not every operand
    static_assert(D % XD == 0, "ring positions");
    // all of geo at once: the compiler would load it piece by piece as it is used, a round trip each
    asm volatile("" ::"s"(geo.x), "s"(geo.wpack), "s"(geo.bias2), "s"(geo.wslab), "s"(geo.xmask), "s"(geo.h), "s"(geo.sh_w), "s"(geo.last), "s"(geo.total), "s"(geo.nload), "s"(geo.rb),
                 "s"(geo.m_ks), "s"(geo.m_ohw), "s"(geo.per), "s"(geo.oh), "s"(geo.taprows));

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = geo.nwaves;
    const int r = lane & 15, q = lane >> 4;
    if (gid >= geo.total)
        return;
    const int outer = (int)quot(gid, geo.m_tile), inner = gid - outer * (geo.mt_inner ? geo.mtiles : geo.ntiles);
    const int mt = geo.mt_inner ? inner : outer, nt = geo.mt_inner ? outer : inner;
    const int cg = (int)quot(wave, geo.m_ks), kslice = wave - cg * geo.ks;
    const int m0 = mt * (16 * MB), n0 = (nt * geo.nwc + cg) * (16 * NB);

    // ---- the first pixel's position; the region starts at its first tap
    int img0 = 0, oh0 = 0, ow0 = 0, q0 = m0;
    if (GATHER != kPoint) {
        img0 = (int)quot_any((uint32_t)m0, geo.m_ohw, geo.s_ohw);
        const int rem0 = m0 - img0 * geo.ohw;
        oh0 = (int)quot_any((uint32_t)rem0, geo.m_ow1, geo.s_ow1), ow0 = rem0 - oh0 * geo.ow;
        q0 = img0 * geo.h * geo.w + oh0 * geo.sh_w + ow0 * geo.stride_w - geo.pads;
    }

    // ---- the region -> LDS, behind a row of pad bytes that stands for the taps outside the image.  LDS rows of an odd number of
    // pieces: 16 pixels' reads of one piece fall on 16 different bank groups.  The pieces that fill the rows up are never read, nor
    // are rows that are not in the tensor: any piece of it will do for them
    if (GATHER != kPoint) {
        const int pad = (int)(CENTRE ? geo.padword ^ geo.xmask : geo.padword);
        for (int c = tid; c < geo.cpr; c += 64 * nwaves)
            *reinterpret_cast<v4i *>(lds + c * 16) = v4i{pad, pad, pad, pad};
    }
    uint8_t *const own = lds + geo.rb + wave * 1024;
    for (int k = 0; k < geo.nload; k++) {
        const int id = (k * nwaves + wave) * 64 + lane, row = (int)quot(id, geo.m_lpr), c = min(id - row * geo.lpr, geo.cpr - 1);
        const uint32_t off = (uint32_t)min(max((q0 + row) * geo.cpr + c, 0), geo.last) * 16;
        __builtin_amdgcn_global_load_lds((gptr_t)(geo.x + off), (lptr_t)(own + k * nwaves * 1024), 16, 0, 0);
    }

    // ---- this wave's slabs of the reduction; weights: row i of a channel tile computes channel 4 NB (i >> 2) + 4 nb + (i & 3) of the
    // wave's 16 NB, so that a lane's accumulators are 4 NB consecutive channels of one pixel
    const int s0 = min(kslice * geo.per, geo.nslab - 1), cnt = min(geo.per, geo.nslab - kslice * geo.per); // none where that is negative
    uint32_t woff[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const int ch = min(n0 + 4 * NB * (r >> 2) + 4 * nb + (r & 3), (int)geo.kout_pad - 1);
        woff[nb] = (uint32_t)(ch * 64 + ((q ^ ((ch >> 2) & 3)) << 4));
    }
    v4i w[D][NB];
    uint64_t wnext = (uint64_t)geo.wpack + (uint64_t)(uint32_t)s0 * geo.wslab;
    auto load_w = [&](v4i(&to)[NB]) { // the next slab
        asm("" : "+s"(wnext));        // the base stays in scalar registers
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
            to[nb] = *reinterpret_cast<gv4i_t>(reinterpret_cast<gbytes_t>(wnext) + woff[nb]);
        wnext += geo.wslab;
    };
    v4i acc[MB][NB], bias[NB];
    const int clane = min(n0 + 4 * NB * q, (int)geo.kout_pad - 4 * NB); // this lane's channels, where it has any
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
        bias[nb] = *reinterpret_cast<const v4i *>(geo.bias2 + clane + 4 * nb);
#pragma unroll
    for (int i = 0; i < D; i++)
        if (i < cnt)
            load_w(w[i]);
    // what the epilogue needs of the arguments, while the loads are under way
    asm volatile("" ::"s"(a.y), "s"(a.out_cs), "s"(a.q.mult), "s"(a.lo), "s"(a.qadd), "s"(a.qmult), "s"(a.res), "s"(a.addq.m0), "s"(a.addq.c0));

    // ---- this lane's pixels m0 + 16 mb + r: the LDS address of their first tap, and which taps lie inside the image
    uint32_t base[MB], mask[GATHER == kPoint ? 1 : MB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        const int m = min(m0 + 16 * mb + r, geo.P - 1) - m0;
        if (GATHER == kPoint) {
            base[mb] = __umul24(m + 1, geo.rb) + 16 * q;
            continue;
        }
        const int xq = ow0 + m, dy = (int)quot(xq, geo.m_ow), ow = xq - dy * geo.ow;
        const int yq = oh0 + dy, dn = (int)quot(yq, geo.m_oh), oh = yq - dn * geo.oh;
        const int ih = oh * geo.stride_h - geo.pad_h, iw = ow * geo.stride_w - geo.pad_w;
        base[mb] = (uint32_t)((((img0 + dn) * geo.h + ih) * geo.w + iw - q0 + 1) * geo.rb) + (GATHER == kWhole ? 16 * q : 0);
        // the columns of one row of taps, once for every row of them: column bits times the first bits of the rows
        const uint32_t cols = (1u << min(geo.S, geo.w - iw)) - (1u << max(0, -iw));
        const uint32_t rows = geo.taprows & ((1u << (min(geo.R, geo.h - ih) * geo.S)) - (1u << (max(0, -ih) * geo.S)));
        mask[mb] = cols * rows;
    }
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
            acc[mb][nb] = kslice == 0 ? bias[nb] : v4i{0, 0, 0, 0};
    const bool has_wzp = FINISH == kAny && a.bwz != 0;
    v4i xsum[FINISH == kAny ? MB : 1];
    if (FINISH == kAny)
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
            xsum[mb] = v4i{0, 0, 0, 0};
    if (CENTRE && geo.xmask != 0) {
        // taps read a pixel several times: each wave re-centres its share of the region once, in LDS
        wait_vmcnt<0>();
        for (int k = 0; k < geo.nload; k++) {
            v4i *at = reinterpret_cast<v4i *>(own + k * nwaves * 1024 + lane * 16);
            *at ^= (int)geo.xmask;
        }
    }
    wait_vmcnt<0>(); // this wave's loads have landed before the others may read them: a barrier alone says nothing of the load unit's writes
    __syncthreads();

    // ---- a slab's pixel operands
    const uint32_t xmask = CENTRE ? 0u : geo.xmask;
    int tap = GATHER == kWhole ? (int)quot((uint32_t)(4 * s0), geo.m_cpr) : 0; // of the next slab
    int cu = GATHER == kPieces ? s0 : 64 * s0 - tap * geo.cpr * 16;           // its first byte in its tap; kPieces: its number
    uint32_t at[MB];
    auto enter_tap = [&]() {
        const int step = ((int)quot((uint32_t)tap, geo.m_s) * (geo.w - geo.S) + tap) * geo.rb;
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
            at[mb] = GATHER == kPoint ? base[mb] : (int)(mask[mb] << (31 - tap)) < 0 ? base[mb] + step : (uint32_t)(16 * q);
    };
    if (GATHER != kPieces)
        enter_tap();
    v4i x[XD][MB];
    auto load_x = [&](v4i(&to)[MB]) { // the next slab's; behind the last one whatever its address names
        if (GATHER != kPieces) {
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
                to[mb] = *reinterpret_cast<const v4i *>(lds + (at[mb] + cu));
            cu = GATHER == kPoint ? min(cu + 64, geo.cpr * 16 - 64) : cu + 64;
            if (GATHER == kWhole && cu == geo.cpr * 16) {
                cu = 0, tap++;
                enter_tap();
            }
            return;
        }
        const int kp = 4 * cu + q, tp = (int)quot((uint32_t)kp, geo.m_cpr);
        const int step = (int)quot((uint32_t)tp, geo.m_s) * (geo.w - geo.S) + tp;
        const uint32_t off = (uint32_t)(step * geo.rb + 16 * (kp - tp * geo.cpr));
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
            to[mb] = *reinterpret_cast<const v4i *>(lds + ((int)(mask[mb] << (31 - tp)) < 0 ? base[mb] + off : 0u));
        cu = min(cu + 1, geo.nslab - 1);
    };
    auto multiply = [&](const v4i(&wf)[NB], const v4i(&xf)[MB]) {
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
            const v4i xs = xf[mb] ^ (int)xmask;
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
                acc[mb][nb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[nb], xs, acc[mb][nb], 0, 0, 0);
            if (has_wzp)
                xsum[mb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{0x01010101, 0x01010101, 0x01010101, 0x01010101}, xs, xsum[mb], 0, 0, 0);
        }
    };
#pragma unroll
    for (int i = 0; i + 1 < XD; i++)
        load_x(x[i]);
    int i0 = 0;
    for (; i0 + 2 * D <= cnt; i0 += D)
#pragma unroll
        for (int j = 0; j < D; j++) {
            load_x(x[(j + XD - 1) % XD]);
            multiply(w[j], x[j % XD]);
            load_w(w[j]);
            __builtin_amdgcn_sched_barrier(0);
        }
    for (; i0 < cnt; i0 += D)
#pragma unroll
        for (int j = 0; j < D; j++) {
            if (i0 + j < cnt) {
                load_x(x[(j + XD - 1) % XD]);
                multiply(w[j], x[j % XD]);
                if (i0 + j + D < cnt)
                    load_w(w[j]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    if (has_wzp)
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    acc[mb][nb][e] = (int32_t)((uint32_t)acc[mb][nb][e] + (uint32_t)a.bwz * (uint32_t)xsum[mb][e]);

    // ---- a tile's bytes: this lane's 4 NB consecutive channels of pixel m
    v4i qm[FINISH == kChannels ? NB : 1], qt[FINISH == kChannels ? NB : 1], qr[FINISH == kChannels ? NB : 1]; // multiplier, shift, rounding and zero point
    auto channels = [&]() {
        if (FINISH != kChannels)
            return;
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            if (a.qmult != nullptr) {
                qm[nb] = *reinterpret_cast<const v4i *>(a.qmult + clane + 4 * nb);
                qt[nb] = *reinterpret_cast<const v4i *>(a.qshift + clane + 4 * nb) - 32;
            } else {
                qm[nb] = v4i{(int)a.q.mult, (int)a.q.mult, (int)a.q.mult, (int)a.q.mult}, qt[nb] = v4i{a.qt, a.qt, a.qt, a.qt};
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
                qr[nb][e] = (2 * a.q.zp + 1) << (qt[nb][e] - 1);
        }
    };
    auto finish = [&](int mb, const v4i(&s)[NB]) {
        const int m = m0 + 16 * mb + r, c0 = n0 + 4 * NB * q;
        if (m >= geo.P)
            return;
        uint32_t out[NB];
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            const int ch = c0 + 4 * nb;
            if (ch >= a.out_cs)
                break;
            if (FINISH == kTensor) {
                out[nb] = a.lo == 0 && a.q.hi == 255 ? conv_requant4<true>(a, s[nb][0], s[nb][1], s[nb][2], s[nb][3])
                                                     : conv_requant4<false>(a, s[nb][0], s[nb][1], s[nb][2], s[nb][3]);
            } else {
                if (FINISH == kAny && a.acc_out != nullptr)
                    *reinterpret_cast<v4i *>(a.acc_out + (size_t)m * a.out_cs + ch) = s[nb];
                int32_t rq[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (FINISH == kChannels) {
                        const int32_t v = (__mulhi(s[nb][e], qm[nb][e]) + qr[nb][e]) >> qt[nb][e];
                        rq[e] = min(max(v, a.lo), a.q.hi);
                    } else {
                        rq[e] = a.qmult ? conv_requant_ch(a, s[nb][e], ch + e) : a.fastq ? conv_requant<true>(a, s[nb][e]) : conv_requant<false>(a, s[nb][e]);
                    }
                }
                if (FINISH == kAny && a.deq_out != nullptr) { // fused dequantize (op_dequantize_run_u8, art/modules/quant/src/op/dequantize.c:111-123)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (ch + e < a.K)
                            a.deq_out[(size_t)m * a.K + ch + e] = __fmul_rn((float)(rq[e] - a.q.zp), a.deq_alpha);
                    continue;
                }
                out[nb] = pack_low_bytes(rq[0], rq[1], rq[2], rq[3]);
            }
            if (a.res != nullptr) { // fused residual add: exactly what the add operator computes from the convolution's stored bytes
                const uint32_t rv = *reinterpret_cast<const uint32_t *>(a.res + (size_t)m * a.out_cs + ch);
                const uint32_t first = a.res_first ? rv : out[nb], second = a.res_first ? out[nb] : rv;
                out[nb] = a.addq.fast ? add_dword<true>(first, second, a.addq) : add_dword<false>(first, second, a.addq);
            }
        }
        if (FINISH == kAny && a.deq_out != nullptr)
            return;
        uint8_t *to = a.y + (size_t)m * a.out_cs + c0;
        if (NB > 1 && (a.out_cs & (4 * NB - 1)) == 0) {
            if (c0 < a.out_cs) {
                if constexpr (NB == 4)
                    *reinterpret_cast<u32x4 *>(to) = u32x4{out[0], out[1], out[2], out[3]};
                else if constexpr (NB == 2)
                    *reinterpret_cast<uint2 *>(to) = make_uint2(out[0], out[1]);
            }
        } else {
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
                if (c0 + 4 * nb < a.out_cs)
                    *reinterpret_cast<uint32_t *>(to + 4 * nb) = out[nb];
        }
    };
    channels();
    if (!SPLIT) {
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
            finish(mb, acc[mb]);
        return;
    }
    // ---- partial sums meet in LDS where the region was
    __syncthreads();
    v4i *const red = reinterpret_cast<v4i *>(lds);
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
            red[((wave * MB + mb) * NB + nb) * 64 + lane] = acc[mb][nb];
    __syncthreads();
    for (int mb = kslice; mb < MB; mb += geo.ks) {
        v4i s[NB];
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
            s[nb] = v4i{0, 0, 0, 0};
        for (int k = 0; k < geo.ks; k++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
                s[nb] += red[(((cg * geo.ks + k) * MB + mb) * NB + nb) * 64 + lane];
        finish(mb, s);
    }
}

// work-groups go to the 8 XCDs in turn: XCD x takes the x-th contiguous eighth of a layer's list
template <int MB, int NB, bool SPLIT, int GATHER, int FINISH>
__global__ __launch_bounds__(512) void conv_resident_kernel(const ResidentGeom geo, const ConvArgs a)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    resident_tile<MB, NB, SPLIT, GATHER, FINISH>(geo, a, (int)(blockIdx.x % 8) * geo.per_xcd + (int)(blockIdx.x / 8), lds);
}

// The same with 32 x 32 tiles, for layers with work for every SIMD: a wave owns 32 MT pixels by 32 NT channels and the whole reduction.
// Both tile sizes multiply at the same rate, but the larger needs half of the operand bytes for it: MT pixel operands of LDS and NT
// weight operands per MT NT multiplies.  In the loop the matrix pipe bounds it (on operands of random bytes a SIMD gives one such multiply
// per 49 clocks); the rest is the fill of LDS before it and the requantisation behind it, which another
// work-group of the CU fills where LDS holds two.  Signed and per-channel results leave through
// the saturating pack of two pixels of a channel.  Measured on rotating tensors, before (the 16 x 16 form or the tile kernel) -> after:
// 46 -> 83, 3x3, 26 images of 101x103 39 -> 24.7 us; 16 -> 16, 3x3, 62 images of 134x182 60 -> 26; int8 with a scale per channel, 96 -> 200,
// 3x3, five images of 75x67 14.2 -> 12.4; 1x1 with a scale per channel 28 -> 16.
template <int MT, int NT, int GATHER, int FINISH>
__global__ __launch_bounds__(512, 2) void conv_resident_wide_kernel(const ResidentGeom geo, const ConvArgs a)
{
    constexpr int D = MT * NT == 8 ? 6 : 8; // steps of weights ahead, two a slab
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    asm volatile("" ::"s"(geo.x), "s"(geo.wpack), "s"(geo.bias2), "s"(geo.wslab), "s"(geo.xmask), "s"(geo.h), "s"(geo.sh_w), "s"(geo.last), "s"(geo.total), "s"(geo.nload), "s"(geo.rb),
                 "s"(geo.m_ohw), "s"(geo.oh), "s"(geo.taprows));
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = geo.nwaves;
    const int p = lane & 31, h = lane >> 5;
    const int gid = (int)(blockIdx.x % 8) * geo.per_xcd + (int)(blockIdx.x / 8);
    if (gid >= geo.total)
        return;
    const int outer = (int)quot(gid, geo.m_tile), inner = gid - outer * (geo.mt_inner ? geo.mtiles : geo.ntiles);
    const int mt = geo.mt_inner ? inner : outer, nt = geo.mt_inner ? outer : inner;
    const int m0 = mt * (32 * MT), n0 = (nt * nwaves + wave) * (32 * NT);

    // ---- the region -> LDS, as above
    const int img0 = (int)quot_any((uint32_t)m0, geo.m_ohw, geo.s_ohw);
    const int rem0 = m0 - img0 * geo.ohw;
    const int oh0 = (int)quot_any((uint32_t)rem0, geo.m_ow1, geo.s_ow1), ow0 = rem0 - oh0 * geo.ow;
    const int q0 = img0 * geo.h * geo.w + oh0 * geo.sh_w + ow0 * geo.stride_w - geo.pads;
    {
        const int pad = (int)(geo.padword ^ geo.xmask);
        for (int c = tid; c < geo.cpr; c += 64 * nwaves)
            *reinterpret_cast<v4i *>(lds + c * 16) = v4i{pad, pad, pad, pad};
    }
    uint8_t *const own = lds + geo.rb + wave * 1024;
    for (int k = 0; k < geo.nload; k++) {
        const int id = (k * nwaves + wave) * 64 + lane, row = (int)quot(id, geo.m_lpr), c = min(id - row * geo.lpr, geo.cpr - 1);
        const uint32_t off = (uint32_t)min(max((q0 + row) * geo.cpr + c, 0), geo.last) * 16;
        __builtin_amdgcn_global_load_lds((gptr_t)(geo.x + off), (lptr_t)(own + k * nwaves * 1024), 16, 0, 0);
    }

    // ---- weights: row i of a channel tile computes channel 16 ((i >> 2) & 1) + 4 (i >> 3) + (i & 3), so that a lane's accumulators are 16
    // consecutive channels of one pixel
    uint32_t woff[NT][2];
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const int ch = min(n0 + 32 * n + 16 * ((p >> 2) & 1) + 4 * (p >> 3) + (p & 3), (int)geo.kout_pad - 1);
#pragma unroll
        for (int kk = 0; kk < 2; kk++)
            woff[n][kk] = (uint32_t)(ch * 64 + (((2 * kk + h) ^ ((ch >> 2) & 3)) << 4));
    }
    v4i w[D][NT];
    uint64_t wnext = (uint64_t)geo.wpack;
    auto load_w = [&](v4i(&to)[NT], int kk) {
        asm("" : "+s"(wnext));
#pragma unroll
        for (int n = 0; n < NT; n++)
            to[n] = *reinterpret_cast<gv4i_t>(reinterpret_cast<gbytes_t>(wnext) + woff[n][kk]);
        wnext += kk ? geo.wslab : 0;
    };
    const int steps = geo.per;
    v16i acc[NT][MT];
    int clane[NT]; // this lane's channels, where it has any
#pragma unroll
    for (int n = 0; n < NT; n++) {
        clane[n] = min(n0 + 32 * n + 16 * h, (int)geo.kout_pad - 16);
        frag::init_acc(acc[n][0], geo.bias2 + clane[n], false);
#pragma unroll
        for (int t = 1; t < MT; t++)
            acc[n][t] = acc[n][0];
    }
#pragma unroll
    for (int i = 0; i < D; i++)
        if (i < steps)
            load_w(w[i], i & 1);
    // a channel's scale each: here, where they are, not behind the reduction, a round trip later
    constexpr bool EARLY = FINISH == kChannels && NT == 1;
    v4i qm_[EARLY ? 4 : 1], qt_[EARLY ? 4 : 1];
    if (EARLY && a.qmult != nullptr)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            qm_[g] = *reinterpret_cast<const v4i *>(a.qmult + clane[0] + 4 * g);
            qt_[g] = *reinterpret_cast<const v4i *>(a.qshift + clane[0] + 4 * g);
        }
    asm volatile("" ::"s"(a.y), "s"(a.out_cs), "s"(a.q.mult), "s"(a.lo), "s"(a.qadd), "s"(a.qmult), "s"(a.res), "s"(a.addq.m0), "s"(a.addq.c0));

    // ---- this lane's pixels m0 + 32 t + p, as above
    uint32_t base[MT], mask[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int m = min(m0 + 32 * t + p, geo.P - 1) - m0;
        const int xq = ow0 + m, dy = (int)quot(xq, geo.m_ow), ow = xq - dy * geo.ow;
        const int yq = oh0 + dy, dn = (int)quot(yq, geo.m_oh), oh = yq - dn * geo.oh;
        const int ih = oh * geo.stride_h - geo.pad_h, iw = ow * geo.stride_w - geo.pad_w;
        base[t] = (uint32_t)((((img0 + dn) * geo.h + ih) * geo.w + iw - q0 + 1) * geo.rb) + (GATHER == kWhole ? 16 * h : 0);
        const uint32_t cols = (1u << min(geo.S, geo.w - iw)) - (1u << max(0, -iw));
        const uint32_t rows = geo.taprows & ((1u << (min(geo.R, geo.h - ih) * geo.S)) - (1u << (max(0, -ih) * geo.S)));
        mask[t] = cols * rows;
    }
    wait_vmcnt<0>(); // this wave's loads have landed
    if (geo.xmask != 0)
        for (int k = 0; k < geo.nload; k++) {
            v4i *at = reinterpret_cast<v4i *>(own + k * nwaves * 1024 + lane * 16);
            *at ^= (int)geo.xmask;
        }
    __syncthreads();

    // ---- a step's pixel operands: 32 bytes of the reduction.  kWhole: channel strides that are multiples of 32, where a step lies in one
    // tap; kPieces: each half of it has a tap of its own
    int tap = 0, cu = 0; // kPieces: cu is the step
    uint32_t at[MT];
    auto enter_tap = [&]() {
        const int step = ((int)quot((uint32_t)tap, geo.m_s) * (geo.w - geo.S) + tap) * geo.rb;
#pragma unroll
        for (int t = 0; t < MT; t++)
            at[t] = (int)(mask[t] << (31 - tap)) < 0 ? base[t] + step : (uint32_t)(16 * h);
    };
    if (GATHER == kWhole)
        enter_tap();
    v4i x[2][MT];
    auto load_x = [&](v4i(&to)[MT]) { // the next step's; behind the last one whatever its address names
        if (GATHER == kWhole) {
#pragma unroll
            for (int t = 0; t < MT; t++)
                to[t] = *reinterpret_cast<const v4i *>(lds + (at[t] + cu));
            cu += 32;
            if (cu == geo.cpr * 16) {
                cu = 0, tap++;
                enter_tap();
            }
            return;
        }
        const int kp = 2 * cu + h, tp = (int)quot((uint32_t)kp, geo.m_cpr);
        const int step = (int)quot((uint32_t)tp, geo.m_s) * (geo.w - geo.S) + tp;
        const uint32_t off = (uint32_t)(step * geo.rb + 16 * (kp - tp * geo.cpr));
#pragma unroll
        for (int t = 0; t < MT; t++)
            to[t] = *reinterpret_cast<const v4i *>(lds + ((int)(mask[t] << (31 - tp)) < 0 ? base[t] + off : 0u));
        cu = min(cu + 1, steps - 1);
    };
    auto multiply = [&](const v4i(&wf)[NT], const v4i(&xf)[MT]) {
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int t = 0; t < MT; t++)
                acc[n][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[n], xf[t], acc[n][t], 0, 0, 0);
    };
    load_x(x[0]);
    int i0 = 0;
    for (; i0 + 2 * D <= steps; i0 += D)
#pragma unroll
        for (int j = 0; j < D; j++) {
            load_x(x[(j + 1) & 1]);
            multiply(w[j], x[j & 1]);
            load_w(w[j], j & 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    for (; i0 < steps; i0 += D)
#pragma unroll
        for (int j = 0; j < D; j++) {
            if (i0 + j < steps) {
                load_x(x[(j + 1) & 1]);
                multiply(w[j], x[j & 1]);
                if (i0 + j + D < steps)
                    load_w(w[j], j & 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        }

    // ---- bytes: 16 consecutive channels of a pixel
    auto store = [&](int t, int c0, const v4i &o) {
        const int m = m0 + 32 * t + p;
        if (m < geo.P && c0 < a.out_cs)
            *reinterpret_cast<v4i *>(a.y + (size_t)m * a.out_cs + c0) = o;
    };
    if constexpr (FINISH == kTensor) {
#pragma unroll
        for (int n = 0; n < NT; n++) {
            const int c0 = n0 + 32 * n + 16 * h;
            if (a.res == nullptr) {
#pragma unroll
                for (int t = 0; t < MT; t++)
                    store(t, c0, frag::requant16(a, acc[n][t], 0));
            } else { // the 32-bit form of the add to 8 bits (wide_applies)
                v4i res[MT];
#pragma unroll
                for (int t = 0; t < MT; t++)
                    res[t] = ldg128(a.res + (size_t)min(m0 + 32 * t + p, geo.P - 1) * a.out_cs + min(c0, a.out_cs - 16));
#pragma unroll
                for (int t = 0; t < MT; t++)
                    store(t, c0, frag::requant_add16(a, acc[n][t], res[t]));
            }
        }
    } else {
        // The clamp from below in front of the shift, then the shifting, saturating pack on two pixels of ONE channel, whose shift is the same:
        // a multiply-add, a maximum and three quarters of a byte permutation a value beside half a pack
        auto channels = [&](auto sgn) {
#pragma unroll
            for (int n = 0; n < NT; n++) {
                v4i out[MT];
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    v4i qm, qt;
                    if (a.qmult != nullptr) {
                        qm = EARLY ? qm_[EARLY ? g : 0] : *reinterpret_cast<const v4i *>(a.qmult + clane[n] + 4 * g);
                        qt = (EARLY ? qt_[EARLY ? g : 0] : *reinterpret_cast<const v4i *>(a.qshift + clane[n] + 4 * g)) - 32;
                    } else {
                        qm = v4i{(int)a.q.mult, (int)a.q.mult, (int)a.q.mult, (int)a.q.mult}, qt = v4i{a.qt, a.qt, a.qt, a.qt};
                    }
                    uint32_t two[4][MT / 2]; // bytes 0 and 1 of a channel's two pixels
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        uint64_t add = (uint64_t)(uint32_t)((2 * a.q.zp + 1) << (qt[e] - 1)) << 32; // rounding and zero point
                        asm("" : "+v"(add));
                        const int32_t plo = a.lo << qt[e];
#pragma unroll
                        for (int t = 0; t < MT / 2; t++) {
                            int32_t v[2];
#pragma unroll
                            for (int u = 0; u < 2; u++)
                                v[u] = max(mulhi_add(acc[n][2 * t + u][4 * g + e], (uint32_t)qm[e], add), plo);
                            if (decltype(sgn)::value)
                                asm("v_ashr_pk_i8_i32 %0, %1, %2, %3" : "=v"(two[e][t]) : "v"(v[0]), "v"(v[1]), "v"(qt[e]));
                            else
                                asm("v_ashr_pk_u8_i32 %0, %1, %2, %3" : "=v"(two[e][t]) : "v"(v[0]), "v"(v[1]), "v"(qt[e]));
                        }
                    }
#pragma unroll
                    for (int t = 0; t < MT / 2; t++) {
                        out[2 * t][g] = (int)(__builtin_amdgcn_perm(two[1][t], two[0][t], 0x0c0c0400u) | __builtin_amdgcn_perm(two[3][t], two[2][t], 0x04000c0cu));
                        out[2 * t + 1][g] = (int)(__builtin_amdgcn_perm(two[1][t], two[0][t], 0x0c0c0501u) | __builtin_amdgcn_perm(two[3][t], two[2][t], 0x05010c0cu));
                    }
                }
#pragma unroll
                for (int t = 0; t < MT; t++)
                    store(t, n0 + 32 * n + 16 * h, out[t]);
            }
        };
        if (a.lo < 0)
            channels(std::true_type{});
        else
            channels(std::false_type{});
    }
}

namespace {

struct PairArgs {
    ResidentGeom geo;
    ConvArgs a;
};

} // namespace

// Two layers that do not depend on each other in one launch: the first work-groups of every XCD take the first layer's tiles.  What it is
// for is a block's 3x3 / stride 2 layer and its 1x1 shortcut on few images, each a launch's latency and little else: 64 -> 128 channels at
// 56x56, one image, 6.8 us as two launches, 5.1 as one; 256 -> 512 at 14x14 7.1 and 4.9; ResNet-18 at batch 1, three such pairs, 97.3 ->
// 88.4 us.  Bound by the larger layer's chain of pixels, weights and sums.
template <int MB, int NB, bool SPLIT>
__global__ __launch_bounds__(512) void conv_resident_pair_kernel(const PairArgs first, const PairArgs second)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int xcd = (int)(blockIdx.x % 8), i = (int)(blockIdx.x / 8);
    const bool behind = i >= first.geo.per_xcd;
    const PairArgs &k = ((const PairArgs *)__builtin_amdgcn_kernarg_segment_ptr())[behind ? 1 : 0]; // by address: no select per argument
    resident_tile<MB, NB, SPLIT, kWhole, kTensor>(k.geo, k.a, xcd * k.geo.per_xcd + i - (behind ? first.geo.per_xcd : 0), lds);
}

namespace {

uint32_t magic(int d) { return (uint32_t)(((1ull << 31) + d - 1) / d); }

// pixel rows that the taps of 16 mb consecutive output pixels span at most (the first tap of the first to the last of the last)
int region_rows(const ConvArgs &a, int mb)
{
    const long long t = std::min(16 * mb, a.P) - 1, turns = std::min<long long>(t, (t + a.OW - 1) / a.OW), imgs = std::min<long long>(turns, (t + a.OH * a.OW - 1) / (a.OH * a.OW));
    const long long row = (long long)a.stride_h * a.W - (long long)(a.OW - 1) * a.stride_w; // from the last pixel of a row to the next one
    const long long img = (long long)a.H * a.W - (long long)(a.OH - 1) * a.stride_h * a.W - (long long)(a.OW - 1) * a.stride_w;
    long long span = (t - turns) * a.stride_w + (turns - imgs) * std::max<long long>(row, a.stride_w) + imgs * std::max({row, img, (long long)a.stride_w});
    span += (long long)(a.R - 1) * a.W + a.S;
    return (int)std::min<long long>(span, 1 << 20);
}

// bytes of a pixel's LDS row: an odd number of 16-byte pieces
int lds_row(const ConvArgs &a) { return 16 * (a.in_cs / 16 | 1); }

int waves_of(const ResidentShape &s) { return s.nwc * std::max(s.ks, 1); }

int lds_bytes(const ConvArgs &a, const ResidentShape &s)
{
    const int chunk = waves_of(s) * 1024;
    const long long row = lds_row(a), region = row + (region_rows(a, s.mb) * row + chunk - 1) / chunk * chunk;
    const long long red = s.ks > 1 ? (long long)chunk * s.mb * s.nb : 0;
    return (int)std::min<long long>(std::max(region, red), 1 << 30);
}

long long tiles(const ConvArgs &a, const ResidentShape &s)
{
    const long long m = (a.P + 16 * s.mb - 1) / (16 * s.mb), n = (a.out_cs + 16 * s.nb * s.nwc - 1) / (16 * s.nb * s.nwc);
    return m * n * std::max(m, n);
}

ResidentGeom geometry(const ConvArgs &a, const ResidentShape &s)
{
    const int MB = s.mb, NB = s.nb, nw = waves_of(s);
    ResidentGeom g;
    g.x = a.x, g.wpack = a.wpack, g.bias2 = a.bias2;
    g.wslab = (uint32_t)a.kout_pad * 64, g.kout_pad = (uint32_t)a.kout_pad, g.padword = a.padword, g.xmask = a.xmask;
    g.h = a.H, g.w = a.W, g.ohw = a.OH * a.OW, g.ow = a.OW, g.sh_w = a.stride_h * a.W, g.stride_w = a.stride_w, g.pads = a.pad_h * a.W + a.pad_w;
    g.cpr = a.in_cs / 16, g.rb = lds_row(a), g.lpr = g.rb / 16, g.last = a.N * a.H * a.W * g.cpr - 1;
    g.mtiles = (a.P + 16 * MB - 1) / (16 * MB), g.ntiles = (a.out_cs + 16 * NB * s.nwc - 1) / (16 * NB * s.nwc);
    g.total = g.mtiles * g.ntiles, g.per_xcd = (g.total + 7) / 8;
    g.mt_inner = (long long)a.nslab * 64 * a.out_cs > (long long)a.N * a.H * a.W * a.in_cs;
    g.m_tile = magic(g.mt_inner ? g.mtiles : g.ntiles);
    g.nload = (region_rows(a, MB) * g.rb + nw * 1024 - 1) / (nw * 1024);
    g.m_cpr = magic(g.cpr), g.m_lpr = magic(g.lpr), g.m_s = magic(a.S), g.m_ks = magic(std::max(s.ks, 1));
    hipq_div_magic((uint32_t)(a.OH * a.OW), &g.m_ohw, &g.s_ohw);
    hipq_div_magic((uint32_t)a.OW, &g.m_ow1, &g.s_ow1);
    g.m_ow = magic(a.OW), g.m_oh = magic(a.OH);
    g.ks = s.ks, g.nwaves = nw, g.nwc = s.nwc, g.per = s.ks ? (a.nslab + s.ks - 1) / s.ks : (a.Ktot + 31) / 32, g.nslab = a.nslab;
    g.oh = a.OH, g.pad_h = a.pad_h, g.pad_w = a.pad_w, g.stride_h = a.stride_h, g.P = a.P, g.R = a.R, g.S = a.S;
    g.taprows = 0;
    for (int i = 0; i < a.R; i++)
        g.taprows |= 1u << (i * a.S);
    return g;
}

template <int MB, int NB, bool SPLIT>
void launch_shape(const ConvArgs &a, const ResidentShape &s, hipStream_t st)
{
    const int nw = s.nwc * s.ks, lds = lds_bytes(a, s);
    const ResidentGeom g = geometry(a, s);
    const dim3 grid((unsigned)(g.per_xcd * 8)), block(64 * nw);
    if (a.bwz != 0 || a.acc_out != nullptr || a.deq_out != nullptr || !(a.qmult != nullptr ? a.fastch : a.fastq))
        hipLaunchKernelGGL((conv_resident_kernel<MB, NB, SPLIT, kPieces, kAny>), grid, block, lds, st, g, a);
    else if (a.qmult != nullptr || a.lo < 0)
        hipLaunchKernelGGL((conv_resident_kernel<MB, NB, SPLIT, kPieces, kChannels>), grid, block, lds, st, g, a);
    else if (a.R == 1 && a.S == 1 && a.stride_h == 1 && a.stride_w == 1 && a.in_cs % 64 == 0)
        hipLaunchKernelGGL((conv_resident_kernel<MB, NB, SPLIT, kPoint, kTensor>), grid, block, lds, st, g, a);
    else if (a.in_cs % 64 == 0)
        hipLaunchKernelGGL((conv_resident_kernel<MB, NB, SPLIT, kWhole, kTensor>), grid, block, lds, st, g, a);
    else
        hipLaunchKernelGGL((conv_resident_kernel<MB, NB, SPLIT, kPieces, kTensor>), grid, block, lds, st, g, a);
}

template <int MT, int NT, int GATHER>
void launch_wide_gather(const ConvArgs &a, const ResidentGeom &g, const dim3 grid, const dim3 block, int lds, hipStream_t st)
{
    if (a.qmult != nullptr || a.lo < 0)
        hipLaunchKernelGGL((conv_resident_wide_kernel<MT, NT, GATHER, kChannels>), grid, block, lds, st, g, a);
    else
        hipLaunchKernelGGL((conv_resident_wide_kernel<MT, NT, GATHER, kTensor>), grid, block, lds, st, g, a);
}

template <int MT, int NT>
void launch_wide(const ConvArgs &a, const ResidentShape &s, hipStream_t st)
{
    const ResidentGeom g = geometry(a, s);
    const dim3 grid((unsigned)(g.per_xcd * 8)), block(64 * s.nwc);
    if (a.in_cs % 32 == 0)
        launch_wide_gather<MT, NT, kWhole>(a, g, grid, block, lds_bytes(a, s), st);
    else
        launch_wide_gather<MT, NT, kPieces>(a, g, grid, block, lds_bytes(a, s), st);
}

template <int MB, int NB>
void launch_tile(const ConvArgs &a, const ResidentShape &s, hipStream_t st)
{
    if (s.ks > 1)
        launch_shape<MB, NB, true>(a, s, st);
    else
        launch_shape<MB, NB, false>(a, s, st);
}

} // namespace

namespace {

// the shapes that are built (tiles of a wave: pixels by channels; waves: channel groups by shares of the reduction)
constexpr ResidentShape kShapes[kResidentShapes] = {{1, 1, 1, 8}, {1, 1, 1, 4}, {2, 1, 1, 8}, {2, 1, 1, 4}, {2, 2, 1, 8}, {2, 2, 1, 4}, {2, 2, 2, 4}, {2, 2, 2, 2}, {4, 1, 1, 8},
                                     {4, 2, 1, 8}, {4, 2, 1, 4}, {4, 4, 1, 4}, {4, 4, 2, 4}, {4, 4, 2, 2}, {8, 2, 1, 2}, {1, 1, 2, 1}, {1, 1, 4, 1}, {2, 1, 4, 1},
                                     {2, 2, 2, 1}, {2, 2, 4, 1}, {4, 1, 4, 1}, {4, 2, 4, 1}, {4, 4, 2, 1}, {4, 4, 4, 1}, {8, 2, 2, 1}, {8, 2, 4, 1}};

bool point(const ConvArgs &a) { return a.R == 1 && a.S == 1 && a.stride_h == 1 && a.stride_w == 1 && a.in_cs % 64 == 0; }

// the 32 x 32 form: no sums to share, weight zero point 128, one-multiply requantisation, whole 16-byte runs of channels to store
bool wide_applies(const ConvArgs &a)
{
    const bool channels = a.qmult != nullptr || a.lo < 0; // the saturating pack is their upper clamp
    return a.bwz == 0 && a.acc_out == nullptr && a.deq_out == nullptr && (a.qmult != nullptr ? a.fastch : a.fastq) && a.out_cs % 16 == 0
        && (!channels || (a.lo < 0 ? a.lo >= -128 && a.q.hi == 127 : a.q.hi == 255))
        && (a.res == nullptr || (!channels && a.addq.fast && a.addq.hi == 255));
}

// Microseconds of a launch.  Layers with one scale and no sign, and those that go through the general requantisation (kAny), in the 16 x 16
// form: fitted to 12 000 launches, 490 layers of 1 to 200 000 pixels and 16 to 8192 channels in every shape that fits LDS (half of them
// within 8 % of the fit, nine in ten within 18); in the 32 x 32 form to 4900, 400 layers of 300 000 to 24 million outputs (nine in ten within
// 20 %).  Layers with a scale per channel or a signed range, whose requantisation takes twice the instructions, in both forms: fitted to
// 2200 layers of 10 outputs to 25 million in every shape that takes less than twice the best one's time (nine in ten within 17 %); of the
// shapes that fit LDS, the one that this picks for them takes 2 % more than the best on average (8 % by the other layers' terms, which spread 300
// work-groups evenly over 256 CUs).

// the 32 x 32 form.  A launch; for every generation of resident work-groups its start and end, and per step and per tile of a wave its
// chain; per CU the multiplies, those of them that are of channels the layer has, the pixels' KB, the weights' KB and the tiles; the
// tensors' MB
double wide_cost(const ConvArgs &a, const ResidentShape &s)
{
    static const double kCost[2][11] = {{2.684, 1.019, 0.0112, 0.0036, 0.0133, 0.0203, 0.0325, 0.0271, 0.0332, 0.1241, 0.0001},  // a step lies in one tap,
                                        {2.888, 0.662, 0.0096, 0.0086, 0.0053, 0.0244, 0.0675, 0.0426, 0.0265, 0.1094, 0.0000}}; // it does not
    // channels' scales or a signed range: a launch; generation, tile x step, step, tile, KB of pixels / wave; CU's multiplies, tiles, those with a
    // scale per channel, KB of pixels, weights; MB
    static const double kChannelCost[2][12] = {{2.07, 1.24, 0.0123, 0.0172, 0.167, 0.0383, 0.0111, 0.0245, 0.0319, 0.00110, 0.00485, 0.129},
                                               {2.68, 0.248, 0.00765, 0.0490, 0.175, 0.0341, 0.00956, 0.0295, 0.0310, 0.00769, 0.00628, 0.106}};
    const bool channels = conv_resident_channels(a), pieces = a.in_cs % 32 != 0;
    const int mt = s.mb / 2, nt = s.nb / 2, nw = s.nwc, steps = (a.Ktot + 31) / 32, ct = (a.out_cs + 31) / 32;
    const int groups = (a.out_cs + 16 * s.nb * nw - 1) / (16 * s.nb * nw);
    const double wgs = (double)((a.P + 16 * s.mb - 1) / (16 * s.mb)) * groups;
    const int waves = mt * nt == 8 || (mt * nt == 4 && (nt == 2 || channels)) ? 2 : mt * nt == 4 || channels ? 3 : 4; // of a SIMD, by their registers
    // five and six waves: two of a work-group on one SIMD, none left for two of the next (the fit was a quarter low with two work-groups)
    const int held = std::max(1, std::min(160 * 1024 / lds_bytes(a, s), channels && nw > 4 ? waves / 2 : 4 * waves / nw));
    const double gens = std::ceil(wgs / (256.0 * held)), cu = std::max(1.0, wgs / 256), most = std::ceil(wgs / 256), used = (double)std::min(nw * nt * groups, ct) / groups;
    const double region = 1e-3 * region_rows(a, s.mb) * lds_row(a), mb = 1e-6 * ((double)a.P * a.out_cs + (double)a.N * a.H * a.W * a.in_cs);
    const double tiles = most * nw * mt * nt;
    if (channels) {
        const double *const k = kChannelCost[pieces];
        return k[0] + gens * (k[1] + steps * (k[2] * mt * nt + k[3]) + k[4] * mt * nt + k[5] * region / nw)
               + most * (0.25 * k[6] * steps * mt * nt * nw + k[9] * region) + tiles * (k[7] + (a.qmult != nullptr ? k[8] : 0)) + cu * k[10] * steps * nt * nw + k[11] * mb;
    }
    const double *const k = kCost[pieces];
    return k[0] + gens * (k[1] + steps * (k[2] * mt * nt + k[6]) + k[9] * mt * nt) + most * 0.25 * steps * mt * (k[3] * nt * nw + k[4] * used) + tiles * k[8]
           + cu * (k[5] * region + k[10] * steps * nt * nw) + k[7] * mb;
}

// The 16 x 16 form.  A launch; for every generation of resident work-groups its start and end; for every slab that a wave takes its chain,
// alone and per pixel tile; per CU the weight and the pixel bytes that it pulls, the output tiles, the partial sums, the pixels that its
// waves locate.
double shape_cost(const ConvArgs &a, const ResidentShape &s)
{
    if (s.ks == 0)
        return wide_cost(a, s);
    // launch, generation, slab, slab x pixel tile, KB of weights, KB of pixels, output tile, partial tile, pixel tile of a SIMD
    static const double kCost[2][4][9] = {
        {{2.505, 0.101, 0.0027, 0.0142, 0.0086, 0.0295, 0.0156, 0, 0},        // whole reductions: 1x1,
         {2.160, 1.013, 0.0079, 0.0177, 0.0083, 0.0270, 0.0302, 0, 0},        // a slab lies in one tap,
         {2.391, 0.560, 0.0304, 0.0198, 0.0065, 0.0286, 0.0260, 0, 0},        // it does not,
         {3.521, 0, 0.0101, 0.0550, 0.0058, 0.0237, 0.0668, 0, 0}},           // weight zero points and the rest
        {{2.279, 0.502, 0, 0.0220, 0.0095, 0.0147, 0.0306, 0.0085, 0},        // shared ones
         {2.225, 0.842, 0, 0.0263, 0.0105, 0.0103, 0.0355, 0.0063, 0.0607},
         {2.243, 0.689, 0.0235, 0.0264, 0.0095, 0.0115, 0.0211, 0.0096, 0.0663},
         {2.438, 0.885, 0.0024, 0.0643, 0.0097, 0.0067, 0.0459, 0.0143, 0.0591}}};
    // channels' scales or a signed range, whole and shared reductions: a launch; generation, slab, slab of 128 pixels (two slabs of weights ahead
    // instead of four), slab x pixel tile, tile, the same with a scale per channel; of the CU with the most work-groups KB of pixels,
    // multiplies of a SIMD, pixel tiles of a SIMD, output tiles; KB of weights; MB
    static const double kChannelCost[2][13] = {{2.64, 0.425, 0.0384, 0.0206, 0.00621, 0.0731, 0.0420, 0.0134, 0.00404, 0.0731, 0, 0.00751, 0.146},
                                               {2.57, 0.542, 0.0642, 0.173, 0, 0.0331, 0.0164, 0.0104, 0.00666, 0.103, 0.0235, 0.00688, 0.0445}};
    const int nw = s.nwc * s.ks, lds = lds_bytes(a, s);
    const double wgs = (double)((a.P + 16 * s.mb - 1) / (16 * s.mb)) * ((a.out_cs + 16 * s.nb * s.nwc - 1) / (16 * s.nb * s.nwc));
    const int regs = 4 * s.mb * s.nb + 4 * s.nb * (s.nb == 1 ? (s.mb == 1 ? 9 : 8) : s.nb == 2 && s.mb < 8 ? 6 : 4) + 8 * s.mb + 40;
    const int waves = std::max(1, std::min(8, 512 / regs)); // of a SIMD
    const int held = std::max(1, std::min(160 * 1024 / lds, 4 * waves / nw));
    const double gens = std::ceil(wgs / (256.0 * held)), per = (a.nslab + s.ks - 1) / s.ks, cu = std::max(1.0, wgs / 256);
    const double region = 1e-3 * region_rows(a, s.mb) * lds_row(a), weights = 1.024 * a.nslab * s.nb * s.nwc;
    const bool any = a.bwz != 0 || !(a.qmult != nullptr ? a.fastch : a.fastq);
    if (conv_resident_channels(a)) {
        const double *const k = kChannelCost[s.ks > 1];
        const double most = std::ceil(wgs / 256), mb = 1e-6 * ((double)a.P * a.out_cs + (double)a.N * a.H * a.W * a.in_cs);
        return k[0] + gens * (k[1] + per * (k[2] + (s.mb == 8 ? k[3] : 0) + k[4] * s.mb) + s.mb * s.nb * (k[5] + (a.qmult != nullptr ? k[6] : 0)))
               + most * (k[7] * region + 0.25 * nw * s.mb * (k[8] * per * s.nb + k[9]) + k[10] * s.mb * s.nb * s.nwc) + cu * k[11] * weights + k[12] * mb;
    }
    const double *const k = kCost[s.ks > 1][any ? 3 : point(a) ? 0 : a.in_cs % 64 == 0 ? 1 : 2];
    return k[0] + gens * (k[1] + per * (k[2] + k[3] * s.mb)) + cu * (k[4] * weights + k[5] * region + k[6] * s.mb * s.nb * s.nwc
           + (s.ks > 1 ? k[7] * nw * s.mb * s.nb : 0) + k[8] * 0.25 * nw * s.mb);
}

} // namespace

bool conv_resident_applies(const ConvArgs &a)
{
    // the first tap of a pixel is never behind that of the pixel before (pads below half of the window); a tap mask has 32 bits, and the
    // loads behind the last slab may enter two taps more; tap numbers by multiplication (m_cpr) hold for 2048 slabs
    return a.group == 1 && a.in_cs % 16 == 0 && a.rowb == a.in_cs && 2 * a.pad_h < a.R && 2 * a.pad_w < a.S && a.R * a.S <= 29 && a.nslab <= 2048;
}

bool conv_resident_cost(const ConvArgs &a, const ResidentShape &s, double *us)
{
    bool built = s.ks == 0 && wide_applies(a) && s.nwc >= 1 && s.nwc <= 8 && (s.mb == 8 || s.mb == 4) && (s.nb == 4 || s.nb == 2);
    for (const ResidentShape &k : kShapes)
        built = built || (k.mb == s.mb && k.nb == s.nb && k.nwc == s.nwc && k.ks == s.ks);
    // LDS, and the ranges of the quotients by multiplication
    if (!built || lds_bytes(a, s) > 160 * 1024 || (a.in_cs / 16 + 1) * (long long)(region_rows(a, s.mb) + 1) + 64 * waves_of(s) >= 65536 || tiles(a, s) >= (1ll << 30)
        || (long long)(a.OW + 16 * s.mb) * a.OW >= (1ll << 30) || (long long)(a.OH + 16 * s.mb + 1) * a.OH >= (1ll << 30))
        return false;
    *us = shape_cost(a, s);
    return true;
}

bool conv_resident_choose(const ConvArgs &a, ResidentShape *shape, double *us)
{
    double best = 1e30;
    for (const ResidentShape &s : kShapes) {
        if (s.mb > 1 && 8 * s.mb >= (a.P + 15) / 16 * 16)
            continue; // half of the rows would be padding
        double t;
        if (conv_resident_cost(a, s, &t) && t < best)
            best = t, *shape = s;
    }
    *us = best;
    return best < 1e30;
}

bool conv_resident_wide_applies(const ConvArgs &a) { return wide_applies(a); }

bool conv_resident_channels(const ConvArgs &a) { return a.bwz == 0 && (a.qmult != nullptr ? a.fastch : a.lo < 0 && a.fastq); }

bool conv_resident_choose_wide(const ConvArgs &a, ResidentShape *shape, double *us)
{
    double best = 1e30;
    for (int mb : {8, 4})
        for (int nb : {4, 2})
            for (int nw = 1; nw <= 8; nw++) {
                const int tiles = (a.out_cs + 16 * nb - 1) / (16 * nb);
                if (nw > tiles || (nw > 1 && (tiles + nw - 2) / (nw - 1) == (tiles + nw - 1) / nw))
                    continue; // the same groups of channels with fewer waves
                const ResidentShape s = {mb, nb, nw, 0};
                double t;
                if (conv_resident_cost(a, s, &t) && t < best)
                    best = t, *shape = s;
            }
    *us = best;
    return best < 1e30;
}

void launch_conv_resident(const ConvArgs &a, const ResidentShape &s, hipStream_t st)
{
    if (s.ks == 0) {
        switch (s.mb * 10 + s.nb) {
        case 84: return launch_wide<4, 2>(a, s, st);
        case 82: return launch_wide<4, 1>(a, s, st);
        case 44: return launch_wide<2, 2>(a, s, st);
        default: return launch_wide<2, 1>(a, s, st);
        }
    }
    switch (s.mb * 10 + s.nb) {
    case 11: launch_tile<1, 1>(a, s, st); break;
    case 21: launch_tile<2, 1>(a, s, st); break;
    case 22: launch_tile<2, 2>(a, s, st); break;
    case 41: launch_tile<4, 1>(a, s, st); break;
    case 42: launch_tile<4, 2>(a, s, st); break;
    case 44: launch_tile<4, 4>(a, s, st); break;
    default: launch_tile<8, 2>(a, s, st); break;
    }
}

namespace {

// both layers as their tiles of whole 64-byte slabs, requantised with one scale
bool pair_applies(const ConvArgs &a)
{
    return conv_resident_applies(a) && a.in_cs % 64 == 0 && a.bwz == 0 && a.acc_out == nullptr && a.deq_out == nullptr && a.qmult == nullptr && a.fastq && a.lo >= 0;
}

template <int MB, int NB>
void launch_pair(const ConvArgs &a, const ResidentShape &s, const ConvArgs &b, const ResidentShape &t, hipStream_t st)
{
    const PairArgs first = {geometry(a, s), a}, second = {geometry(b, t), b};
    const dim3 grid((unsigned)((first.geo.per_xcd + second.geo.per_xcd) * 8)), block(64 * s.nwc * s.ks);
    const int lds = std::max(lds_bytes(a, s), lds_bytes(b, t));
    if (s.ks > 1 || t.ks > 1)
        hipLaunchKernelGGL((conv_resident_pair_kernel<MB, NB, true>), grid, block, lds, st, first, second);
    else
        hipLaunchKernelGGL((conv_resident_pair_kernel<MB, NB, false>), grid, block, lds, st, first, second);
}

} // namespace

void conv_resident_pair_costs(const ConvArgs &a, ResidentPairCosts *costs)
{
    const bool applies = pair_applies(a);
    for (int i = 0; i < kResidentShapes; i++) {
        const ResidentShape &s = kShapes[i];
        double t;
        const bool padding = s.mb > 1 && 8 * s.mb >= (a.P + 15) / 16 * 16; // half of the rows
        costs->us[i] = applies && s.mb * s.nb <= 8 && !padding && conv_resident_cost(a, s, &t) ? t : 0;
    }
}

bool conv_resident_choose_pair(const ResidentPairCosts &a, const ResidentPairCosts &b, ResidentShape *sa, ResidentShape *sb)
{
    double best = 1e30;
    for (int i = 0; i < kResidentShapes; i++)
        for (int j = 0; a.us[i] > 0 && j < kResidentShapes; j++) {
            const ResidentShape &s = kShapes[i], &t = kShapes[j];
            if (!(b.us[j] > 0) || s.mb != t.mb || s.nb != t.nb || s.nwc * s.ks != t.nwc * t.ks)
                continue;
            // the larger one's time, and half of what the smaller one takes beside its launch: its tiles share CUs
            const double c = std::max(a.us[i], b.us[j]) + 0.5 * (std::min(a.us[i], b.us[j]) - 2.2);
            if (c < best)
                best = c, *sa = s, *sb = t;
        }
    return best < 1e30;
}

void launch_conv_resident_pair(const ConvArgs &a, const ResidentShape &s, const ConvArgs &b, const ResidentShape &t, hipStream_t st)
{
    switch (s.mb * 10 + s.nb) {
    case 11: launch_pair<1, 1>(a, s, b, t, st); break;
    case 21: launch_pair<2, 1>(a, s, b, t, st); break;
    case 22: launch_pair<2, 2>(a, s, b, t, st); break;
    case 41: launch_pair<4, 1>(a, s, b, t, st); break;
    default: launch_pair<4, 2>(a, s, b, t, st); break;
    }
}

} // namespace hipq
