// Convolutions over few pixels - fully-connected layers, the last stages of a network at a small batch - as a weight stream over
// every CU.  gfx950 only.
//
// Reproduces op_quant_ip_u8xu8_run (art/modules/quant/src/op/ip.cpp:133-209) and op_conv_2d_u8xu8_run
// (art/modules/quant/src/op/conv_2d_uint8_impl.c:39-165) and their int8 variants bit for bit.
#include "conv_stream.h"

namespace hipq {

// ------------------------------------------------------------------------------------------------
// Fully-connected layers and other 1x1 / stride 1 layers over a few hundred pixels at most (op_quant_ip_u8xu8_run,
// art/modules/quant/src/op/ip.cpp:133-209, with the batch as the pixels).  Such a layer is a weight stream: every weight
// byte is used once per pixel row and the weights are many times larger than the activations, so the time is the time
// it takes to pull the weights out of HBM, and that takes every CU.  The tile kernels cannot give every CU a share (a
// 128-row by 4096-column problem has 32 of their tiles); this kernel cuts the output into narrow column strips instead:
//   * a work-group owns 16*NB output channels of 16*MB pixel rows and the whole reduction, on v_mfma_i32_16x16x64_i8:
//     a weight fragment (16 rows of a 64-byte slab, 1 KB of the packed weights) is used by MB multiplies, a pixel
//     fragment by NB, all of one wave;
//   * the NW waves split the reduction in chunks of 128 bytes of k (two slabs: whole cache lines of the pixel rows), and
//     each wave streams ITS chunks through LDS stages of its own, R deep, with the load unit (global_load_lds_dwordx4,
//     eight lanes per 128-byte line: loading the MFMA operand straight into registers would make neighbouring lanes ask
//     for 16 bytes of sixteen different rows, a quarter of the L1 rate).  No barrier in the loop: a wave waits for its
//     own loads (vmcnt) and refills a stage once its own reads of it have returned (lgkmcnt);
//   * 16-byte piece c of pixel row r sits at piece c ^ (r & 7) of its 128-byte LDS row, the blocks of eight rows are
//     spaced so that rows r and r + 8 start in different halves of the banks, the weights keep their packed order: the
//     fragment reads are free of bank conflicts;
//   * the waves' partial sums meet once, in LDS, and the waves share the epilogue.
//   * k runs over the taps and their channels in 16-byte pieces (a channel stride is a multiple of 16, so no piece straddles two
//     taps): chunk c of a pixel's reduction is its pieces 8 c .. 8 c + 7, each read from the neighbouring pixel its tap points at
//     or, outside the image and beyond the last tap, from the pad source.  Channel strides that are no multiple of 128 went
//     to the tile kernels before, which walk such a reduction in one or two work-groups' 64-byte steps: a 7307 -> 11 layer on
//     6 pixels took 26.6 us;
//   * HAS_WZP (weight zero point other than 128): the sum of a pixel's re-centred bytes, which the zero point multiplies, is
//     the product with a weight operand of ones - every accumulator row holds it - and joins each wave's partial sums.
template <int MB, int NB>
struct StreamCfg {
    static constexpr int ROWS = 16 * MB;
    static constexpr int XI = ROWS / 8;            // pixel loads per chunk: 8 rows of 128 bytes each
    static constexpr int PER = XI + 2 * NB;        // loads per chunk
    // block j of 8 pixel rows sits at j * 1024 + ((j + 1) >> 1) * 128: the two blocks of a 16-row fragment start in
    // different halves of the banks
    static constexpr int XBYTES = XI * 1024 + (XI / 2 + 1) * 128;
    static constexpr int STAGE = XBYTES + 2 * NB * 1024;
    static constexpr int R0 = (160 * 1024) / (4 * STAGE);
    static constexpr int R = R0 > 4 ? 4 : R0;      // stages per wave (four waves)
    static_assert(R >= 2 && (R - 1) * PER <= 63, "stage count / vmcnt range");
};

struct StreamGeom {
    int mtiles, ntiles; // pixel tiles and column strips
    float inv_cs;       // 1 / in_cs: a quotient of it is off by one at most (k < 2^22, the host checks) and then corrected
    int magic_s;        // tap / S == (tap * magic_s) >> 16 for tap <= 256 (R * S at most that, the host checks)
};

// CONVX: any kernel size, stride and padding (a convolution over few pixels - the last stages of a network at batch 1 -
// is the same weight stream); otherwise 1x1 / stride 1 without padding.  WHOLE: channel strides that are multiples of 128, where a
// chunk lies in one tap and its position is wave-uniform (1 % of ResNet-18 at batch 1).
template <int MB, int NB, bool CONVX, bool WHOLE, bool HAS_WZP>
__global__ __launch_bounds__(256) void conv_mfma_stream_kernel(const ConvArgs a, const StreamGeom geo)
{
    using Cfg = StreamCfg<MB, NB>;
    constexpr int NW = 4, NT = MB * NB, R = Cfg::R, STAGE = Cfg::STAGE, PER = Cfg::PER, XI = Cfg::XI;
    constexpr int WOFF = Cfg::XBYTES; // the weight slabs follow the pixel rows in a stage
    static_assert(NW * R * STAGE >= NW * NT * 1024, "the stages double as the reduction buffer");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NW * R * STAGE];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    // Work-groups go to the 8 XCDs in turn: XCD x takes the x-th contiguous eighth of the list in which the m-tiles of a column
    // strip are neighbours, so that the second reader of a strip's weights finds them in that XCD's L2.  (Strips dealt to
    // the XCDs whole left six of them idle on a layer with two: 48 -> 64 channels, 3x3, on 3136 pixels 10.6 us.)
    const int total = geo.mtiles * geo.ntiles, idx = (int)blockIdx.x >> 3, tile = ((int)blockIdx.x & 7) * (int)(gridDim.x >> 3) + idx;
    if (tile >= total)
        return;
    const int nt = tile / geo.mtiles, mt = tile - nt * geo.mtiles;
    const int n0 = nt * (16 * NB), m0 = mt * (16 * MB);

    const int nch = (a.nslab + 1) >> 1;                          // chunks of two slabs
    const int cnt = wave < nch ? (nch - wave + NW - 1) / NW : 0; // chunks of this wave
    // Every work-group reads the same pixel rows: each starts the reduction at a different chunk, so that they do not
    // all ask for the same lines at the same time (the order of an exact integer sum is free).
    const int rot = (nt * 7 + mt * 3) % nch;
    auto chunk_of = [&](int t) {
        int c = wave + NW * t + rot;
        return c >= nch ? c - nch : c;
    };
    uint8_t *const wl = lds + wave * (R * STAGE);
    // load lane l of pixel instruction j: row 8 j + (l >> 3), LDS piece l & 7 = logical piece (l & 7) ^ (row & 7)
    const int xrow = lane >> 3, xoff = ((lane & 7) ^ xrow) << 4;
    const uint8_t *wsrc = a.wpack + (size_t)n0 * 64 + lane * 16;
    const size_t wslab = (size_t)a.kout_pad * 64;
    // CONVX: this lane's pixel of load j - first input row and column of its window, pixel index of its image's origin
    int wih[CONVX ? XI : 1], wiw[CONVX ? XI : 1], wpix[CONVX ? XI : 1];
    if (CONVX) {
        const int ohw = a.OH * a.OW;
#pragma unroll
        for (int j = 0; j < XI; j++) {
            const int m = min(m0 + 8 * j + xrow, a.P - 1);
            const int n = fast_div(m, ohw, a.inv_ohw), rem = m - n * ohw;
            const int oh = fast_div(rem, a.OW, a.inv_ow), ow = rem - oh * a.OW;
            wih[j] = oh * a.stride_h - a.pad_h, wiw[j] = ow * a.stride_w - a.pad_w, wpix[j] = n * a.H * a.W;
        }
    }
    auto issue = [&](int t) {
        const int chunk = chunk_of(t);
        uint8_t *st = wl + (t % R) * STAGE;
        if (CONVX) {
            int tap, coff, kr; // this lane's piece of the reduction: which tap, which of its channels
            if (WHOLE) {
                tap = chunk / (a.in_cs >> 7), coff = (chunk - tap * (a.in_cs >> 7)) * 128 + xoff;
                kr = tap / a.S;
            } else {
                const int k = chunk * 128 + xoff;
                tap = (int)((float)k * geo.inv_cs), coff = k - tap * a.in_cs;
                if (coff < 0)
                    tap--, coff += a.in_cs;
                if (coff >= a.in_cs)
                    tap++, coff -= a.in_cs;
                kr = (tap * geo.magic_s) >> 16;
            }
            const int ks = tap - kr * a.S;
#pragma unroll
            for (int j = 0; j < XI; j++) {
                const int ih = wih[j] + kr, iw = wiw[j] + ks;
                const bool ok = (WHOLE || kr < a.R) && (unsigned)ih < (unsigned)a.H && (unsigned)iw < (unsigned)a.W;
                const uint8_t *src = ok ? a.x + (uint32_t)((wpix[j] + ih * a.W + iw) * a.in_cs + coff) : a.padbuf + (xoff & 48);
                __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(st + j * 1024 + ((j + 1) >> 1) * 128), 16, 0, 0);
            }
        } else {
            // a piece beyond the pixel's channels meets weights that add nothing: any bytes of the tensor will do
            const int k = chunk * 128 + xoff, off = WHOLE || k < a.in_cs ? k : 0;
#pragma unroll
            for (int j = 0; j < XI; j++) {
                // rows beyond the last pixel repeat it, their results are dropped; formed here and not kept over the loop, which
                // took 128 x 4096 x 4096 from 9.05 to 9.31 us
                const int m = min(m0 + 8 * j + xrow, a.P - 1);
                __builtin_amdgcn_global_load_lds((gptr_t)(a.x + (uint32_t)(m * a.in_cs + off)), (lptr_t)(st + j * 1024 + ((j + 1) >> 1) * 128), 16, 0, 0);
            }
        }
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
                __builtin_amdgcn_global_load_lds((gptr_t)(wsrc + (size_t)(2 * chunk + h) * wslab + nb * 1024),
                                                 (lptr_t)(st + WOFF + (h * NB + nb) * 1024), 16, 0, 0);
    };

    v4i acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
            acc[mb][nb] = v4i{0, 0, 0, 0};
    v4i xsum[MB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
        xsum[mb] = v4i{0, 0, 0, 0};

    for (int u = 0; u < R - 1 && u < cnt; u++)
        issue(u);
    // fragment addresses inside a stage: weights in packed order; pixel row 16 mb + r lives in block 2 mb + (r >> 3)
    // (rows r and r + 8 fall into different halves of the banks), piece (4 h + q) of the row at piece ^ (r & 7)
    const int wfo = WOFF + r * 64 + ((q ^ ((r >> 2) & 3)) << 4);
    const int xfo = (r >> 3) * 1152 + (r & 7) * 128; // + 2176 per 16-row fragment
    for (int t = 0; t < cnt; t++) {
        // this wave's fragment reads of chunk t - 1 have returned (the load unit's LDS writes are not ordered against
        // pending reads), then its stage is refilled
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
        if (t + R - 1 < cnt)
            issue(t + R - 1);
        const int ahead = min(R - 1, cnt - 1 - t); // chunks younger than t in flight
        if (ahead >= 3)
            wait_vmcnt<3 * PER>();
        else if (ahead == 2)
            wait_vmcnt<(R > 2 ? 2 : 0) * PER>();
        else if (ahead == 1)
            wait_vmcnt<PER>();
        else
            wait_vmcnt<0>();
        const uint8_t *st = wl + (t % R) * STAGE;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v4i wf[NB];
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
                wf[nb] = *reinterpret_cast<const v4i *>(st + wfo + (h * NB + nb) * 1024);
#pragma unroll
            for (int mb = 0; mb < MB; mb++) {
                const v4i xs = *reinterpret_cast<const v4i *>(st + mb * 2176 + xfo + (((4 * h + q) ^ (r & 7)) << 4)) ^ (int)a.xmask;
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
                    acc[mb][nb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[nb], xs, acc[mb][nb], 0, 0, 0);
                if (HAS_WZP)
                    xsum[mb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{0x01010101, 0x01010101, 0x01010101, 0x01010101}, xs, xsum[mb], 0, 0, 0);
            }
        }
    }

    // ---- the waves' partial sums meet in LDS; wave w finishes the tiles w, w + NW, ...
    __syncthreads(); // every wave is done with its stages; no load is in flight any more
    int32_t *red = reinterpret_cast<int32_t *>(lds); // [wave][tile][register][lane]
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                red[((wave * NT + mb * NB + nb) * 4 + v) * 64 + lane]
                    = HAS_WZP ? (int32_t)((uint32_t)acc[mb][nb][v] + (uint32_t)a.bwz * (uint32_t)xsum[mb][v]) : acc[mb][nb][v];
    __syncthreads();
#pragma unroll
    for (int tl = 0; tl < (NT + NW - 1) / NW; tl++) {
        const int own = wave + tl * NW;
        if (own >= NT)
            break;
        const int mb = own / NB, nb = own % NB;
        const int m = m0 + mb * 16 + r, ko = n0 + nb * 16 + 4 * q; // this lane: 4 consecutive channels of one pixel
        const v4i bias = *reinterpret_cast<const v4i *>(a.bias2 + ko);
        int32_t v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            uint32_t s = (uint32_t)bias[e];
#pragma unroll
            for (int w = 0; w < NW; w++)
                s += (uint32_t)red[((w * NT + own) * 4 + e) * 64 + lane];
            v[e] = (int32_t)s;
        }
        if (m >= a.P || ko >= a.out_cs)
            continue;
        if (a.acc_out != nullptr)
            *reinterpret_cast<v4i *>(a.acc_out + (size_t)m * a.out_cs + ko) = v4i{v[0], v[1], v[2], v[3]};
        int32_t rq[4];
#pragma unroll
        for (int e = 0; e < 4; e++)
            rq[e] = a.qmult ? conv_requant_ch(a, v[e], ko + e) : a.fastq ? conv_requant<true>(a, v[e]) : conv_requant<false>(a, v[e]);
        if (a.deq_out != nullptr) { // fused dequantize (op_dequantize_run_u8, art/modules/quant/src/op/dequantize.c:111-123)
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (ko + e < a.K)
                    a.deq_out[(size_t)m * a.K + ko + e] = __fmul_rn((float)(rq[e] - a.q.zp), a.deq_alpha);
            continue;
        }
        uint32_t packed = pack_low_bytes(rq[0], rq[1], rq[2], rq[3]);
        if (a.res) { // fused residual add: exactly what the add operator computes from the convolution's stored bytes
            const uint32_t rv = *reinterpret_cast<const uint32_t *>(a.res + (size_t)m * a.out_cs + ko);
            packed = a.res_first ? add_dword<false>(rv, packed, a.addq) : add_dword<false>(packed, rv, a.addq);
        }
        *reinterpret_cast<uint32_t *>(a.y + (size_t)m * a.out_cs + ko) = packed;
    }
}

template <int MB, int NB>
static void launch_shape(const ConvArgs &a, hipStream_t st)
{
    const bool fc = a.R == 1 && a.S == 1 && a.stride_h == 1 && a.stride_w == 1 && a.pad_h == 0 && a.pad_w == 0;
    const int mtiles = (a.P + 16 * MB - 1) / (16 * MB), ntiles = (a.out_cs + 16 * NB - 1) / (16 * NB);
    const dim3 grid((mtiles * ntiles + 7) / 8 * 8), block(256);
    const StreamGeom geo = {mtiles, ntiles, 1.f / (float)a.in_cs, 65536 / a.S + 1};
    const int kind = (fc ? 0 : 3) + (a.bwz != 0 ? 2 : a.in_cs % 128 != 0 ? 1 : 0);
    switch (kind) {
    case 0: hipLaunchKernelGGL((conv_mfma_stream_kernel<MB, NB, false, true, false>), grid, block, 0, st, a, geo); break;
    case 1: hipLaunchKernelGGL((conv_mfma_stream_kernel<MB, NB, false, false, false>), grid, block, 0, st, a, geo); break;
    case 2: hipLaunchKernelGGL((conv_mfma_stream_kernel<MB, NB, false, false, true>), grid, block, 0, st, a, geo); break;
    case 3: hipLaunchKernelGGL((conv_mfma_stream_kernel<MB, NB, true, true, false>), grid, block, 0, st, a, geo); break;
    case 4: hipLaunchKernelGGL((conv_mfma_stream_kernel<MB, NB, true, false, false>), grid, block, 0, st, a, geo); break;
    default: hipLaunchKernelGGL((conv_mfma_stream_kernel<MB, NB, true, false, true>), grid, block, 0, st, a, geo); break;
    }
}

void launch_conv_stream(const ConvArgs &a, const StreamShape &s, hipStream_t st)
{
    switch (s.mb * 10 + s.nb) {
    case 81: launch_shape<8, 1>(a, st); break;
    case 42: launch_shape<4, 2>(a, st); break;
    case 41: launch_shape<4, 1>(a, st); break;
    case 22: launch_shape<2, 2>(a, st); break;
    case 21: launch_shape<2, 1>(a, st); break;
    case 12: launch_shape<1, 2>(a, st); break;
    default: launch_shape<1, 1>(a, st); break;
    }
}

} // namespace hipq
