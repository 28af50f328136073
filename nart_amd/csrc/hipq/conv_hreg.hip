// 3x3 / stride 1 / pad 1 convolutions on images of any size, with or without a residual add.  gfx950 only.
//
// Reproduces op_conv_2d_u8xu8_run (art/modules/quant/src/op/conv_2d_uint8_impl.c:39-165) and, with a residual,
// op_quant_add_run (art/modules/quant/src/op/add.c:83-148) bit for bit, like the tile kernels of conv.hip.
//
// The tile kernels stream both operands through LDS in 64-byte steps of the reduction with a barrier each, and a step is a round
// trip of 0.2 - 0.3 us whatever is in it; the register-fed kernel (conv_wreg.hip) has no such steps but cuts images into
// 7 x 7 patches.  Here a work-group owns 32 MT consecutive output pixels of the flattened (image, row, column) index space -
// no size wastes a lane but in the last tile - and the whole reduction:
//   * the pixels that its taps touch, [m0 - W - 1, m0 + 32 MT + W + 1), go to LDS once; tap (r, s) of pixel m is row
//     m - m0 + r W + s.  Taps that leave the image find another row or image there: a 9-bit mask per lane sends them to a row
//     of pad bytes instead;
//   * a wave owns 32 output channels for all of the pixels and loads its weight operands from memory in fragment order
//     (ConvArgs::wfrag), D slabs ahead: no barrier in the loop, no exchange between waves;
//   * what bounds a work-group is the weight bytes it pulls through its CU's L1 (2 KB per wave and slab at some 75 KB/us)
//     beside MT x 2 multiplies of 32 cycles per slab: four pixel tiles balance the two where there are pixels enough, two
//     waves instead of four halve the bytes per CU where there are CUs enough.
// Requirements (checked by the host): uint8 tensors, weight zero point 128, per-tensor scale, one-multiply requantisation,
// dense channel strides, 64, 128, 256 or 512 input channels.
#include "conv_hreg.h"

#include <algorithm>

#include "conv_frag.h"

namespace hipq {

using namespace frag;

namespace {

struct HregGeom {
    int ntile, nnb; // pixel tiles, channel groups
    int rows;       // pixel rows in LDS, without the row of pad bytes behind them
    int nload;      // 1 KB loads per wave that fill LDS
};

} // namespace

template <int CPT, int MT, int NW, bool ADD>
__global__ __launch_bounds__(64 * NW, 2) void conv_hreg_kernel(const ConvArgs a, const HregGeom geo)
{
    constexpr int RB = 64 * CPT, CPR = RB / 16; // bytes and 16-byte pieces of a pixel row
    constexpr int STOT = 9 * CPT, D = MT == 4 ? 6 : 8;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p = lane & 31, h = lane >> 5;
    // work-groups go to the 8 XCDs in turn: XCD x takes the x-th contiguous eighth of the list, in which the channel
    // groups of one pixel tile are neighbours (they read the same pixels)
    const int gid = (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8);
    if (gid >= geo.ntile * geo.nnb)
        return;
    const int tile = gid / geo.nnb, nb = gid - tile * geo.nnb, m0 = tile * (32 * MT);

    // ---- the pixels -> LDS: 16-byte piece c of row r at piece c ^ swz(r); the row behind them and whatever fills up the last
    // loads read the pad source
    for (int k = 0; k < geo.nload; k++) {
        const int id = (k * NW + wave) * 64 + lane, row = id / CPR, c = (id % CPR) ^ swz<RB>(row);
        const int q = m0 - a.W - 1 + row;
        const bool in = row < geo.rows && (unsigned)q < (unsigned)a.P;
        const uint8_t *src = in ? a.x + (uint32_t)(q * RB + c * 16) : a.padbuf + (c & 3) * 16;
        __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(lds + (k * NW + wave) * 1024), 16, 0, 0);
    }

    const int ct0 = (nb * NW + wave) * 32; // the wave's output channels
    const size_t wslab = (size_t)a.kout_pad * 64;
    const uint8_t *w0 = a.wfrag + (size_t)ct0 * 64 + lane * 16;
    auto ldw = [&](int s, int kk) { return ldg128(w0 + (size_t)s * wslab + kk * 1024); };
    WeightRing1<D> ring;
    ring_fill1<STOT, D>(ring, ldw);
    v4i res[MT];
    if (ADD) {
#pragma unroll
        for (int t = 0; t < MT; t++)
            res[t] = ldg128(a.res + (size_t)min(m0 + 32 * t + p, a.P - 1) * a.out_cs + min(ct0 + 16 * h, a.out_cs - 16));
    }

    // the lane's pixels m0 + 32 t + p: which of the nine taps lie inside the image
    int mask[MT];
    const int hw = a.H * a.W;
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int m = min(m0 + 32 * t + p, a.P - 1);
        const int n = fast_div(m, hw, a.inv_ohw), rem = m - n * hw;
        const int y = fast_div(rem, a.W, a.inv_ow), x = rem - y * a.W;
        const int cols = (x > 0 ? 1 : 0) | 2 | (x + 1 < a.W ? 4 : 0);
        mask[t] = (y > 0 ? cols : 0) | cols << 3 | (y + 1 < a.H ? cols << 6 : 0);
    }
    v16i acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++)
        init_acc(acc[t], a.bias2 + ct0 + 16 * h, false);

    auto ldb = [&](int s, int kk, int t) {
        const int tap = s / CPT, cb = s % CPT, r = tap / 3;
        const int row = (mask[t] >> tap) & 1 ? 32 * t + p + r * a.W + (tap - 3 * r) : geo.rows;
        // a row starts at a multiple of its own length (of 256 bytes for longer ones): the swizzled piece is an XOR on the address
        const int base = row * RB + ((h ^ swz<RB>(row)) << 4);
        return *reinterpret_cast<const v4i *>(lds + ((base ^ ((4 * (cb & 3) + 2 * kk) << 4)) + (cb >> 2) * 256));
    };
    // The wave's share of the pixels has landed: re-centre it once, in LDS.  Nine taps of up to four waves would do it 36 times
    // otherwise, four vector instructions for each of the multiplies that they are issued between.
    wait_vmcnt<0>();
    uint8_t *own = lds + wave * 1024 + lane * 16;
#pragma unroll 4
    for (int k = 0; k < geo.nload; k++) {
        v4i *at = reinterpret_cast<v4i *>(own + k * (NW * 1024));
        *at ^= (int)a.xmask;
    }
    __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    reduce_all<STOT, MT, D>(acc, ring, 0, ldw, ldb);
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int m = m0 + 32 * t + p;
        const v4i o = ADD ? requant_add16(a, acc[t], res[t]) : requant16(a, acc[t], 0);
        if (m < a.P && ct0 + 16 * h < a.out_cs)
            *reinterpret_cast<v4i *>(a.y + (size_t)m * a.out_cs + ct0 + 16 * h) = o;
    }
}

namespace {

struct HregShape {
    int mt, nw;
};

int lds_bytes(const ConvArgs &a, const HregShape &s)
{
    const int rows = 32 * s.mt + 2 * a.W + 2, chunk = s.nw * 1024;
    return ((rows + 1) * a.in_cs + chunk - 1) / chunk * chunk;
}

// Microseconds for one shape: 2.6 beside the reduction, a slab as long as the slower of its multiplies and its weight bytes,
// once for every work-group that a CU gets.  (On 26 layers 0.76 to 1.72 of the measured time over all shapes, the middle half 0.90
// to 1.18; the shape it picks is at most 14 % behind the best one, once 28 %.)
double shape_cost(const ConvArgs &a, const HregShape &s)
{
    const double slab = std::max(0.031 * s.mt, 0.029 * s.nw) + 0.004 * s.mt;
    const long long wgs = (long long)((a.P + 32 * s.mt - 1) / (32 * s.mt)) * ((a.out_cs + 32 * s.nw - 1) / (32 * s.nw));
    const double lds_fill = lds_bytes(a, s) / 60e3;
    return 2.6 + (double)((wgs + 255) / 256) * (a.nslab * slab + lds_fill);
}

bool choose_shape(const ConvArgs &a, HregShape *shape, double *us)
{
    static const HregShape cand[] = {{4, 4}, {2, 4}, {1, 4}, {4, 2}, {2, 2}, {1, 2}};
    double best = 1e9;
    for (const HregShape &s : cand) {
        if (lds_bytes(a, s) > 160 * 1024)
            continue;
        const double c = shape_cost(a, s);
        if (c < best)
            best = c, *shape = s;
    }
    *us = best;
    return best < 1e9;
}

template <int CPT, int MT, int NW>
void launch_shape(const ConvArgs &a, hipStream_t st)
{
    HregGeom geo;
    geo.ntile = (a.P + 32 * MT - 1) / (32 * MT), geo.nnb = (a.out_cs + 32 * NW - 1) / (32 * NW);
    geo.rows = 32 * MT + 2 * a.W + 2;
    const unsigned lds = (unsigned)lds_bytes(a, {MT, NW});
    geo.nload = (int)lds / (NW * 1024);
    const dim3 grid((unsigned)((geo.ntile * geo.nnb + 7) / 8 * 8)), block(64 * NW);
    if (a.res != nullptr)
        hipLaunchKernelGGL((conv_hreg_kernel<CPT, MT, NW, true>), grid, block, lds, st, a, geo);
    else
        hipLaunchKernelGGL((conv_hreg_kernel<CPT, MT, NW, false>), grid, block, lds, st, a, geo);
}

template <int CPT>
void launch_cpt(const ConvArgs &a, const HregShape &s, hipStream_t st)
{
    switch (s.mt * 10 + s.nw) {
    case 44: launch_shape<CPT, 4, 4>(a, st); break;
    case 24: launch_shape<CPT, 2, 4>(a, st); break;
    case 14: launch_shape<CPT, 1, 4>(a, st); break;
    case 42: launch_shape<CPT, 4, 2>(a, st); break;
    case 22: launch_shape<CPT, 2, 2>(a, st); break;
    default: launch_shape<CPT, 1, 2>(a, st); break;
    }
}

} // namespace

bool conv_hreg_applies(const ConvArgs &a, double *us)
{
    if (!(a.R == 3 && a.S == 3 && a.pad_h == 1 && a.pad_w == 1 && a.stride_h == 1 && a.stride_w == 1 && a.group == 1 && a.bwz == 0
          && a.xmask != 0 && a.lo >= 0 && a.fastq && a.qmult == nullptr && a.acc_out == nullptr && a.deq_out == nullptr && a.wfrag != nullptr
          && a.C == a.in_cs && (a.in_cs == 64 || a.in_cs == 128 || a.in_cs == 256 || a.in_cs == 512) && a.out_cs % 16 == 0
          && a.nslab == 9 * a.in_cs / 64 && (a.res == nullptr || (a.addq.fast && a.addq.hi == 255))))
        return false;
    HregShape s;
    return choose_shape(a, &s, us);
}

void launch_conv_hreg(const ConvArgs &a, hipStream_t st)
{
    HregShape s = {1, 2};
    double us;
    choose_shape(a, &s, &us);
    switch (a.in_cs) {
    case 64: launch_cpt<1>(a, s, st); break;
    case 128: launch_cpt<2>(a, s, st); break;
    case 256: launch_cpt<4>(a, s, st); break;
    default: launch_cpt<8>(a, s, st); break;
    }
}

} // namespace hipq
