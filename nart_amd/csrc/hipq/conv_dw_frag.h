// A depthwise 3x3 layer on the matrix cores, for kernels that keep the tensors around it on the chip (conv_invres.hip,
// conv_dwpoint.hip): 32 pixels x 32 channels of it are nine multiplies, tap by tap a diagonal matrix of the channels' weights times the
// pixels' re-centred rows of 32 bytes at that tap.
#pragma once

#include "conv_frag.h"

namespace hipq {
namespace frag {

__device__ static __forceinline__ void lds_order()
{
    // a wave's LDS instructions execute in the order they are issued; this keeps the compiler to it
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// the channel of a slice of 32 that row p of a multiply stands for: a lane's 16 accumulators are then consecutive channels
__device__ static __forceinline__ int slice_channel(int p)
{
    return 16 * ((p >> 2) & 1) + 4 * (p >> 3) + (p & 3);
}

// The matrix of a tap is diagonal: a lane holds its row's own channel's weight where its half of the columns has that channel, in the
// byte that is the channel's, and zeros.
struct DiagonalTap {
    uint32_t sel[3], dm[4]; // byte s of a dword to the channel's place in its dword; which of the four dwords that is

    __device__ __forceinline__ DiagonalTap(int lane)
    {
        const int ch = slice_channel(lane & 31);
        const bool diagonal = (ch >> 4) == (lane >> 5);
#pragma unroll
        for (int s = 0; s < 3; s++)
            sel[s] = 0x0c0c0c0cu ^ ((0x0cu ^ s) << (8 * (ch & 3)));
#pragma unroll
        for (int j = 0; j < 4; j++) {
            dm[j] = diagonal && ((ch & 15) >> 2) == j ? ~0u : 0u;
            asm("" : "+v"(dm[j])); // masks in registers: an AND each, not a select
        }
    }

    // w: the channel's weights of a kernel row, a byte each
    __device__ __forceinline__ v4i matrix(int w, int s) const
    {
        const uint32_t b = __builtin_amdgcn_perm(0, (uint32_t)w, sel[s]);
        return v4i{(int)(b & dm[0]), (int)(b & dm[1]), (int)(b & dm[2]), (int)(b & dm[3])};
    }
};

// 16 accumulators (16 consecutive channels of a position) -> their bytes, re-centred (XOR 0x80 = 128 less, as signed bytes).  The rounding
// and the zero point ride along in the 64-bit multiply-add, and the last shift saturates to signed bytes, which have the 128 in
// the constants: 5 to 8 % of these kernels' time.
__device__ static __forceinline__ v4i requant_centred(const ConvArgs &a, const v16i &s)
{
    uint64_t add = (uint64_t)(uint32_t)(a.qadd - (128 << a.qt)) << 32;
    uint32_t mult = a.q.mult;
    asm("" : "+s"(add));
    asm("" : "+v"(mult));
    const int32_t plo = (a.lo - 128) * (1 << a.qt), phi = ((a.q.hi - 127) * (1 << a.qt)) - 1;
    v4i o;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        int32_t r[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            r[k] = mulhi_add(s[4 * g + k], mult, add);
            asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r[k]) : "v"(r[k]), "s"(plo), "v"(phi));
        }
        uint32_t b;
        asm("v_ashr_pk_i8_i32 %0, %1, %2, %3" : "=v"(b) : "v"(r[0]), "v"(r[1]), "s"(a.qt));
        asm("v_ashr_pk_i8_i32 %0, %1, %2, %3 op_sel:[0,0,0,1]" : "+v"(b) : "v"(r[2]), "v"(r[3]), "s"(a.qt));
        o[g] = (int)b;
    }
    // a matrix instruction may read these next, two wait states behind the vector instruction that wrote them at the earliest: the
    // compiler, which sees to that, does not see what the assembly above writes
    asm("s_nop 1" : "+v"(o));
    return o;
}

} // namespace frag
} // namespace hipq
