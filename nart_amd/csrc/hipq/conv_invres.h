// Inverted residual blocks - 1x1, depthwise 3x3, 1x1 [, add] - as one kernel (conv_invres.hip).
#pragma once

#include "conv_shared.h"

namespace hipq {

// e: the expanding 1x1 layer; d: the depthwise 3x3 layer; p: the projecting 1x1 layer (p.res and p.addq: with the residual
// add).  Can conv_invres_kernel compute them as one launch?
bool conv_invres_applies(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p);
// Is it faster than the separate launches?
bool conv_invres_preferred(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p);
// The launch and its name, conv_invres_s<stride>_<patch>_k<k-steps>_n<channel tiles>; wanted: 0 patches of 2x4 outputs, 1 4x8,
// 2 8x8, 3 a patch per wave, 4 one of 4x8 at stride 1, -1 (or a shape that is not built for these channels) by cost
void launch_conv_invres(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, int wanted, hipStream_t st);
const char *conv_invres_name(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, int wanted);

} // namespace hipq
