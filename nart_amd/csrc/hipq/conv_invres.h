// Inverted residual blocks - 1x1, depthwise 3x3, 1x1 [, add] - as one kernel (conv_invres.hip).
#pragma once

#include "conv_shared.h"

namespace hipq {

// e: the expanding 1x1 layer; d: the depthwise 3x3 layer; p: the projecting 1x1 layer (p.res and p.addq: with the residual
// add).  Can conv_invres_kernel compute them as one launch?
bool conv_invres_applies(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p);
// Is it faster than the separate launches?
bool conv_invres_preferred(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p);
void launch_conv_invres(const ConvArgs &e, const ConvArgs &d, const ConvArgs &p, hipStream_t st);

} // namespace hipq
