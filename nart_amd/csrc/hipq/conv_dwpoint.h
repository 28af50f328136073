// A depthwise 3x3 layer and the 1x1 layer behind it [, add] as one kernel (conv_dwpoint.hip).
#pragma once

#include "conv_shared.h"

namespace hipq {

// d: the depthwise 3x3 layer; p: the 1x1 layer that reads it (p.res and p.addq: with the residual add).  Can
// conv_dwpoint_kernel compute them as one launch?
bool conv_dwpoint_applies(const ConvArgs &d, const ConvArgs &p);
// What that launch takes, and what the two launches it replaces do, in us by the fits (see conv_dwpoint.hip)
double conv_dwpoint_us(const ConvArgs &d, const ConvArgs &p);
double conv_dwpoint_apart_us(const ConvArgs &d, const ConvArgs &p);
// The launch and its name, conv_dwpoint_s<stride>_<patch>_n<channel tiles>; wanted: an index of kShapes, -1 (or one that is not built
// for this stride) by cost
void launch_conv_dwpoint(const ConvArgs &d, const ConvArgs &p, int wanted, hipStream_t st);
const char *conv_dwpoint_name(const ConvArgs &d, const ConvArgs &p, int wanted);
int conv_dwpoint_shapes();

} // namespace hipq
