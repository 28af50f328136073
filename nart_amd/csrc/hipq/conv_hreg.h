// 3x3 / stride 1 / pad 1 convolutions with the pixels in LDS and the weights straight in registers (conv_hreg.hip).
#pragma once

#include "conv_shared.h"

namespace hipq {

// Can conv_hreg_kernel compute this launch (a.res: with the residual add)?  *us: what it is expected to take.
bool conv_hreg_applies(const ConvArgs &a, double *us);
void launch_conv_hreg(const ConvArgs &a, hipStream_t st);

} // namespace hipq
