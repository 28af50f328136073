// Convolutions over few pixels as a weight stream (conv_stream.hip).
#pragma once

#include "conv_shared.h"

namespace hipq {

// a work-group's share: 16 * mb pixels by 16 * nb output channels, nw waves
struct StreamShape {
    int mb, nb, nw;
};

void launch_conv_stream(const ConvArgs &a, const StreamShape &s, hipStream_t st);

} // namespace hipq
