// Convolutions whose input pixels stay in LDS while the weights go straight into registers (conv_resident.hip).
#pragma once

#include "conv_shared.h"

namespace hipq {

// a work-group's share: 16 mb pixels by 16 nb nwc output channels; ks waves share every reduction, so it has nwc ks of them.  ks = 0: the
// form with 32 x 32 tiles (mb and nb even), nwc waves
struct ResidentShape {
    int mb, nb, nwc, ks;
};

// Can conv_resident_kernel compute a plan's launches?
bool conv_resident_applies(const ConvArgs &a);
// Can it in this shape?  *us: what it is expected to take.
bool conv_resident_cost(const ConvArgs &a, const ResidentShape &s, double *us);
// the cheapest shape; false: none
bool conv_resident_choose(const ConvArgs &a, ResidentShape *shape, double *us);
// the same among the shapes with 32 x 32 tiles, which not every launch of a plan can take: conv_resident_wide_applies
bool conv_resident_wide_applies(const ConvArgs &a);
bool conv_resident_choose_wide(const ConvArgs &a, ResidentShape *shape, double *us);
// a scale per channel or a signed range in the one-multiply requantisation: layers that have a fit of their own
bool conv_resident_channels(const ConvArgs &a);
// two layers that do not depend on each other in one launch.  conv_resident_pair_costs: what each shape takes for a layer (a plan keeps
// it: computing it takes longer than the rest of a launch); conv_resident_choose_pair: shapes for both; false: they do not run that way
constexpr int kResidentShapes = 26;
struct ResidentPairCosts {
    double us[kResidentShapes]; // 0: not in this shape
};
void conv_resident_pair_costs(const ConvArgs &a, ResidentPairCosts *costs);
bool conv_resident_choose_pair(const ResidentPairCosts &a, const ResidentPairCosts &b, ResidentShape *sa, ResidentShape *sb);
void launch_conv_resident_pair(const ConvArgs &a, const ResidentShape &s, const ConvArgs &b, const ResidentShape &t, hipStream_t st);
void launch_conv_resident(const ConvArgs &a, const ResidentShape &s, hipStream_t st);

} // namespace hipq
