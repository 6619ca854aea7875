// Table of the precompiled contraction kernel variants (one accessor per line
// of contraction_variants.def, each defined in its own translation unit, then the
// GEMM kernels outside that family).
#include "common.hpp"

namespace tracea_amd {

#define TRACEA_VARIANT(name, bm, bn, bk, wm, wn, stages, direct) \
  const ContractionVariant &contraction_variant_##name();
#include "contraction_variants.def"
#undef TRACEA_VARIANT

namespace {
typedef const ContractionVariant &(*Accessor)();
const Accessor kAccessors[] = {
#define TRACEA_VARIANT(name, bm, bn, bk, wm, wn, stages, direct) &contraction_variant_##name,
#include "contraction_variants.def"
#undef TRACEA_VARIANT
};
constexpr int kFamily = (int)(sizeof(kAccessors) / sizeof(kAccessors[0]));

// Launched by the dispatcher itself (launch_gemm_rows, launch_gemm_ragged): members here so that they can be named,
// forced, timed by the tuner and recorded like the others.
int not_through_the_table(const ContractionArgs &, bool, int, bool, hipStream_t) { return (int)hipErrorInvalidValue; }
const ContractionVariant kOthers[] = {
    {"t48x64x64_w1x4_w16_rows", kGemmRowsMax, 64, 64, 1, 4, 2, kPipelineRows, 0, &not_through_the_table, 16},
    {"t64x64x64_w2x2_w16_any", 64, 64, 64, 2, 2, 2, kPipelineAny, 0, &not_through_the_table, 16},
    {"t128x128x64_w2x4_w16_any", 128, 128, 64, 2, 4, 2, kPipelineAny, 0, &not_through_the_table, 16},
};
}  // namespace

int contraction_variant_count() { return kFamily + (int)(sizeof(kOthers) / sizeof(kOthers[0])); }
const ContractionVariant &contraction_variant(int i) { return i < kFamily ? kAccessors[i]() : kOthers[i - kFamily]; }

}  // namespace tracea_amd
