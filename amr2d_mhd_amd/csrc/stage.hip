// One specialisation (AMR_SPEC, kStage*) of the stage kernels for one tile
// (AMR_TILE cells a side): the Makefile builds this file once per pair, so
// that the large straight-line kernels compile in parallel.
#include "stage.hpp"

#ifndef AMR_SPEC
#define AMR_SPEC 0
#define AMR_TILE 20
#endif

namespace amr {

template <>
void launch_stage_tile<AMR_SPEC, AMR_TILE>(int variant, const FieldPtrs& F, const LeafItem* leaves, int nleaf,
                                           const InstParams* ip, int step, DevError* err, hipStream_t s,
                                           hipEvent_t ev_start, hipEvent_t ev_stop, const int32_t* counts) {
  constexpr int T = AMR_TILE, G = T == 24 ? 4 : 2, SPEC = AMR_SPEC;
#define AMR_STAGE_ARGS F, leaves, nleaf, ip, step, err, s, ev_start, ev_stop, counts
  switch (stage_kernel_of(variant)) {
    case kStageNarrow: launch_stage_variant<T, G, 256, false, 3, SPEC>(AMR_STAGE_ARGS); break;
    case kStageStrips: launch_stage_strips<T, G, 4, SPEC>(AMR_STAGE_ARGS); break;
    default: launch_stage_variant<T, G, 768, true, 1, SPEC>(AMR_STAGE_ARGS); break;
  }
}

}  // namespace amr
