// One specialisation (AMR_SPEC) of the persistent step kernel for one tile
// (AMR_TILE), built like stage.hip.
#include "step.hpp"

#ifndef AMR_SPEC
#define AMR_SPEC 0
#define AMR_TILE 20
#endif

namespace amr {

template <>
const void* step_kernel_tile<AMR_SPEC, AMR_TILE>(int lanes_idx) {
  constexpr int G = AMR_TILE == 24 ? 4 : 2;
  return lanes_idx ? (const void*)step_kernel<AMR_TILE, G, 512, AMR_SPEC>
                   : (const void*)step_kernel<AMR_TILE, G, 256, AMR_SPEC>;
}

}  // namespace amr
