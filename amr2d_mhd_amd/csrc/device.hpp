// FP64 HIP kernels of the AMR2D-MHD step for gfx950.
//
// Layout: every slot field is [slot][var][j][i] with NT x NT tiles
// (NT = 16 + 2*nghosts), i fastest, so a wavefront reads 64 consecutive
// doubles of one row.  One workgroup handles one leaf block; the block's
// primitive tile and its face fluxes live in LDS for the whole stage.
// No MFMA: nothing on this path is a dense contraction.
#pragma once
#include <hip/hip_ext.h>

#include <algorithm>
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "physics.hpp"

namespace amr {

namespace {

constexpr int kThreads = 256;

// per-instance error records: of the errors an instance's kernels meet, the
// one the reference's sequential execution meets first is kept (see
// DevError), and a failing instance never touches another instance's record
__device__ inline void report(DevError* err, int inst, unsigned long long key) {
  atomicMax(&err[inst].nkey, ~key);
}

#define AMR_DISPATCH_TILE(NT, NG, CALL)                                    \
  do {                                                                     \
    if (NT == 20 && NG == 2) { constexpr int T = 20, G = 2; (void)G; CALL; }        \
    else if (NT == 24 && NG == 4) { constexpr int T = 24, G = 4; (void)G; CALL; }   \
    else if (NT == 12 && NG == 2) { constexpr int T = 12, G = 2; (void)G; CALL; }   \
  } while (0)

}  // namespace

}  // namespace amr
