// The stage kernels: reconstruction, Riemann fluxes and RK update of a leaf.
#pragma once
#include "device.hpp"

namespace amr {

namespace {

// ------------------------------------------------------------------ stage
// MUSCL2D.cpp:13-121 + the RK update of main.cpp:147-157 / 179-189 for one
// leaf: primitives of the whole tile, edge states, normal-B override from the
// faces, Riemann fluxes on [nxminb,nxmax]^2, then every cell of the tile is
// advanced (the residual is zero outside [nxminb,nxmax]^2).
//
// TPB lanes per leaf; the face fluxes are kept in LDS for the RK update (FLDS)
// or read back from the global ff/gg the block has just written (25.6 KB of
// LDS instead of 64.8, so that three workgroups share a CU).  Which of the
// kernels a launch takes: stage_rule (kernels.hpp).
// A face costs about 1400 issue slots of FP64 work, so a block's ten
// wavefronts of faces take 7.7 us on one CU (three to a SIMD; a wavefront alone
// takes 2.6), the loads and primitives before them 2.0 to 2.4 us, the update
// 1.5 us.  SPEC = kStageHLLDMuscl (kStageHLLCMuscl, kStageHLLDWeno5) fixes the
// solver and the reconstruction's family at compile time, used when every leaf
// of the launch has them.
template <int NT, int NG, bool FLDS>
struct StageLds {
  static constexpr int N2 = NT * NT;
  static constexpr int LO = NG - 1, HI = NT - 1 - NG, NF = HI - LO + 1;
  static constexpr int NFL = FLDS ? 8 * NF * (NF + 1) : 1;
  // doubles: primitive tile, x-face and y-face fluxes
  static constexpr int kDoubles = 8 * N2 + 2 * NFL;
};

// the Riemann solver of a stage specialisation (generic: the instance's)
template <int SPEC>
__device__ inline int spec_solver(int inst_solver) {
  return SPEC == kStageHLLCMuscl ? (int)kFluxHLLC : SPEC != kStageGeneric ? (int)kFluxHLLD : inst_solver;
}

// Primitives of tile cell c into sWc[k * VS] (k = 0..7) with the checks of
// meshblock.cpp:135-142 / 163-176, cell by cell: pressure, then velocity
// NaN.  Bits set in *flags: kTileNan for a NaN primitive where the limiter's
// edge check applies, kTileWide for a primitive outside the exponent range of
// the FAST reconstruction, kTileSpatial for a z velocity or field that is not
// +0.
enum { kTileNan = 1, kTileWide = 2, kTileSpatial = 4 };

// primitives w of the conserved state u; returns the flags it sets
__device__ AMR_INLINE int tile_prim(const double* u, double g, double* w) {
  ExpSpan us, rs, ws;
  rs.add(u[0]);
#pragma unroll
  for (int k = 1; k < 4; k++) us.add(u[k]);
  cons_to_prim<true>(u, g, w);
  if (!(us.within(-860, 400) && rs.within(-100, 100))) cons_to_prim<false>(u, g, w);
#pragma unroll
  for (int k = 0; k < 8; k++) ws.add(w[k]);
  return (ws.within(kPrimLo, kPrimHi) ? 0 : kTileWide) |
         ((__double_as_longlong(w[3]) | __double_as_longlong(w[7])) ? kTileSpatial : 0);
}

template <int NT, int NG>
__device__ AMR_INLINE void stage_prim_cell(const double* __restrict__ Qin, double g, int lim, int step, const LeafItem& L,
                                       DevError* err, int c, double* sWc, int VS, int* flags) {
  constexpr int N2 = NT * NT, LO = NG - 1, HI = NT - 1 - NG;
  double u[8], w[8];
#pragma unroll
  for (int k = 0; k < 8; k++) u[k] = Qin[k * N2 + c];
  const int tile = tile_prim(u, g, w);
#pragma unroll
  for (int k = 0; k < 8; k++) sWc[k * VS] = w[k];
  const int i = c % NT, j = c / NT;
  if (w[4] <= 0 && i > LO && i < HI + 1 && j > LO && j < HI + 1)
    report(err, L.inst, error_key(step, L.nb, 0, i, j, 0, L.nb, kErrPressure));
  if (step == 2 && (isnan(w[1]) || isnan(w[2]) || isnan(w[3])))
    report(err, L.inst, error_key(step, L.nb, 0, i, j, 1, L.nb, kErrNanVel));
  if (tile) atomicOr(flags, tile);
  if (lim < kLimWENO3) {
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 8; k++) bad |= isnan(w[k]);
    if (bad) atomicOr(flags, kTileNan);
  }
}

// Edge states left and right of a face in its own frame (normal velocity and
// field in components 1 and 5; the normal field itself comes from the faces),
// one limiter or WENO order at a time: LIM is a compile-time constant, so the
// 14 limited slopes of a face form one straight run of independent divisions
// (a limiter chosen inside the loop over components put a chain of scalar
// branches between them).  W: the left cell's component 0 in LDS, VS: stride
// of a component, s: of a cell along the normal.  planar: the z components of
// the whole tile are +0, whose edge values are +0 under every limiter and
// WENO order (0 + phi 0): four of the 14 need no quotient.
template <int LIM, bool FAST, bool ZONLY>
__device__ AMR_INLINE void face_edges_some(const double* W, int VS, int s, int ydir, double dxl, double* wl,
                                           double* wr) {
  // tile component of the face frame's component k
  const int comp[8] = {0, 1 + ydir, 2 - ydir, 3, 4, -1, 6 - ydir, 7};
#pragma unroll
  for (int k = 0; k < 8; k++) {
    if (k == 5 || (k == 3 || k == 7) != ZONLY) continue;
    const double* Wk = W + comp[k] * VS;
    if constexpr (LIM == kLimWENO5) {
      wl[k] = weno5_edge<FAST>(Wk[-2 * s], Wk[-s], Wk[0], Wk[s], Wk[2 * s], true);
      wr[k] = weno5_edge<FAST>(Wk[-s], Wk[0], Wk[s], Wk[2 * s], Wk[3 * s], false);
    } else if constexpr (LIM == kLimWENO3) {
      wl[k] = weno3_edge<FAST>(Wk[-s], Wk[0], Wk[s], true);
      wr[k] = weno3_edge<FAST>(Wk[0], Wk[s], Wk[2 * s], false);
    } else {
      const double a = Wk[0] - Wk[-s], b = Wk[s] - Wk[0], d = Wk[2 * s] - Wk[s];
      wl[k] = muscl_plus<FAST>(LIM, Wk[0], a, b, dxl);
      wr[k] = muscl_minus<FAST>(LIM, Wk[s], b, d, dxl);
    }
    // the edges one component after another: hoisting the loads of all of them
    // costs 6 registers and gains nothing (the waves of a SIMD cover for them)
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int LIM, bool FAST>
__device__ AMR_INLINE void face_edges(const double* W, int VS, int s, int ydir, double dxl, bool planar, double* wl,
                                      double* wr) {
  face_edges_some<LIM, FAST, false>(W, VS, s, ydir, dxl, wl, wr);
  wl[3] = wr[3] = wl[7] = wr[7] = 0.;
  if (!planar) face_edges_some<LIM, FAST, true>(W, VS, s, ydir, dxl, wl, wr);
}

template <int SPEC, bool FAST>
__device__ AMR_INLINE void face_edges_of(int lim, const double* W, int VS, int s, int ydir, double dxl, bool planar,
                                         double* wl, double* wr) {
  constexpr bool muscl_only = SPEC == kStageHLLDMuscl || SPEC == kStageHLLCMuscl, weno5_only = SPEC == kStageHLLDWeno5;
  if constexpr (weno5_only) {
    face_edges<kLimWENO5, FAST>(W, VS, s, ydir, dxl, planar, wl, wr);
  } else {
#define AMR_EDGES(LIM) \
  case LIM: face_edges<LIM, FAST>(W, VS, s, ydir, dxl, planar, wl, wr); break
    switch (lim) {
      AMR_EDGES(kLim1st);
      AMR_EDGES(kLimNoSL);
      AMR_EDGES(kLimMinmod);
      AMR_EDGES(kLimVanLeer);
      AMR_EDGES(kLimSuperbee);
      AMR_EDGES(kLimMC);
      AMR_EDGES(kLimKoren);
      AMR_EDGES(kLimCada);
      default:
        if constexpr (!muscl_only) {
          if (lim == kLimWENO3) face_edges<kLimWENO3, FAST>(W, VS, s, ydir, dxl, planar, wl, wr);
          else face_edges<kLimWENO5, FAST>(W, VS, s, ydir, dxl, planar, wl, wr);
        }
    }
#undef AMR_EDGES
  }
}

// Flux fl, in the tile's frame, of the face above the left cell W along x
// (ydir = 0) or y from the tile's primitives (component stride VS, cell stride
// s along the normal) and the face's normal field bn.  tile: the tile's flags.
template <int SPEC>
__device__ AMR_INLINE int tile_face_flux(const double* W, int VS, int s, int lim, int solver, double g, double dxl,
                                         double bn, int tile, int ydir, double* fl) {
  const bool planar = !(tile & kTileSpatial);
  int st = 0;
  bool ok = false;
  if (!(tile & kTileWide)) {
    double wl[8], wr[8];
    wl[5] = wr[5] = bn;
    face_edges_of<SPEC, true>(lim, W, VS, s, ydir, dxl, planar, wl, wr);
    ok = fast_flux(solver, wl, wr, g, fl, &st);
  }
  if (!ok) {
    asm volatile("" ::: "memory");  // the tile is read again, not kept in registers across the fast path
    double wl[8], wr[8];
    wl[5] = wr[5] = bn;
    face_edges_of<SPEC, false>(lim, W, VS, s, ydir, dxl, planar, wl, wr);
    st = normal_flux(solver, wl, wr, g, fl);
  }
  if (ydir) swap_xy(fl);
  return st;
}

// Flux fl of the x face (ydir = 0: between cells (i, j) and (i + 1, j)) or
// y face (between (i, j) and (i, j + 1)) from the primitives in sWb (cell
// (i, j) of variable k at sWb[k * VS + j * NT + i]) and the face B, with the
// solver-failure and NaN-flux checks of MUSCL2D.cpp:62-115.
template <int NT, int SPEC>
__device__ AMR_INLINE void stage_face(const double* sWb, int VS, const double* __restrict__ B, int lim, int solver,
                                      double g, double dxl, int tile, int i, int j, int ydir, int step,
                                      const LeafItem& L, DevError* err, double* fl) {
  constexpr int N2 = NT * NT;
  const int s = ydir ? NT : 1;  // stride along the face normal
  const int c = j * NT + i;     // left cell; right cell is c + s
  const int st = tile_face_flux<SPEC>(sWb + c, VS, s, lim, solver, g, dxl, B[ydir * N2 + c + s], tile, ydir, fl);
  // per (i, j) the x face (solver, NaN), then the y face
  if (st) report(err, L.inst, error_key(step, L.nb, 2, i, j, ydir ? 3 : 0, L.nb, kErrHLLC));
  bool nan = false;
#pragma unroll
  for (int k = 0; k < 8; k++) nan |= isnan(fl[k]);
  if (nan) report(err, L.inst, error_key(step, L.nb, 2, i, j, ydir ? 4 : 1, L.nb, kErrNanFlux));
}

// Residual of the eight components of a cell from its flux differences dF
// (x) and dG (y) over dx: 16 quotients by one denominator.
__device__ AMR_INLINE void stage_residual(const double* dF, const double* dG, double dxl, double* res) {
  ExpSpan n;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    n.add(dF[k]);
    n.add(dG[k]);
  }
  const bool ok = n.within(-860, 480) && dxl >= 0x1p-100 && dxl <= 0x1p100;
  const Den<true> r = den<true>(dxl);
#pragma unroll
  for (int k = 0; k < 8; k++) res[k] = quot(dF[k], r) + quot(dG[k], r);
  if (!ok) {
#pragma unroll
    for (int k = 0; k < 8; k++) res[k] = dF[k] / dxl + dG[k] / dxl;
  }
}

// What the RK update of a cell reads besides its residual, loaded before the
// barrier that ends the face phase so that the loads are in flight while the
// workgroup's last waves finish.
// U, Us and Uw may alias (Uw is U): every input of a cell is loaded before the
// first store to it, and its elements are read and written by one lane only.
struct RkInput {
  double u[8], us[8];
};

__device__ AMR_INLINE void stage_rk_load(int step, const double* U, const double* Us, int c, int N2, RkInput& in) {
#pragma unroll
  for (int k = 0; k < 8; k++) in.u[k] = U[k * N2 + c];
  if (step != 1) {
#pragma unroll
    for (int k = 0; k < 8; k++) in.us[k] = Us[k * N2 + c];
  }
}

// RK update of the eight components of cell c of the tile from their
// residuals (main.cpp:147-157 / 179-189; SSP-RK3 build-defined).
__device__ AMR_INLINE void stage_rk_cell(int step, int rk, double dt, const double* res, const RkInput& in, double* Us,
                                         double* Uw, int c, int N2) {
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int e = k * N2 + c;
    if (step == 1) Us[e] = in.u[k] - dt * res[k];
    else if (rk == 2) Uw[e] = 0.5 * (in.u[k] + in.us[k] - dt * res[k]);
    else if (step == 2) Us[e] = 0.75 * in.u[k] + 0.25 * (in.us[k] - dt * res[k]);
    else Uw[e] = (1. / 3.) * in.u[k] + (2. / 3.) * (in.us[k] - dt * res[k]);
  }
}

// One leaf, all TPB lanes of the workgroup; sW/sF/sG/sFlags: the workgroup's
// LDS (StageLds layout).  The caller separates two calls on the same LDS by a
// workgroup barrier.
template <int NT, int NG, int TPB, bool FLDS, int SPEC>
__device__ AMR_INLINE void stage_block(const FieldPtrs& F, const LeafItem L, const InstParams* __restrict__ ip, int step,
                                   DevError* err, double* sW, double* sF, double* sG, int* sFlags) {
  using S = StageLds<NT, NG, FLDS>;
  constexpr int N2 = S::N2, LO = S::LO, HI = S::HI, NF = S::NF;
  const InstParams& P = ip[L.inst];
  const double g = P.gamma, dxl = P.dx[L.lev], dt = P.dt;
  const int lim = SPEC == kStageHLLDWeno5 ? (int)kLimWENO5 : P.limiter;
  const int solver = spec_solver<SPEC>(P.solver);
  const size_t t8 = (size_t)L.gs * 8 * N2, t2 = (size_t)L.gs * 2 * N2;
  const double* Qin = F.f[step == 1 ? kU : kUs] + t8;
  const double* __restrict__ B = F.f[step == 1 ? kBi : kBis] + t2;
  double* ff = F.f[kFF] + t8;
  double* gg = F.f[kGG] + t8;
  const int tid = threadIdx.x;
  if (tid == 0) *sFlags = 0;
  __syncthreads();

  for (int c = tid; c < N2; c += TPB) stage_prim_cell<NT, NG>(Qin, g, lim, step, L, err, c, sW + c, N2, sFlags);
  if (FLDS) {
    // stale edge fluxes ff[LO][j], gg[i][LO] enter the residual of ghost cells
    for (int q = tid; q < 8 * NF; q += TPB) {
      const int k = q / NF, r = q % NF;
      sF[k * NF * (NF + 1) + r * (NF + 1)] = ff[k * N2 + (LO + r) * NT + LO];
      sG[k * NF * (NF + 1) + 0 * NF + r] = gg[k * N2 + LO * NT + LO + r];
    }
  }
  __syncthreads();
  if (*sFlags & kTileNan) {
    if (tid == 0) report(err, L.inst, error_key(step, L.nb, 1, 0, 0, 0, L.nb, kErrNanEdge));
    return;
  }

  const int tile = *sFlags;
  for (int q = tid; q < 2 * NF * NF; q += TPB) {
    const int ydir = q >= NF * NF;
    const int r = ydir ? q - NF * NF : q;
    const int i = LO + r % NF, j = LO + r / NF;
    const int c = j * NT + i;
    double fl[8];
    stage_face<NT, SPEC>(sW, N2, B, lim, solver, g, dxl, tile, i, j, ydir, step, L, err, fl);
    if (!ydir) {
#pragma unroll
      for (int k = 0; k < 8; k++) {
        ff[k * N2 + c + 1] = fl[k];
        if (FLDS) sF[k * NF * (NF + 1) + (j - LO) * (NF + 1) + (i + 1 - LO)] = fl[k];
      }
    } else {
#pragma unroll
      for (int k = 0; k < 8; k++) {
        gg[k * N2 + c + NT] = fl[k];
        if (FLDS) sG[k * NF * (NF + 1) + (j + 1 - LO) * NF + (i - LO)] = fl[k];
      }
    }
  }
  const double* U = F.f[kU] + t8;
  double* Us = F.f[kUs] + t8;
  double* Uw = F.f[kU] + t8;
  RkInput rk;
  if (tid < N2) stage_rk_load(step, U, Us, tid, N2, rk);
  __syncthreads();  // also orders this workgroup's ff/gg stores before the reads below

  for (int c = tid; c < N2; c += TPB) {
    if (c != tid) stage_rk_load(step, U, Us, c, N2, rk);
    const int i = c % NT, j = c / NT;
    const bool in = i >= LO && i <= HI && j >= LO && j <= HI;
    double res[8];
#pragma unroll
    for (int k = 0; k < 8; k++) res[k] = 0.;
    if (in) {
      double dF[8], dG[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        if (FLDS) {
          const double* Fk = sF + k * NF * (NF + 1);
          const double* Gk = sG + k * NF * (NF + 1);
          const int fi = (j - LO) * (NF + 1) + (i - LO);
          const int gi = (j - LO) * NF + (i - LO);
          dF[k] = Fk[fi + 1] - Fk[fi];
          dG[k] = Gk[gi + NF] - Gk[gi];
        } else {
          const double* Fk = ff + k * N2;
          const double* Gk = gg + k * N2;
          dF[k] = Fk[c + 1] - Fk[c];
          dG[k] = Gk[c + NT] - Gk[c];
        }
      }
      stage_residual(dF, dG, dxl, res);
    }
    stage_rk_cell(step, P.rk, dt, res, rk, Us, Uw, c, N2);
  }
}

template <int NT, int NG, int TPB, bool FLDS, int WPE, int SPEC = kStageGeneric>
__global__ __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(WPE))) void stage_kernel(
    FieldPtrs F, const LeafItem* __restrict__ leaves, const InstParams* __restrict__ ip, int step, DevError* err,
    const int32_t* __restrict__ counts) {
  using S = StageLds<NT, NG, FLDS>;
  __shared__ double lds[S::kDoubles];
  __shared__ int sFlags;
  if (counts && (int)blockIdx.x >= counts[kCountLeaves]) return;
  stage_block<NT, NG, TPB, FLDS, SPEC>(F, leaves[blockIdx.x], ip, step, err, lds, lds + 8 * S::N2,
                                       lds + 8 * S::N2 + S::NFL, &sFlags);
}

// ------------------------------------------------------------ stage strips
// The same stage with each leaf split into K row strips, one workgroup per
// strip, so that small trees still fill the device and a CU holds several
// strips whose load, face and update phases overlap.  The interior rows
// [LO, HI] are divided into K nearly equal parts; the first strip also
// updates the ghost rows below LO, the last those above HI.  A strip forms
// the primitives of its rows and NG rows either side, the x faces of its
// rows and the y faces below and above them -- the y faces on its lower
// edge are also formed by the strip below, with the same operations and so
// the same values, and written to gg by that strip only.  Results equal the
// whole-leaf kernel's bit for bit.  The workgroup of item q = leaf * K +
// strip is launched with id b such that q = (b % 8) * per + b / 8: the
// strips of one leaf run on the same XCD (workgroups are dealt to the 8 XCDs
// round robin) and share the rows they both read in its L2.
template <int NT, int NG, int K>
struct StripGeom {
  static constexpr int LO = NG - 1, HI = NT - 1 - NG, NF = HI - LO + 1;
  static constexpr int kRows = (NF + K - 1) / K;            // interior rows of the largest strip
  static constexpr int kPrimRows = kRows + 2 * NG;           // primitive rows it needs
  // x faces + y faces, at most: the first strip has the most rows, the others
  // the shared y-face row below them too
  static constexpr int kRest = NF - kRows;                   // rows of the other strips
  static constexpr int kRows1 = (kRest + K - 2) / (K - 1);   // of the largest of them
  static constexpr int kFaces = kRows >= kRows1 + 1 ? 2 * kRows * NF : (2 * kRows1 + 1) * NF;
  static constexpr int kLanes = (kFaces + 63) / 64 * 64;
  // doubles: primitives, x fluxes (stale edge face + NF per row), y fluxes
  static constexpr int kDoubles = 8 * kPrimRows * NT + 8 * kRows * (NF + 1) + 8 * (kRows + 1) * NF;
  __device__ static int row0(int s) { return LO + (s * NF + K - 1) / K; }
};

template <int NT, int NG, int K, int SPEC>
__global__ __launch_bounds__((StripGeom<NT, NG, K>::kLanes)) __attribute__((amdgpu_waves_per_eu(3))) void stage_strip_kernel(
    FieldPtrs F, const LeafItem* __restrict__ leaves, int nleaf, const InstParams* __restrict__ ip, int step,
    DevError* err, const int32_t* __restrict__ counts) {
  using Gm = StripGeom<NT, NG, K>;
  constexpr int N2 = NT * NT, LO = Gm::LO, HI = Gm::HI, NF = Gm::NF, TPB = Gm::kLanes;
  constexpr int PR = Gm::kPrimRows, XR = Gm::kRows;
  __shared__ double lds[Gm::kDoubles];
  __shared__ int sFlags;
  if (counts) nleaf = counts[kCountLeaves];
  const int per = (nleaf * K + 7) / 8;
  const int item = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if ((int)(blockIdx.x / 8) >= per || item >= nleaf * K) return;
  const LeafItem L = leaves[item / K];
  const int strip = item % K;
  const int jr0 = Gm::row0(strip), jr1 = Gm::row0(strip + 1) - 1;  // interior rows
  const int r0 = strip == 0 ? 0 : jr0, r1 = strip == K - 1 ? NT - 1 : jr1;  // updated rows
  const int pr0 = jr0 - NG > 0 ? jr0 - NG : 0, pr1 = jr1 + NG < NT - 1 ? jr1 + NG : NT - 1;
  const int ya = jr0 > LO + 1 ? jr0 : LO + 1;  // first computed y-face row (face jj: cells jj - 1, jj)
  const int nx = (jr1 - jr0 + 1) * NF, ny = (jr1 + 1 - ya + 1) * NF;
  double* sW = lds;                     // [k][PR][NT], row pr0 first
  double* sF = lds + 8 * PR * NT;       // [k][XR][NF + 1]: x faces LO .. HI + 1 of rows jr0 ..
  double* sG = sF + 8 * XR * (NF + 1);  // [k][XR + 1][NF]: y faces of rows jr0 .. jr1 + 1
  const double* sWb = sW - pr0 * NT;    // cell (i, j), variable k at sWb[k * PR * NT + j * NT + i]

  const InstParams& P = ip[L.inst];
  const double g = P.gamma, dxl = P.dx[L.lev], dt = P.dt;
  const int lim = SPEC == kStageHLLDWeno5 ? (int)kLimWENO5 : P.limiter;
  const int solver = spec_solver<SPEC>(P.solver);
  const size_t t8 = (size_t)L.gs * 8 * N2, t2 = (size_t)L.gs * 2 * N2;
  const double* Qin = F.f[step == 1 ? kU : kUs] + t8;
  const double* __restrict__ B = F.f[step == 1 ? kBi : kBis] + t2;
  double* ff = F.f[kFF] + t8;
  double* gg = F.f[kGG] + t8;
  const int tid = threadIdx.x;
  if (tid == 0) sFlags = 0;
  __syncthreads();

  for (int c = pr0 * NT + tid; c <= pr1 * NT + NT - 1; c += TPB)
    stage_prim_cell<NT, NG>(Qin, g, lim, step, L, err, c, sW + (c - pr0 * NT), PR * NT, &sFlags);
  // stale edge fluxes ff[LO][j] of the strip's rows and, in the first strip, gg[i][LO]
  for (int q = tid; q < 8 * (jr1 - jr0 + 1); q += TPB) {
    const int k = q / (jr1 - jr0 + 1), r = q % (jr1 - jr0 + 1);
    sF[k * XR * (NF + 1) + r * (NF + 1)] = ff[k * N2 + (jr0 + r) * NT + LO];
  }
  if (jr0 == LO)
    for (int q = tid; q < 8 * NF; q += TPB) {
      const int k = q / NF, r = q % NF;
      sG[k * (XR + 1) * NF + r] = gg[k * N2 + LO * NT + LO + r];
    }
  __syncthreads();
  if (sFlags & kTileNan) {
    // the whole-leaf kernel reports this (and writes nothing) when any
    // primitive of the tile is NaN; the strip holding it reports the same key
    if (tid == 0) report(err, L.inst, error_key(step, L.nb, 1, 0, 0, 0, L.nb, kErrNanEdge));
    return;
  }

  const int tile = sFlags;
  for (int q = tid; q < nx + ny; q += TPB) {
    const int ydir = q >= nx;
    const int r = ydir ? q - nx : q;
    const int i = LO + r % NF;
    // x face (i, i + 1) of row j, or y face jj = ya + r / NF between rows j = jj - 1 and jj
    const int j = ydir ? ya + r / NF - 1 : jr0 + r / NF;
    const int c = j * NT + i;
    double fl[8];
    stage_face<NT, SPEC>(sWb, PR * NT, B, lim, solver, g, dxl, tile, i, j, ydir, step, L, err, fl);
    if (!ydir) {
#pragma unroll
      for (int k = 0; k < 8; k++) {
        ff[k * N2 + c + 1] = fl[k];
        sF[k * XR * (NF + 1) + (j - jr0) * (NF + 1) + (i + 1 - LO)] = fl[k];
      }
    } else {
      const bool own = j >= jr0;  // the face below the strip belongs to the strip below
#pragma unroll
      for (int k = 0; k < 8; k++) {
        if (own) gg[k * N2 + c + NT] = fl[k];
        sG[k * (XR + 1) * NF + (j + 1 - jr0) * NF + (i - LO)] = fl[k];
      }
    }
  }
  const double* U = F.f[kU] + t8;
  double* Us = F.f[kUs] + t8;
  double* Uw = F.f[kU] + t8;
  const int c0 = r0 * NT + tid, c1 = r1 * NT + NT - 1;
  RkInput rk;
  if (c0 <= c1) stage_rk_load(step, U, Us, c0, N2, rk);
  __syncthreads();

  for (int c = c0; c <= c1; c += TPB) {
    if (c != c0) stage_rk_load(step, U, Us, c, N2, rk);
    const int i = c % NT, j = c / NT;
    const bool in = i >= LO && i <= HI && j >= LO && j <= HI;
    double res[8];
#pragma unroll
    for (int k = 0; k < 8; k++) res[k] = 0.;
    if (in) {
      double dF[8], dG[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const double* Fk = sF + k * XR * (NF + 1);
        const double* Gk = sG + k * (XR + 1) * NF;
        const int fi = (j - jr0) * (NF + 1) + (i - LO);
        const int gi = (j - jr0) * NF + (i - LO);
        dF[k] = Fk[fi + 1] - Fk[fi];
        dG[k] = Gk[gi + NF] - Gk[gi];
      }
      stage_residual(dF, dG, dxl, res);
    }
    stage_rk_cell(step, P.rk, dt, res, rk, Us, Uw, c, N2);
  }
}

template <int T, int G, int TPB, bool FLDS, int WPE, int SPEC>
void launch_stage_variant(const FieldPtrs& F, const LeafItem* leaves, int nleaf, const InstParams* ip, int step,
                          DevError* err, hipStream_t s, hipEvent_t ev_start, hipEvent_t ev_stop,
                          const int32_t* counts) {
  if (ev_start && ev_stop) {
    // events attached to the dispatch itself: they time the kernel, not the launch
    hipExtLaunchKernelGGL((stage_kernel<T, G, TPB, FLDS, WPE, SPEC>), dim3(nleaf), dim3(TPB), 0, s, ev_start,
                          ev_stop, 0, F, leaves, ip, step, err, counts);
    return;
  }
  stage_kernel<T, G, TPB, FLDS, WPE, SPEC><<<nleaf, TPB, 0, s>>>(F, leaves, ip, step, err, counts);
}

template <int T, int G, int K, int SPEC>
void launch_stage_strips(const FieldPtrs& F, const LeafItem* leaves, int nleaf, const InstParams* ip, int step,
                         DevError* err, hipStream_t s, hipEvent_t ev_start, hipEvent_t ev_stop,
                         const int32_t* counts) {
  constexpr int TPB = StripGeom<T, G, K>::kLanes;
  const unsigned grid = 8u * (unsigned)((nleaf * K + 7) / 8);
  if (ev_start && ev_stop) {
    hipExtLaunchKernelGGL((stage_strip_kernel<T, G, K, SPEC>), dim3(grid), dim3(TPB), 0, s, ev_start, ev_stop, 0, F,
                          leaves, nleaf, ip, step, err, counts);
    return;
  }
  stage_strip_kernel<T, G, K, SPEC><<<grid, TPB, 0, s>>>(F, leaves, nleaf, ip, step, err, counts);
}

}  // namespace

}  // namespace amr
