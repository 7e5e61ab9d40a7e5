// Launchers of the step's kernels, and the kernels that are no templates:
// regrid data transfer and the pointwise parity entry points.
#include "phases.hpp"

namespace amr {

namespace {

__global__ __launch_bounds__(kThreads) void fill_kernel(FillProgram P, FillSet set, int NT,
                                                        const int32_t* __restrict__ counts) {
  for (int i = blockIdx.x * kThreads + threadIdx.x; i < set.copy_words; i += gridDim.x * kThreads)
    set.copy_dst[i] = set.copy_src[i];
  if (counts && (int)blockIdx.x >= counts[kCountChunks]) return;
  fill_chunk(P, set, NT, blockIdx.x, threadIdx.x, true);
}

// the program's ops by destination
__global__ __launch_bounds__(kFillChunk) void ring_table_kernel(FillProgram P, int NT, int ng, uint64_t* ring,
                                                                uint32_t version) {
  const int w = blockIdx.x, q = find_segment(P, w);
  const FillOp op = P.ops[q][(w - P.cprefix[q]) * kFillChunk + threadIdx.x];
  if (op.op == kFillNop) return;
  const int r = ring_index(NT, ng, op.dst_cell % NT, op.dst_cell / NT);
  if (r >= 0) ring[(size_t)op.dst_gs * ring_cells(NT, ng) + r] = ring_entry(version, op.op, op.src_cell, op.src);
}

// ------------------------------------------------------------------ regrid
// refine.cpp:17-36: minmod-limited quarter-slope prolongation of one value
__device__ inline double prolong(const double* Q, int NT, int i, int j, int sx, int sy) {
  const int c = j * NT + i;
  double v = Q[c];
  double r = (Q[c] - Q[c - 1]) / (Q[c + 1] - Q[c] + kEps);
  double phi = 0.25 * limiter(kLimMinmod, r, 0) * (Q[c + 1] - Q[c]);
  v = sx == 0 ? v - phi : v + phi;
  r = (Q[c] - Q[c - NT]) / (Q[c + NT] - Q[c] + kEps);
  phi = 0.25 * limiter(kLimMinmod, r, 0) * (Q[c + NT] - Q[c]);
  v = sy == 0 ? v - phi : v + phi;
  return v;
}

// refineBi_CT.cpp:4-50: quadratic face reconstruction sampled at the son face
__device__ inline double prolong_face(const double* B, int NT, int N2, int i, int j, int k, int signx, int signy) {
  const double* Bx = B;
  const double* By = B + N2;
  const int c = j * NT + i;
  const double x_jm = Bx[c - NT], x0 = Bx[c], x_jp = Bx[c + NT];
  const double x_ip = Bx[c + 1], x_ipjm = Bx[c + 1 - NT], x_ipjp = Bx[c + 1 + NT];
  const double y_im = By[c - 1], y0 = By[c], y_ip = By[c + 1];
  const double y_imjp = By[c - 1 + NT], y_jp = By[c + NT], y_ipjp = By[c + 1 + NT];
  const double DyBxm = limiter(kLimMinmod, (x0 - x_jm) / (x_jp - x0 + kEps), 0) * (x_jp - x0);
  const double DyBxp = limiter(kLimMinmod, (x_ip - x_ipjm) / (x_ipjp - x_ip + kEps), 0) * (x_ipjp - x_ip);
  const double DxBym = limiter(kLimMinmod, (y0 - y_im) / (y_ip - y0 + kEps), 0) * (y_ip - y0);
  const double DxByp = limiter(kLimMinmod, (y_jp - y_imjp) / (y_ipjp - y_jp + kEps), 0) * (y_ipjp - y_jp);
  const double ax = (x_ip - x0), by = -1. * ax;
  const double ay = 0.5 * (DyBxp + DyBxm), bx = 0.5 * (DxByp + DxBym);
  const double axy = (DyBxp - DyBxm), byy = axy / (-2.);
  const double bxy = (DxByp - DxBym), axx = bxy / (-2.);
  const double ayy = 0., bxx = 0.;
  if (k == 0) {
    const double a0 = 0.5 * (x_ip + x0) - 0.25 * axx;
    const double sx = signx == 0 ? 0 : 0.5, sy = signy == 0 ? -0.25 : 0.25;
    return a0 + ax * sx + ay * sy + axx * sx * sx + axy * sx * sy + ayy * sy * sy;
  }
  const double b0 = 0.5 * (y_jp + y0) - 0.25 * byy;
  const double sx = signx == 0 ? -0.25 : 0.25, sy = signy == 0 ? 0 : 0.5;
  return b0 + bx * sx + by * sy + bxx * sx * sx + bxy * sx * sy + byy * sy * sy;
}

// refine.cpp:38-59 + refineBi_CT.cpp:52-74 (+ the sons' U2W p<=0 check)
template <int NT, int NG>
__global__ __launch_bounds__(kThreads) void refine_kernel(FieldPtrs F, const RegridOp* __restrict__ ops,
                                                          const InstParams* __restrict__ ip, DevError* err) {
  constexpr int N2 = NT * NT, NX2 = (NT - 1) / 2;
  const RegridOp op = ops[blockIdx.y];
  const int q = blockIdx.z;  // son 0..3
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c >= N2) return;
  const int i = c % NT, j = c / NT;
  const int sx = (i + NG) % 2, sy = (j + NG) % 2;
  const int pi = (q & 1) ? (i - NG + 2) / 2 + NX2 : (i + NG) / 2;
  const int pj = (q & 2) ? (j - NG + 2) / 2 + NX2 : (j + NG) / 2;
  const double* Up = F.f[kU] + (size_t)op.parent_gs * 8 * N2;
  double* Us = F.f[kU] + (size_t)op.son_gs[q] * 8 * N2;
  double u[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    u[k] = prolong(Up + k * N2, NT, pi, pj, sx, sy);
    Us[k * N2 + c] = u[k];
  }
  double w[8];
  cons_to_prim(u, ip[op.inst].gamma, w);
  // refine.cpp:69-83: U2W of son 1..4 in turn; then refineBi_CT.cpp:59-71
  // over (i, j, k) with the four sons innermost
  const int seq = op.seq;
  if (w[4] <= 0 && i > NG - 1 && i < NT - NG && j > NG - 1 && j < NT - NG)
    report(err, op.inst, error_key(kOrdRefine, seq, q, i, j, 0, op.son_nb + q, kErrPressure));
  const double* Bp = F.f[kBi] + (size_t)op.parent_gs * 2 * N2;
  double* Bs = F.f[kBi] + (size_t)op.son_gs[q] * 2 * N2;
  for (int k = 0; k < 2; k++) {
    const double v = prolong_face(Bp, NT, N2, pi, pj, k, sx, sy);
    if (isnan(v)) report(err, op.inst, error_key(kOrdRefine, seq, 4, i, j, 4 * k + q, op.nb, kErrRefineNan));
    Bs[k * N2 + c] = v;
  }
}

// coarsen.cpp:7-157 + coarsenBi_CT.cpp:7-155 through precomputed per-cell
// source maps (last write wins): map = son | i1 << 8 | j1 << 16, -1 = untouched
template <int NT, int NG>
__global__ __launch_bounds__(kThreads) void coarsen_kernel(FieldPtrs F, const RegridOp* __restrict__ ops,
                                                           const int32_t* __restrict__ cmapU,
                                                           const int32_t* __restrict__ cmapB,
                                                           const InstParams* __restrict__ ip, DevError* err) {
  constexpr int N2 = NT * NT;
  const RegridOp op = ops[blockIdx.y];
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c >= N2) return;
  const int i = c % NT, j = c / NT;
  double* Ud = F.f[kU] + (size_t)op.parent_gs * 8 * N2;
  const int m = cmapU[c];
  if (m >= 0) {
    const int s = m & 0xff, i1 = (m >> 8) & 0xff, j1 = (m >> 16) & 0xff;
    const double* Uq = F.f[kU] + (size_t)op.son_gs[s] * 8 * N2;
    const int a = j1 * NT + i1;
    double u[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const double* Q = Uq + k * N2;
      double v = 0.;
      v += Q[a];
      v += Q[a + NT];
      v += Q[a + 1];
      v += Q[a + 1 + NT];
      u[k] = 0.25 * v;
      Ud[k * N2 + c] = u[k];
    }
    double w[8];
    cons_to_prim(u, ip[op.inst].gamma, w);
    if (w[4] <= 0 && i > NG - 1 && i < NT - NG && j > NG - 1 && j < NT - NG)
      report(err, op.inst, error_key(kOrdCoarsen, op.seq, 0, i, j, 0, op.nb, kErrPressure));
  }
  double* Bd = F.f[kBi] + (size_t)op.parent_gs * 2 * N2;
  for (int k = 0; k < 2; k++) {
    const int mb = cmapB[k * N2 + c];
    if (mb < 0) continue;
    const int s = mb & 0xff, i1 = (mb >> 8) & 0xff, j1 = (mb >> 16) & 0xff;
    const double* Q = F.f[kBi] + (size_t)op.son_gs[s] * 2 * N2 + k * N2;
    const int a = j1 * NT + i1;
    double v = 0.;
    v += Q[a];
    v += Q[k == 0 ? a + NT : a + 1];
    Bd[k * N2 + c] = 0.5 * v;
  }
}

// ----------------------------------------------------- parity entry points
// One face pair a lane, one solver a kernel so that only its registers count
// (three waves per SIMD).  Bound by the 196 bytes a face: a million HLLD faces
// took 51.6 us with the compiler's divisions and the six-region solver, 42.6 now,
// a copy of the same bytes 42; moving the eight components through LDS in
// whole lines takes 5% longer (a lane's 64 bytes are one half line).
constexpr int kFaceLanes = 128;

__device__ AMR_INLINE void face_pair(const double* __restrict__ wL, const double* __restrict__ wR, size_t q, int dir,
                                     double* l, double* r) {
#pragma unroll
  for (int k = 0; k < 8; k++) {
    l[k] = wL[8 * q + k];
    r[k] = wR[8 * q + k];
  }
  if (dir == 1) {
    swap_xy(l);
    swap_xy(r);
  }
}

template <int SOLVER>
__global__ __launch_bounds__(kFaceLanes) __attribute__((amdgpu_waves_per_eu(3))) void riemann_batch_kernel(
    int dir, double g, int n, const double* wL, const double* wR, double* flux, int32_t* status) {
  const size_t q = (size_t)blockIdx.x * kFaceLanes + threadIdx.x;
  if (q >= (size_t)n) return;
  double f[8];
  int st = 0;
  bool ok;
  {
    double l[8], r[8];
    face_pair(wL, wR, q, dir, l, r);
    ok = fast_flux(SOLVER, l, r, g, f, &st);
  }
  if (!ok) {
    asm volatile("" ::: "memory");  // the states are read again, not kept in registers
    double l[8], r[8];
    face_pair(wL, wR, q, dir, l, r);
    st = normal_flux(SOLVER, l, r, g, f);
  }
  if (dir == 1) swap_xy(f);
  status[q] = st;
#pragma unroll
  for (int k = 0; k < 8; k++) flux[8 * q + k] = f[k];
}

// edge states of whole tiles, any tile size and ghost depth: out = [tile][4: xL xR yL yR][8][NT][NT]
// (celledges.cpp ranges for MUSCL, WENO2D_primvar.cpp ranges for WENO)
__global__ void recon_batch_kernel(int NT, int ng, int lim, double dxl, const double* W, double* out) {
  const int N2 = NT * NT;
  const int t = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N2) return;
  const int i = c % NT, j = c / NT;
  const double* Wt = W + (size_t)t * 8 * N2;
  double* o = out + (size_t)t * 4 * 8 * N2;
  const bool weno = lim == kLimWENO3 || lim == kLimWENO5;
  const int lo = weno ? ng - 1 : 0, hi = weno ? NT - ng : NT - 2;
  if (i < lo || i > hi || j < lo || j > hi) return;
  for (int k = 0; k < 8; k++) {
    const double* Wk = Wt + k * N2;
    for (int dir = 0; dir < 2; dir++) {
      if ((dir == 0 && k == 5) || (dir == 1 && k == 6)) continue;
      const int s = dir == 0 ? 1 : NT;
      double L, R;
      if (lim == kLimWENO5) {
        L = weno5_edge(Wk[c - 2 * s], Wk[c - s], Wk[c], Wk[c + s], Wk[c + 2 * s], true);
        R = weno5_edge(Wk[c - 2 * s], Wk[c - s], Wk[c], Wk[c + s], Wk[c + 2 * s], false);
      } else if (lim == kLimWENO3) {
        L = weno3_edge(Wk[c - s], Wk[c], Wk[c + s], true);
        R = weno3_edge(Wk[c - s], Wk[c], Wk[c + s], false);
      } else {
        const int idx = dir == 0 ? i : j;
        const int cm = idx > 0 ? c - s : c;  // backward difference, index 0 duplicates 1
        const double d0 = idx > 0 ? Wk[c] - Wk[cm] : Wk[c + s] - Wk[c];
        const double d1 = Wk[c + s] - Wk[c];
        L = muscl_plus(lim, Wk[c], d0, d1, dxl);
        R = muscl_minus(lim, Wk[c], d0, d1, dxl);
      }
      o[((dir * 2 + 0) * 8 + k) * N2 + c] = L;
      o[((dir * 2 + 1) * 8 + k) * N2 + c] = R;
    }
  }
}

__global__ void zero_kernel(double* p, size_t n) {
  for (size_t e = (size_t)blockIdx.x * kThreads + threadIdx.x; e < n; e += (size_t)gridDim.x * kThreads) p[e] = 0.;
}

// The same with the tile in LDS, one workgroup a tile and one limiter a kernel,
// for tiles of up to 28 cells a side (50 KB) with the ghost depth their stencil needs:
// W is read once, the quotients take their FAST forms in tiles within the
// range, and with `fill` the entries outside the computed range are written
// as zeros, so that the caller need not clear `out` first.  Bound by writing
// out: 3000 tiles of 20 x 20, MC, 205 us with the clearing pass and loads of
// every neighbour from global memory, 87 now (384 MB; a copy moves 4.65 TB/s).
constexpr int kReconMaxNT = 28;

template <int LIM, bool FAST>
__device__ AMR_INLINE void recon_edges(const double* Wk, int s, bool first, double dxl, double& L, double& R) {
  if constexpr (LIM == kLimWENO5) {
    L = weno5_edge<FAST>(Wk[-2 * s], Wk[-s], Wk[0], Wk[s], Wk[2 * s], true);
    R = weno5_edge<FAST>(Wk[-2 * s], Wk[-s], Wk[0], Wk[s], Wk[2 * s], false);
  } else if constexpr (LIM == kLimWENO3) {
    L = weno3_edge<FAST>(Wk[-s], Wk[0], Wk[s], true);
    R = weno3_edge<FAST>(Wk[-s], Wk[0], Wk[s], false);
  } else {
    const double d1 = Wk[s] - Wk[0], d0 = first ? d1 : Wk[0] - Wk[-s];  // index 0 duplicates 1
    L = muscl_plus<FAST>(LIM, Wk[0], d0, d1, dxl);
    R = muscl_minus<FAST>(LIM, Wk[0], d0, d1, dxl);
  }
}

template <int LIM>
__global__ __launch_bounds__(kThreads) void recon_tile_kernel(int NT, int ng, double dxl, const double* __restrict__ W,
                                                              double* __restrict__ out, int fill) {
  extern __shared__ double sW[];
  __shared__ int sWide;
  const int N2 = NT * NT, tid = threadIdx.x;
  const double* Wt = W + (size_t)blockIdx.x * 8 * N2;
  double* o = out + (size_t)blockIdx.x * 4 * 8 * N2;
  if (tid == 0) sWide = 0;
  __syncthreads();
  ExpSpan span;
  for (int c = tid; c < 8 * N2; c += kThreads) {
    const double w = Wt[c];
    span.add(w);
    sW[c] = w;
  }
  if (!span.within(kPrimLo, kPrimHi)) sWide = 1;
  __syncthreads();
  const bool wide = sWide;
  constexpr bool weno = LIM == kLimWENO3 || LIM == kLimWENO5;
  const int lo = weno ? ng - 1 : 0, hi = weno ? NT - ng : NT - 2;
  for (int c = tid; c < N2; c += kThreads) {
    const int j = c / NT, i = c - j * NT;
    const bool in = i >= lo && i <= hi && j >= lo && j <= hi;
    if (!in && !fill) continue;
    for (int k = 0; k < 8; k++) {
      const double* Wk = sW + k * N2 + c;
#pragma unroll
      for (int dir = 0; dir < 2; dir++) {
        const bool skip = k == 5 + dir;  // the normal field comes from the faces
        if (skip && !fill) continue;
        double L = 0., R = 0.;
        if (in && !skip) {
          const bool first = (dir ? j : i) == 0;
          if (!wide) recon_edges<LIM, true>(Wk, dir ? NT : 1, first, dxl, L, R);
          else recon_edges<LIM, false>(Wk, dir ? NT : 1, first, dxl, L, R);
        }
        o[((dir * 2 + 0) * 8 + k) * N2 + c] = L;
        o[((dir * 2 + 1) * 8 + k) * N2 + c] = R;
      }
    }
  }
}

}  // namespace

// ---------------------------------------------------------------- launchers
bool tile_supported(int NT, int ng) { return (NT == 20 && ng == 2) || (NT == 24 && ng == 4) || (NT == 12 && ng == 2); }

// the instance of a specialised function for a tile of NT cells a side
#define AMR_SPEC_TILE(SPEC, FN, ...)                     \
  do {                                                   \
    if (NT == 20 && ng == 2) return FN<SPEC, 20>(__VA_ARGS__); \
    if (NT == 24 && ng == 4) return FN<SPEC, 24>(__VA_ARGS__); \
    if (NT == 12 && ng == 2) return FN<SPEC, 12>(__VA_ARGS__); \
  } while (0)

void launch_stage(int NT, int ng, int variant, int spec, const FieldPtrs& F, const LeafItem* leaves, int nleaf,
                  const InstParams* ip, int step, DevError* err, hipStream_t s, hipEvent_t ev_start,
                  hipEvent_t ev_stop, const int32_t* counts) {
  if (nleaf <= 0) return;
#define AMR_STAGE_ARGS variant, F, leaves, nleaf, ip, step, err, s, ev_start, ev_stop, counts
  if (spec == kStageHLLCMuscl)
    AMR_SPEC_TILE(kStageHLLCMuscl, launch_stage_tile, AMR_STAGE_ARGS);
  else if (spec == kStageHLLDMuscl)
    AMR_SPEC_TILE(kStageHLLDMuscl, launch_stage_tile, AMR_STAGE_ARGS);
  else if (spec == kStageHLLDWeno5 && NT == 24 && ng == 4)
    launch_stage_tile<kStageHLLDWeno5, 24>(AMR_STAGE_ARGS);
  else
    AMR_SPEC_TILE(kStageGeneric, launch_stage_tile, AMR_STAGE_ARGS);
#undef AMR_STAGE_ARGS
}

void launch_emf(int NT, const FieldPtrs& F, const LeafItem* leaves, int nleaf, const InstParams* ip, int step,
                int rk, DevError* err, hipStream_t s, const int32_t* counts) {
  if (nleaf <= 0) return;
  dim3 grid((NT * NT + kThreads - 1) / kThreads, nleaf);
  AMR_DISPATCH_TILE(NT, (NT == 24 ? 4 : 2),
                    (emf_kernel<T><<<grid, kThreads, 0, s>>>(F, leaves, ip, step == rk, err, step, counts)));
}

void launch_bupdate(int NT, const FieldPtrs& F, const LeafItem* leaves, int nleaf, const InstParams* ip, int step,
                    int rk, hipStream_t s, const int32_t* counts) {
  if (nleaf <= 0) return;
  dim3 grid((NT * NT + kThreads - 1) / kThreads, nleaf);
  AMR_DISPATCH_TILE(NT, (NT == 24 ? 4 : 2),
                    (bupdate_kernel<T><<<grid, kThreads, 0, s>>>(F, leaves, ip, step, rk, counts)));
}

void launch_bsync(int NT, const FieldPtrs& F, const LeafItem* leaves, int nleaf, int last, hipStream_t s,
                  const int32_t* counts) {
  if (nleaf <= 0) return;
  dim3 grid((NT * NT + kThreads - 1) / kThreads, nleaf);
  AMR_DISPATCH_TILE(NT, (NT == 24 ? 4 : 2), (bsync_kernel<T><<<grid, kThreads, 0, s>>>(F, leaves, last, counts)));
}

void launch_ct(int NT, int ng, const FieldPtrs& F, const LeafItem* leaves, int nleaf, const InstParams* ip, int step,
               int rk, const FillTables& all, const FillTables& tail, const RingTable& ring, DevError* err,
               hipStream_t s) {
  if (nleaf <= 0) return;
  auto program = [](const FillTables& T) { return FillProgram{T.ops, T.gen, T.cprefix, T.ninst}; };
  CtArgs A{F,        leaves,   ip,       all.gen, ring.entries, ring.version,  step,         rk,
           ring.emf, ring.old, ring.rdx, err,     nleaf,        program(tail), program(all), 0, 0};
  A.ntail = step == 1 ? tail.nchunks : 0;  // of Bi
  AMR_DISPATCH_TILE(NT, ng, (ct_emf_kernel<T, G><<<nleaf + ct_tail_wgs<T>(A.ntail), kCtLanes<T>, 0, s>>>(A)));
  A.ntail = tail.nchunks;
  A.nall = all.nchunks;
  AMR_DISPATCH_TILE(NT, ng, (ct_faces_kernel<T, G><<<nleaf + 2 * (ct_tail_wgs<T>(A.ntail) + ct_flux_wgs<T>(A.nall)),
                                                     kCtLanes<T>, 0, s>>>(A)));
}

void launch_ring_table(int NT, int ng, const FillOp* const* inst_ops, const int32_t* cprefix, int ninst, int nchunks,
                       const RingTable& ring, hipStream_t s) {
  if (nchunks <= 0) return;
  const FillProgram P{inst_ops, nullptr, cprefix, ninst};
  ring_table_kernel<<<nchunks, kFillChunk, 0, s>>>(P, NT, ng, ring.entries, ring.version);
}

// Up to this many chunks the fills of U (and Bi) take two components a workgroup
// (fill_parts_kernel): a workgroup a chunk leaves CUs idle and its loads in one
// queue.  Both ways: tails of 9 chunks 5.9 -> 4.0 us, U at 120 chunks 6.0 -> 5.3, at
// 256 to 319 9.9 -> 9.1, at 320 to 399 10.2 and 10.2, at 400 to 511 11.1 and 11.4.
constexpr int kFillPartsChunks = 320;

void launch_fill(int NT, const FillOp* const* inst_ops, const FillGen* const* inst_gen, const int32_t* cprefix,
                 int ninst, int nchunks, const FillSet& set, hipStream_t s, const int32_t* counts) {
  static_assert(kFillChunk == kThreads, "one workgroup per fill chunk");
  if (nchunks <= 0 || set.n <= 0) return;
  FillProgram P{inst_ops, inst_gen, cprefix, ninst};
  const int a = set.nv[0], b = set.n > 1 ? set.nv[1] : 0, c = set.n > 2 ? set.nv[2] : 0;
  const int ka = set.kind[0], kb = set.n > 1 ? set.kind[1] : -1, kc = set.n > 2 ? set.kind[2] : -1;
  constexpr int C = kFillCell, F = kFillFace, E = kFillEdge;
  if (nchunks <= kFillPartsChunks && set.n == 1 && a == 8 && ka == C)
    fill_parts_kernel<0><<<dim3(nchunks, 4), kThreads, 0, s>>>(P, set, NT, counts);
  else if (nchunks <= kFillPartsChunks && set.n == 2 && a == 8 && b == 2 && ka == C && kb == F)
    fill_parts_kernel<2><<<dim3(nchunks, 5), kThreads, 0, s>>>(P, set, NT, counts);
  else if (set.n == 1 && a == 8 && ka == C) fill_kernel_nv<8, 0, 0, C, 0, 0><<<nchunks, kThreads, 0, s>>>(P, set, NT, counts);
  else if (set.n == 1 && a == 2 && ka == F)
    fill_kernel_nv<2, 0, 0, F, 0, 0><<<nchunks, kThreads, 0, s>>>(P, set, NT, counts);
  else if (set.n == 1 && a == 1 && ka == E)
    fill_kernel_nv<1, 0, 0, E, 0, 0><<<nchunks, kThreads, 0, s>>>(P, set, NT, counts);
  else if (set.n == 2 && a == 8 && b == 2 && ka == C && kb == F)
    fill_kernel_nv<8, 2, 0, C, F, 0><<<nchunks, kThreads, 0, s>>>(P, set, NT, counts);
  else if (set.n == 2 && a == 8 && b == 8 && ka == F && kb == F)
    fill_kernel_nv<8, 8, 0, F, F, 0><<<nchunks, kThreads, 0, s>>>(P, set, NT, counts);
  else if (set.n == 3 && a == 2 && b == 8 && c == 8 && ka == F && kb == F && kc == F)
    fill_kernel_nv<2, 8, 8, F, F, F><<<nchunks, kThreads, 0, s>>>(P, set, NT, counts);
  else fill_kernel<<<nchunks, kThreads, 0, s>>>(P, set, NT, counts);
}

void launch_cfl_criteria(int NT, int ng, const FieldPtrs& F, const double* W, const LeafItem* leaves, int nleaf,
                         const InstParams* ip, double* lam_grad, DevError* err, hipStream_t s,
                         const int32_t* counts) {
  if (nleaf <= 0) return;
  AMR_DISPATCH_TILE(NT, ng,
                    (cfl_criteria_kernel<T, G><<<nleaf, kThreads, 0, s>>>(F, W, leaves, ip, lam_grad, err, counts)));
}

void launch_refine(int NT, int ng, const FieldPtrs& F, const RegridOp* ops, int nops, const InstParams* ip,
                   DevError* err, hipStream_t s) {
  if (nops <= 0) return;
  dim3 grid((NT * NT + kThreads - 1) / kThreads, nops, 4);
  AMR_DISPATCH_TILE(NT, ng, (refine_kernel<T, G><<<grid, kThreads, 0, s>>>(F, ops, ip, err)));
}

void launch_coarsen(int NT, int ng, const FieldPtrs& F, const RegridOp* ops, int nops, const int32_t* cmapU,
                    const int32_t* cmapB, const InstParams* ip, DevError* err, hipStream_t s) {
  if (nops <= 0) return;
  dim3 grid((NT * NT + kThreads - 1) / kThreads, nops);
  AMR_DISPATCH_TILE(NT, ng, (coarsen_kernel<T, G><<<grid, kThreads, 0, s>>>(F, ops, cmapU, cmapB, ip, err)));
}

// the step kernel instance for (tile, specialisation, lanes), or null
const void* step_kernel_fn(int NT, int ng, int spec, int lanes_idx) {
  if (spec == kStageHLLDMuscl) AMR_SPEC_TILE(kStageHLLDMuscl, step_kernel_tile, lanes_idx);
  else if (spec == kStageHLLDWeno5 && NT == 24 && ng == 4) return step_kernel_tile<kStageHLLDWeno5, 24>(lanes_idx);
  else AMR_SPEC_TILE(kStageGeneric, step_kernel_tile, lanes_idx);
  return nullptr;
}

int step_kernel_grid(int NT, int ng, int spec, int lanes_idx) {
  const void* fn = step_kernel_fn(NT, ng, spec, lanes_idx);
  if (!fn || lanes_idx < 0 || lanes_idx > 1) return 0;
  int dev = 0, cus = 0, per_cu = 0, coop = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, kStepLanes[lanes_idx], 0) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return coop ? per_cu * cus : 0;
}

int launch_step(int NT, int ng, int spec, int lanes_idx, int grid, const StepArgs& A, hipStream_t s,
                hipEvent_t ev_start, hipEvent_t ev_stop) {
  const void* fn = step_kernel_fn(NT, ng, spec, lanes_idx);
  if (!fn || grid <= 0) return 1;
  StepArgs a = A;
  void* args[] = {&a};
  if (ev_start) hipEventRecord(ev_start, s);
  const hipError_t e = hipLaunchCooperativeKernel(fn, dim3(grid), dim3(kStepLanes[lanes_idx]), args, 0, s);
  if (ev_stop) hipEventRecord(ev_stop, s);
  return e == hipSuccess ? 0 : 1;
}

void launch_riemann_batch(int solver, int dir, double gamma, int n, const double* wL, const double* wR, double* flux,
                          int32_t* status, hipStream_t s) {
  if (n <= 0) return;
  const int blocks = (int)(((int64_t)n + kFaceLanes - 1) / kFaceLanes);
  auto run = [&](auto kernel) { kernel<<<blocks, kFaceLanes, 0, s>>>(dir, gamma, n, wL, wR, flux, status); };
  if (solver == kFluxRusanov) run(riemann_batch_kernel<kFluxRusanov>);
  else if (solver == kFluxHLLE) run(riemann_batch_kernel<kFluxHLLE>);
  else if (solver == kFluxHLLC) run(riemann_batch_kernel<kFluxHLLC>);
  else run(riemann_batch_kernel<kFluxHLLD>);
}

void launch_recon_batch(int NT, int ng, int lim, double dx, int nt, const double* W, double* out, bool fill,
                        hipStream_t s) {
  if (nt <= 0) return;
  const int need = lim == kLimWENO5 ? 3 : lim == kLimWENO3 ? 2 : 0;  // ghost depth of the stencil
  if (NT <= kReconMaxNT && ng >= need) {
    const size_t lds = sizeof(double) * 8 * NT * NT;
    auto run = [&](auto kernel) { kernel<<<nt, kThreads, lds, s>>>(NT, ng, dx, W, out, fill); };
    switch (lim) {
      case kLim1st: return run(recon_tile_kernel<kLim1st>);
      case kLimNoSL: return run(recon_tile_kernel<kLimNoSL>);
      case kLimMinmod: return run(recon_tile_kernel<kLimMinmod>);
      case kLimVanLeer: return run(recon_tile_kernel<kLimVanLeer>);
      case kLimSuperbee: return run(recon_tile_kernel<kLimSuperbee>);
      case kLimMC: return run(recon_tile_kernel<kLimMC>);
      case kLimKoren: return run(recon_tile_kernel<kLimKoren>);
      case kLimCada: return run(recon_tile_kernel<kLimCada>);
      case kLimWENO3: return run(recon_tile_kernel<kLimWENO3>);
      default: return run(recon_tile_kernel<kLimWENO5>);
    }
  }
  // (a kernel, not hipMemsetAsync: the call may be part of a captured graph)
  if (fill) zero_kernel<<<1024, kThreads, 0, s>>>(out, (size_t)4 * 8 * NT * NT * nt);
  dim3 grid((NT * NT + 127) / 128, nt);
  recon_batch_kernel<<<grid, 128, 0, s>>>(NT, ng, lim, dx, W, out);
}

}  // namespace amr
