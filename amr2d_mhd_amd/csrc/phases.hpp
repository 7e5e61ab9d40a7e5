// Device code of the other phases of a step: constrained transport, ghost
// fills, the CFL bound and the refinement indicators.
#pragma once
#include "device.hpp"

namespace amr {

namespace {

// --------------------------------------------------------------------- CT
// CT2D.cpp:28-75 (CTtype 2) gas pressure and fast speed of one cell of the
// stage state q (the reference's per-block p and C arrays, formed here per
// corner for the four cells around it, by the same expressions)
__device__ inline void ct2_pc(const double* q, int N2, int c, double g, double& p, double& C) {
  const double q0 = q[c], q1 = q[N2 + c], q2 = q[2 * N2 + c], q3 = q[3 * N2 + c], q4 = q[4 * N2 + c],
               q5 = q[5 * N2 + c], q6 = q[6 * N2 + c], q7 = q[7 * N2 + c];
  p = (g - 1) * (q4 - 0.5 * ((q1 * q1 + q2 * q2 + q3 * q3) / q0 + (q5 * q5 + q6 * q6 + q7 * q7)));
  C = sqrt((g * p + (q5 * q5 + q6 * q6 + q7 * q7)) / q0);
}

// CT2D.cpp:28-75: the CTtype 2 ("upwind") weight at the corner of cell c:
// psi = dPx / (dPx + dPy) where the pressure jump around the corner exceeds half
// the smallest pressure (sw1) and the flow is compressive beyond a tenth of the
// smallest fast speed (sw2), else 0.5; the velocity divergence keeps the
// reference's terms as written (two y-velocity quotients divide q2 by itself,
// CT2D.cpp:45).  q is the stage state (Us, or U on the last stage).
template <int NT>
__device__ inline double ct2_weight(const double* q, int c, double g) {
  constexpr int N2 = NT * NT;
  // cells (i, j), (i, j-1), (i-1, j), (i-1, j-1) of the reference's [i][j]
  const int c00 = c, c0m = c - NT, cm0 = c - 1, cmm = c - 1 - NT;
  double p00, p0m, pm0, pmm, C00, C0m, Cm0, Cmm;
  ct2_pc(q, N2, c00, g, p00, C00);
  ct2_pc(q, N2, c0m, g, p0m, C0m);
  ct2_pc(q, N2, cm0, g, pm0, Cm0);
  ct2_pc(q, N2, cmm, g, pmm, Cmm);
  const double beta = 0.5, delta = 0.1;
  const double dPx = 0.5 * fabs(p00 + p0m - pm0 - pmm);
  const double dPy = 0.5 * fabs(p00 + pm0 - p0m - pmm);
  const double* q0 = q;
  const double* q1 = q + N2;
  const double* q2 = q + 2 * N2;
  const double divV = 0.5 * (q1[c00] / q0[c00] + q1[c0m] / q0[c0m] - q1[cm0] / q0[cm0] - q1[cmm] / q0[cmm]) +
                      0.5 * (q2[c00] / q0[c00] + q2[cm0] / q2[cm0] - q2[c0m] / q2[c0m] - q2[cmm] / q0[cmm]);
  double tP = pmm < p0m ? pmm : p0m;
  const double tP1 = pm0 < p00 ? pm0 : p00;
  tP = tP < tP1 ? tP : tP1;
  const bool sw1 = (dPx + dPy) > beta * tP;
  double tC = Cmm < C0m ? Cmm : C0m;
  const double tC1 = Cm0 < C00 ? Cm0 : C00;
  tC = tC < tC1 ? tC : tC1;
  const bool sw2 = (-delta * tC) > divV;
  double psi = 0.5;
  if (sw1 && sw2) psi = dPx / (dPx + dPy);
  return psi;
}

// CT2D.cpp:15-75: corner EMF from the face fluxes for i,j in [1,NT-1].
// CTtype 1: the mean of the four face values.  CTtype 2: the y-flux and x-flux
// pairs weighted 1 - psi and psi.
template <int NT>
__device__ inline void emf_cell(const FieldPtrs& F, const LeafItem L, const InstParams* __restrict__ ip, int last,
                                DevError* err, int step, int c) {
  constexpr int N2 = NT * NT;
  const int i = c % NT, j = c / NT;
  if (i < 1 || j < 1) return;
  const double* gg5 = F.f[kGG] + (size_t)L.gs * 8 * N2 + 5 * N2;
  const double* ff6 = F.f[kFF] + (size_t)L.gs * 8 * N2 + 6 * N2;
  const InstParams& P = ip[L.inst];
  if (P.ct_type != 2) {
    F.f[kEMF][(size_t)L.gs * N2 + c] = 0.25 * ((gg5[c - 1] + gg5[c]) - (ff6[c - NT] + ff6[c]));
    return;
  }
  const double psi = ct2_weight<NT>(F.f[last ? kU : kUs] + (size_t)L.gs * 8 * N2, c, P.gamma);
  if (psi < 0 || psi > 1) report(err, L.inst, error_key(step, kSeqCt | L.nb, 0, i, j, 0, L.nb, kErrCtPsi));
  F.f[kEMF][(size_t)L.gs * N2 + c] = 0.5 * (1. - psi) * (gg5[c - 1] + gg5[c]) - 0.5 * psi * (ff6[c - NT] + ff6[c]);
}

template <int NT>
__global__ __launch_bounds__(kThreads) void emf_kernel(FieldPtrs F, const LeafItem* __restrict__ leaves,
                                                       const InstParams* __restrict__ ip, int last, DevError* err,
                                                       int step, const int32_t* __restrict__ counts) {
  if (counts && (int)blockIdx.y >= counts[kCountLeaves]) return;
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c < NT * NT) emf_cell<NT>(F, leaves[blockIdx.y], ip, last, err, step, c);
}

// CT2D.cpp:78-92: face-B RK update from the edge EMF.  Stage input B (Bi for
// step 1, else Bis), written array Bn (Bi on the last stage, else Bis) and
// the step's starting value B0 = Bi; SSP-RK3 stages 2-3 are build-defined.
__device__ inline double face_rk(int rk, int step, double B, double Bn, double B0, double dt, double res) {
  if (step == 1) return B - dt * res;
  if (rk == 2) return 0.5 * (B + Bn - dt * res);
  if (step == 2) return 0.75 * B0 + 0.25 * (B - dt * res);
  return (1. / 3.) * B0 + (2. / 3.) * (B - dt * res);
}

template <int NT>
__device__ inline void bupdate_cell(const FieldPtrs& F, const LeafItem L, const InstParams* __restrict__ ip, int step,
                                    int rk, int c) {
  constexpr int N2 = NT * NT;
  const int i = c % NT, j = c / NT;
  const InstParams& P = ip[L.inst];
  const double dt = P.dt, dxl = P.dx[L.lev];
  const double* E = F.f[kEMF] + (size_t)L.gs * N2;
  const double* B = F.f[step == 1 ? kBi : kBis] + (size_t)L.gs * 2 * N2;
  const double* B0 = F.f[kBi] + (size_t)L.gs * 2 * N2;
  double* Bn = F.f[step == rk ? kBi : kBis] + (size_t)L.gs * 2 * N2;
  const int cjp = j < NT - 1 ? c + NT : c;
  const int cip = i < NT - 1 ? c + 1 : c;
  const double rx = (1. / dxl) * (E[cjp] - E[c]);
  const double ry = -(1. / dxl) * (E[cip] - E[c]);
  const double bx = face_rk(rk, step, B[c], Bn[c], B0[c], dt, rx);
  const double by = face_rk(rk, step, B[N2 + c], Bn[N2 + c], B0[N2 + c], dt, ry);
  Bn[c] = bx;
  Bn[N2 + c] = by;
}

template <int NT>
__global__ __launch_bounds__(kThreads) void bupdate_kernel(FieldPtrs F, const LeafItem* __restrict__ leaves,
                                                           const InstParams* __restrict__ ip, int step, int rk,
                                                           const int32_t* __restrict__ counts) {
  if (counts && (int)blockIdx.y >= counts[kCountLeaves]) return;
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c < NT * NT) bupdate_cell<NT>(F, leaves[blockIdx.y], ip, step, rk, c);
}

// CT2D.cpp:95-123: cell-centred B from the updated faces Bn + energy correction
template <int NT>
__device__ inline void sync_cell(const double* Bn, double* q, int c, double q4, double q5, double q6) {
  constexpr int N2 = NT * NT;
  const int i = c % NT, j = c / NT;
  const int ip = i < NT - 1 ? i + 1 : i, jp = j < NT - 1 ? j + 1 : j;
  const double bx = 0.5 * (Bn[j * NT + ip] + Bn[j * NT + ip - 1]);
  const double by = 0.5 * (Bn[N2 + jp * NT + i] + Bn[N2 + (jp - 1) * NT + i]);
  q[4 * N2 + c] = q4 + 0.5 * ((bx * bx + by * by) - ((q5 * q5) + (q6 * q6)));
  q[5 * N2 + c] = bx;
  q[6 * N2 + c] = by;
}

template <int NT>
__device__ inline void bsync_cell(const FieldPtrs& F, const LeafItem L, int last, int c) {
  constexpr int N2 = NT * NT;
  double* q = F.f[last ? kU : kUs] + (size_t)L.gs * 8 * N2;
  sync_cell<NT>(F.f[last ? kBi : kBis] + (size_t)L.gs * 2 * N2, q, c, q[4 * N2 + c], q[5 * N2 + c], q[6 * N2 + c]);
}

template <int NT>
__global__ __launch_bounds__(kThreads) void bsync_kernel(FieldPtrs F, const LeafItem* __restrict__ leaves, int last,
                                                         const int32_t* __restrict__ counts) {
  if (counts && (int)blockIdx.y >= counts[kCountLeaves]) return;
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c < NT * NT) bsync_cell<NT>(F, leaves[blockIdx.y], last, c);
}

// -------------------------------------------------------------- ghost fill
// Single-pass execution of a compiled fill program.  Every destination's value
// is a function of the pre-fill state only; a workgroup evaluates all values
// of its chunk of ops, synchronises, then writes them.  The compiler places
// each op that reads an element some other op writes in the same chunk as
// that writer, so reads always see pre-fill values.
struct FillCtx {
  const double* base;
  int nv, kind, N2, NT;
  const FillGen* gen;
};

__device__ inline double fill_elem(const FillCtx& f, int64_t gs, int cell, int k) {
  return f.base[((size_t)gs * f.nv + k) * f.N2 + cell];
}

// explicit operand of a general restriction (always a pre-fill element)
__device__ inline double fill_ref(const FillCtx& f, int64_t ref, int k) {
  return fill_elem(f, ref >> 16, (int)(ref & 0xffff), k);
}

// boundary.cpp (0.25 x 2x2 sum in misc.cpp:35-48 order), boundaryfc.cpp
// (0.5 x face pair: along j for component 0, along i otherwise) and
// boundaryec.cpp (injection); v[] holds (i1,j1),(i1,j1+1),(i1+1,j1),(i1+1,j1+1)
__device__ inline double restrict_combine(int kind, int k, double v00, double v01, double v10, double v11) {
  double v = 0.;
  if (kind == kFillCell) {
    v += v00;
    v += v01;
    v += v10;
    v += v11;
    return 0.25 * v;
  }
  if (kind == kFillFace) {
    v += v00;
    v += k == 0 ? v01 : v10;
    return 0.5 * v;
  }
  return v00;
}

__device__ inline double gen_value(const FillCtx& f, const FillGen& g, int k) {
  return restrict_combine(f.kind, k, fill_ref(f, g.ref[0], k), fill_ref(f, g.ref[1], k), fill_ref(f, g.ref[2], k),
                          fill_ref(f, g.ref[3], k));
}

__device__ inline double fill_value(const FillCtx& f, const FillOp& op, int k) {
  if (op.op == kFillCopy) return fill_elem(f, op.src, op.src_cell, k);
  if (op.op == kFillRestrict) {
    const int a = op.src_cell;
    return restrict_combine(f.kind, k, fill_elem(f, op.src, a, k), fill_elem(f, op.src, a + f.NT, k),
                            fill_elem(f, op.src, a + 1, k), fill_elem(f, op.src, a + 1 + f.NT, k));
  }
  return gen_value(f, f.gen[op.src], k);
}

// The program is a concatenation of per-instance segments of whole chunks:
// chunk w belongs to the instance q with cprefix[q] <= w < cprefix[q+1].
struct FillProgram {
  const FillOp* const* ops;
  const FillGen* const* gen;
  const int32_t* cprefix;
  int ninst;
};

__device__ inline int find_segment(const FillProgram& P, int w) {
  int lo = 0, hi = P.ninst;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (P.cprefix[mid] <= w) lo = mid;
    else hi = mid;
  }
  return lo;
}

template <int NV>
__device__ inline void fill_field(const FillCtx& f, double* base, const FillOp& op, bool live) {
  double v[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = live ? fill_value(f, op, k) : 0.;
  __syncthreads();  // every read of the chunk precedes every write
  if (live) {
#pragma unroll
    for (int k = 0; k < NV; k++) base[((size_t)op.dst_gs * NV + k) * f.N2 + op.dst_cell] = v[k];
  }
}

// One chunk of the program per kFillChunk lanes (`lane` within the chunk); a
// workgroup may run several chunks side by side, and every lane of it calls
// this together (it synchronises the workgroup).  valid = false: no chunk.
__device__ inline void fill_chunk(const FillProgram& P, const FillSet& set, int NT, int w, int lane, bool valid) {
  FillOp op{};
  op.op = kFillNop;
  int q = 0;
  if (valid) {
    q = find_segment(P, w);
    op = P.ops[q][(w - P.cprefix[q]) * kFillChunk + lane];
  }
  const bool live = op.op != kFillNop;
  for (int fi = 0; fi < set.n; fi++) {
    const FillCtx f{set.base[fi], set.nv[fi], set.kind[fi], NT * NT, NT, valid ? P.gen[q] : nullptr};
    if (set.nv[fi] == 8) fill_field<8>(f, set.base[fi], op, live);
    else if (set.nv[fi] == 2) fill_field<2>(f, set.base[fi], op, live);
    else fill_field<1>(f, set.base[fi], op, live);
  }
}

// restrict_combine for a kind fixed at compile time (the same IEEE
// operations, no branch on the kind between an op's loads)
template <int KIND>
__device__ inline double restrict_kind(int k, double v00, double v01, double v10, double v11) {
  double v = 0.;
  if constexpr (KIND == kFillCell) {
    v += v00;
    v += v01;
    v += v10;
    v += v11;
    return 0.25 * v;
  } else if constexpr (KIND == kFillFace) {
    v += v00;
    v += k == 0 ? v01 : v10;
    return 0.5 * v;
  } else {
    return v00;
  }
}

// the NV components of one field of combine kind KIND for an op whose
// operands are the elements e[t] (block slot << 16 | cell): one (copy) or
// four (restriction, 2x2 order)
template <int NV, int KIND, bool COPY>
__device__ inline void fill_gather(const double* __restrict__ base, int N2, const int64_t* e, double* v) {
  if constexpr (COPY) {
    const double* p = base + (size_t)(e[0] >> 16) * NV * N2 + (e[0] & 0xffff);
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = p[(size_t)k * N2];
  } else {
    const double* p0 = base + (size_t)(e[0] >> 16) * NV * N2 + (e[0] & 0xffff);
    const double* p1 = base + (size_t)(e[1] >> 16) * NV * N2 + (e[1] & 0xffff);
    const double* p2 = base + (size_t)(e[2] >> 16) * NV * N2 + (e[2] & 0xffff);
    const double* p3 = base + (size_t)(e[3] >> 16) * NV * N2 + (e[3] & 0xffff);
#pragma unroll
    for (int k = 0; k < NV; k++)
      v[k] = restrict_kind<KIND>(k, p0[(size_t)k * N2], p1[(size_t)k * N2], p2[(size_t)k * N2], p3[(size_t)k * N2]);
  }
}

// The same for a set of up to three fields with NV0, NV1, NV2 components
// (0: absent) and combine kinds K0, K1, K2, fixed at compile time: every value
// of every field of the chunk is read before the one barrier, then all are
// written.  The op's kind and operand elements are decoded once, outside the
// loops over fields and components, so that all of an op's loads are in
// flight together (branches per component made each component's loads wait
// for the previous ones).
template <int NV0, int NV1, int NV2, int K0, int K1, int K2>
__device__ inline void fill_chunk_nv(const FillProgram& P, const FillSet& set, int NT, int w, int lane, bool valid) {
  FillOp op{};
  op.op = kFillNop;
  int q = 0;
  if (valid) {
    q = find_segment(P, w);
    op = P.ops[q][(w - P.cprefix[q]) * kFillChunk + lane];
  }
  const bool live = op.op != kFillNop;
  const int N2 = NT * NT;
  double v0[NV0 > 0 ? NV0 : 1], v1[NV1 > 0 ? NV1 : 1], v2[NV2 > 0 ? NV2 : 1];
  if (live) {
    int64_t e[4];
    if (op.op == kFillCopy) {
      e[0] = src_ref(op.src, op.src_cell);
      if constexpr (NV0 > 0) fill_gather<NV0, K0, true>(set.base[0], N2, e, v0);
      if constexpr (NV1 > 0) fill_gather<NV1, K1, true>(set.base[1], N2, e, v1);
      if constexpr (NV2 > 0) fill_gather<NV2, K2, true>(set.base[2], N2, e, v2);
    } else {
      if (op.op == kFillRestrict) {
        const int a = op.src_cell;
        e[0] = src_ref(op.src, a);
        e[1] = src_ref(op.src, a + NT);
        e[2] = src_ref(op.src, a + 1);
        e[3] = src_ref(op.src, a + 1 + NT);
      } else {
        const FillGen& g = P.gen[q][op.src];
#pragma unroll
        for (int t = 0; t < 4; t++) e[t] = g.ref[t];
      }
      if constexpr (NV0 > 0) fill_gather<NV0, K0, false>(set.base[0], N2, e, v0);
      if constexpr (NV1 > 0) fill_gather<NV1, K1, false>(set.base[1], N2, e, v1);
      if constexpr (NV2 > 0) fill_gather<NV2, K2, false>(set.base[2], N2, e, v2);
    }
  }
  __syncthreads();  // every read of the chunk precedes every write
  if (live) {
#pragma unroll
    for (int k = 0; k < NV0; k++) set.base[0][((size_t)op.dst_gs * NV0 + k) * N2 + op.dst_cell] = v0[k];
#pragma unroll
    for (int k = 0; k < NV1; k++) set.base[1][((size_t)op.dst_gs * NV1 + k) * N2 + op.dst_cell] = v1[k];
#pragma unroll
    for (int k = 0; k < NV2; k++) set.base[2][((size_t)op.dst_gs * NV2 + k) * N2 + op.dst_cell] = v2[k];
  }
}

// {U} or {U, Bi} (NB = 2) with a chunk's components over four workgroups, two each,
// and Bi's in a fifth (blockIdx.y)
template <int NB>
__global__ __launch_bounds__(kThreads) void fill_parts_kernel(FillProgram P, FillSet set, int NT,
                                                              const int32_t* __restrict__ counts) {
  if (blockIdx.y == 0)
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < set.copy_words; i += gridDim.x * kThreads)
      set.copy_dst[i] = set.copy_src[i];
  if (counts && (int)blockIdx.x >= counts[kCountChunks]) return;
  const int w = blockIdx.x, q = find_segment(P, w);
  const FillOp op = P.ops[q][(w - P.cprefix[q]) * kFillChunk + threadIdx.x];
  const int N2 = NT * NT;
  int64_t e[4] = {src_ref(op.src, op.src_cell), 0, 0, 0};
  if (op.op == kFillRestrict) {
    e[1] = e[0] + NT;
    e[2] = e[0] + 1;
    e[3] = e[0] + 1 + NT;
  } else if (op.op == kFillGeneral) {
    const FillGen& g = P.gen[q][op.src];
#pragma unroll
    for (int t = 0; t < 4; t++) e[t] = g.ref[t];
  }
  auto run = [&](int nv, int k0, double* base, auto combine) {
    constexpr int N = 2;
    double v[N];
    if (op.op != kFillNop) {
      const double* p0 = base + ((size_t)(e[0] >> 16) * nv + k0) * N2 + (e[0] & 0xffff);
      if (op.op == kFillCopy) {
#pragma unroll
        for (int k = 0; k < N; k++) v[k] = p0[(size_t)k * N2];
      } else {
        const double* p1 = base + ((size_t)(e[1] >> 16) * nv + k0) * N2 + (e[1] & 0xffff);
        const double* p2 = base + ((size_t)(e[2] >> 16) * nv + k0) * N2 + (e[2] & 0xffff);
        const double* p3 = base + ((size_t)(e[3] >> 16) * nv + k0) * N2 + (e[3] & 0xffff);
#pragma unroll
        for (int k = 0; k < N; k++)
          v[k] = combine(k, p0[(size_t)k * N2], p1[(size_t)k * N2], p2[(size_t)k * N2], p3[(size_t)k * N2]);
      }
    }
    __syncthreads();  // every read of the chunk precedes every write
    if (op.op != kFillNop) {
      double* o = base + ((size_t)op.dst_gs * nv + k0) * N2 + op.dst_cell;
#pragma unroll
      for (int k = 0; k < N; k++) o[(size_t)k * N2] = v[k];
    }
  };
  if (NB && blockIdx.y == 4)
    run(2, 0, set.base[1],
        [](int k, double a, double b, double c, double d) { return restrict_kind<kFillFace>(k, a, b, c, d); });
  else
    run(8, blockIdx.y * 2, set.base[0],
        [](int k, double a, double b, double c, double d) { return restrict_kind<kFillCell>(k, a, b, c, d); });
}

// The step's other field sets (engine.cpp) with their combine kinds: {U, Bi},
// {Bi, ff, gg}, {ff, gg}, one cell field, one face field, EMF; any other set takes
// the per-field path.
template <int NV0, int NV1, int NV2, int K0, int K1, int K2>
__global__ __launch_bounds__(kThreads) void fill_kernel_nv(FillProgram P, FillSet set, int NT,
                                                           const int32_t* __restrict__ counts) {
  for (int i = blockIdx.x * kThreads + threadIdx.x; i < set.copy_words; i += gridDim.x * kThreads)
    set.copy_dst[i] = set.copy_src[i];
  if (counts && (int)blockIdx.x >= counts[kCountChunks]) return;
  fill_chunk_nv<NV0, NV1, NV2, K0, K1, K2>(P, set, NT, blockIdx.x, threadIdx.x, true);
}

// --------------------------------------------- constrained transport, fused
// The flux fills of a stage and CT2D.cpp:11-124 as two launches where every block
// a program reads or writes is a leaf (the others run fill, emf, fill, bupdate,
// fill and bsync as launches of their own): ct_emf_kernel forms the corner EMF
// and its ghost fill, ct_faces_kernel the face update, its ghost fill and the
// cell sync.  A fill applied to a value that its source block forms in the same
// phase is that formula evaluated at the source cell, so a ghost element needs
// nothing another workgroup writes: one workgroup a leaf, its ring's ops from the
// table by destination, and the filled fluxes looked up the same way.  What is
// read at other blocks is not written in the same launch: the EMF goes to a
// scratch copy (`emf`) from which the second kernel reads, the faces a stage
// updates in place (all but the first stage's) are read from a copy the first
// kernel made (`old`), and workgroups past the leaves' fill in memory what the
// other kernel reads: Bi with ct_emf_kernel (the first stage's second fill of
// it: its linked tails), the fluxes with ct_faces_kernel.
//
// A stage's fill and CT as six launches, each at the floor of launch and latency,
// then as these two: 19.4 -> 9.0 us at 16 blocks, 26.1 -> 12.8 at 180, 34.8 ->
// 19.4 at 430 on average over the two stages.  The leaves' part is bound by the
// chain of dependent loads (leaf, table entries, operands): a loop over the cells
// with 256 lanes, or a load of the source's level before its cell size, took 9 us
// more at 180 blocks.  The last stage's flux fill is bound by the cache lines of
// the ghost columns (two of 16 elements of each used): 9.4 us of the kernel at
// 180 blocks against 6.2 in the first stage; with both fields in a lane 12.1.
struct CtArgs {
  FieldPtrs F;
  const LeafItem* leaves;
  const InstParams* ip;
  const FillGen* const* gen;
  const uint64_t* ring;  // [slot][ring_cells]
  uint32_t version;
  int step, rk;
  double* emf;           // [slot][N2]
  double* old;           // [slot][2][N2]: the updated faces before the stage
  double* rdx;           // [slot] 1 / dx of the leaf, by ct_emf_kernel for ct_faces_kernel
  DevError* err;
  int nleaf;
  FillProgram tail, all;   // the programs' linked tails, and the whole programs
  int ntail, nall;         // chunks that the launch's workgroups past the leaves run
};

// one lane a cell: a workgroup's loads are one round of memory latency each
// (leaf, ring entry, operands); at least one fill chunk a workgroup
template <int NT>
constexpr int kCtLanes = (NT * NT + 63) / 64 * 64 < kFillChunk ? kFillChunk : (NT * NT + 63) / 64 * 64;
template <int NT>
constexpr int kCtChunks = kCtLanes<NT> / kFillChunk;  // fill chunks an extra workgroup runs

// workgroups of a field's n chunks of linked tails (kept whole) and of unlinked ops
template <int NT>
__host__ __device__ constexpr int ct_tail_wgs(int n) { return (n + kCtChunks<NT> - 1) / kCtChunks<NT>; }
template <int NT>
__host__ __device__ constexpr int ct_flux_wgs(int n) { return (n * kFillChunk + kCtLanes<NT> - 1) / kCtLanes<NT>; }

// workgroup wg of a field's linked tails
template <int NT, int NV>
__device__ inline void ct_fill_tails(const CtArgs& A, double* field, int wg) {
  const int sub = threadIdx.x / kFillChunk, w = wg * kCtChunks<NT> + sub;
  FillSet set{};
  set.base[0] = field;
  fill_chunk_nv<NV, 0, 0, kFillFace, 0, 0>(A.tail, set, NT, w, threadIdx.x % kFillChunk,
                                           sub < kCtChunks<NT> && w < A.ntail);
}

// Workgroup wg of a flux field's unlinked ops, which read nothing that a fill
// writes, so that any lane may run any of them.  All of them in the last
// stage; before it memory has to hold only (besides what the linked tails read)
// the face x = LO of a row (ff) and y = LO of a column (gg), which the next
// stage's residual of the ghost cells beside them reads: an eighth of the ring in
// one of the two fields.  The rest is written by the last stage.
template <int NT, int NG>
__device__ inline void ct_fill_fluxes(const CtArgs& A, double* field, bool isx, int wg) {
  constexpr int N2 = NT * NT, LO = NG - 1;
  const int e = wg * kCtLanes<NT> + threadIdx.x, w = e / kFillChunk;
  if (w >= A.nall) return;
  const int q = find_segment(A.all, w), k = w - A.all.cprefix[q];
  if (k >= A.all.cprefix[q + 1] - A.all.cprefix[q] - (A.tail.cprefix[q + 1] - A.tail.cprefix[q])) return;
  const FillOp op = A.all.ops[q][k * kFillChunk + e % kFillChunk];
  if (op.op == kFillNop || (A.step != A.rk && (isx ? op.dst_cell % NT : op.dst_cell / NT) != LO)) return;
  int64_t e0 = src_ref(op.src, op.src_cell), ei = e0, ej = e0;
  if (op.op == kFillRestrict) {
    ei = e0 + 1;
    ej = e0 + NT;
  } else if (op.op == kFillGeneral) {
    const FillGen& g = A.all.gen[q][op.src];
    e0 = g.ref[0];
    ej = g.ref[1];
    ei = g.ref[2];
  }
  const bool copy = op.op == kFillCopy;
  double* o = field + (size_t)op.dst_gs * 8 * N2 + op.dst_cell;
  const double* p0 = field + (size_t)(e0 >> 16) * 8 * N2 + (e0 & 0xffff);
  const double* pi = field + (size_t)(ei >> 16) * 8 * N2 + (ei & 0xffff);
  const double* pj = field + (size_t)(ej >> 16) * 8 * N2 + (ej & 0xffff);
  double v[8], r[8];  // (a copy's second operand is its first)
#pragma unroll
  for (int c = 0; c < 8; c++) {
    v[c] = p0[c * N2];
    r[c] = (c ? pi : pj)[c * N2];
  }
#pragma unroll
  for (int c = 0; c < 8; c++) o[c * N2] = copy ? v[c] : restrict_kind<kFillFace>(c, v[c], r[c], r[c], 0.);
}

// where element x of slot gs takes its filled value from: offsets into a field of
// eight components, of one element or of the two of a face pair
struct FaceRef {
  size_t o0, o1;
  bool pair;
};
template <int NT, int NG>
__device__ AMR_INLINE FaceRef face_ref(const CtArgs& A, const FillGen* gen, int64_t gs, int x) {
  constexpr int N2 = NT * NT, R = ring_cells(NT, NG);
  const int r = ring_index(NT, NG, x % NT, x / NT);
  const uint64_t e = r < 0 ? 0 : A.ring[(size_t)gs * R + r];
  size_t o0 = (size_t)gs * 8 * N2 + x, o1 = o0;
  bool pair = false;
  if ((e >> 40) == A.version) {
    const int op = (int)((e >> 38) & 3);
    o0 = (size_t)(e & 0xfffffff) * 8 * N2 + ((e >> 28) & 0x3ff);
    pair = op != kFillCopy;
    o1 = pair ? o0 + 1 : o0;
    if (op == kFillGeneral) {
      const FillGen& G = gen[e & 0xfffffff];
      const int64_t r0 = G.ref[0], r1 = G.ref[2];
      o0 = (size_t)(r0 >> 16) * 8 * N2 + (r0 & 0xffff);
      o1 = (size_t)(r1 >> 16) * 8 * N2 + (r1 & 0xffff);
    }
  }
  return {o0, o1, pair};
}
// the filled value of a component other than the first
__device__ AMR_INLINE double face_filled(const FaceRef& r, double v0, double v1) {
  return r.pair ? restrict_combine(kFillFace, 1, v0, 0., v1, 0.) : v0;
}

template <int NT, int NG>
__global__ __launch_bounds__(kCtLanes<NT>) void ct_emf_kernel(CtArgs A) {
  constexpr int N2 = NT * NT, R = ring_cells(NT, NG);
  if ((int)blockIdx.x >= A.nleaf) return ct_fill_tails<NT, 2>(A, A.F.f[kBi], blockIdx.x - A.nleaf);
  const LeafItem L = A.leaves[blockIdx.x];
  const InstParams& P = A.ip[L.inst];
  const int last = A.step == A.rk, c = threadIdx.x;
  if (c == 0) A.rdx[L.gs] = 1. / P.dx[L.lev];
  if (c >= N2) return;
  const int r = ring_index(NT, NG, c % NT, c / NT);
  const uint64_t e = r < 0 ? 0 : A.ring[(size_t)L.gs * R + r];
  if (A.step > 1) {
    const double* B = A.F.f[last ? kBi : kBis] + (size_t)L.gs * 2 * N2;
    double* o = A.old + (size_t)L.gs * 2 * N2;
    const double b0 = B[c], b1 = B[N2 + c];
    o[c] = b0;
    o[N2 + c] = b1;
  }
  // the element whose pre-fill value this one takes (injection for restrictions)
  int64_t gs = L.gs;
  int a = c;
  if ((e >> 40) == A.version) {
    gs = (int64_t)(e & 0xfffffff);
    a = (int)((e >> 28) & 0x3ff);
    if (((e >> 38) & 3) == kFillGeneral) {
      const int64_t ref = A.gen[L.inst][gs].ref[0];
      gs = ref >> 16;
      a = (int)(ref & 0xffff);
    }
  }
  double v;
  if (a % NT < 1 || a < NT) {
    v = A.F.f[kEMF][(size_t)gs * N2 + a];  // row and column 0 keep what they hold
  } else {
    const double* gg5 = A.F.f[kGG] + 5 * N2;
    const double* ff6 = A.F.f[kFF] + 6 * N2;
    const FillGen* gen = A.gen[L.inst];
    const FaceRef rm = face_ref<NT, NG>(A, gen, gs, a - 1), r0 = face_ref<NT, NG>(A, gen, gs, a),
                  rj = face_ref<NT, NG>(A, gen, gs, a - NT);
    const double gm0 = gg5[rm.o0], gm1 = gg5[rm.o1], g00 = gg5[r0.o0], g01 = gg5[r0.o1], fj0 = ff6[rj.o0],
                 fj1 = ff6[rj.o1], f00 = ff6[r0.o0], f01 = ff6[r0.o1];
    const double g0 = face_filled(rm, gm0, gm1), g1 = face_filled(r0, g00, g01), f0 = face_filled(rj, fj0, fj1),
                 f1 = face_filled(r0, f00, f01);
    if (P.ct_type != 2) {
      v = 0.25 * ((g0 + g1) - (f0 + f1));
    } else {
      // (the range check of the weight, CT2D.cpp:60, where a block keeps its own
      // value: a quotient a / (a + b) of magnitudes cannot leave [0, 1])
      const double psi = ct2_weight<NT>(A.F.f[last ? kU : kUs] + (size_t)gs * 8 * N2, a, P.gamma);
      if ((psi < 0 || psi > 1) && gs == L.gs && a == c)
        report(A.err, L.inst, error_key(A.step, kSeqCt | L.nb, 0, c % NT, c / NT, 0, L.nb, kErrCtPsi));
      v = 0.5 * (1. - psi) * (g0 + g1) - 0.5 * psi * (f0 + f1);
    }
  }
  A.emf[(size_t)L.gs * N2 + c] = v;
}

// both components of the updated faces at cell c of slot gs
template <int NT>
__device__ AMR_INLINE void face_values(const CtArgs& A, double dt, int64_t gs, int c, double* v) {
  constexpr int N2 = NT * NT;
  const double* E = A.emf + (size_t)gs * N2;
  const size_t t2 = (size_t)gs * 2 * N2;
  const double* Bi = A.F.f[kBi] + t2;
  const double* old = A.old + t2;  // of the array the stage updates in place
  const bool last = A.step == A.rk;
  const double* B = A.step == 1 ? Bi : last ? A.F.f[kBis] + t2 : old;
  const double* B0 = A.step == 1 ? Bi : last ? old : Bi;  // the step's starting faces
  const int i = c % NT, j = c / NT;
  const double e0 = E[c], ej = E[j < NT - 1 ? c + NT : c], ei = E[i < NT - 1 ? c + 1 : c];
  const double bx = B[c], by = B[N2 + c], b0x = B0[c], b0y = B0[N2 + c];
  const double rdx = A.rdx[gs];
  // face_rk: its Bn (RK2's second stage) is the starting value too
  v[0] = face_rk(A.rk, A.step, bx, b0x, b0x, dt, rdx * (ej - e0));
  v[1] = face_rk(A.rk, A.step, by, b0y, b0y, dt, -rdx * (ei - e0));
}

template <int NT, int NG>
__global__ __launch_bounds__(kCtLanes<NT>) __attribute__((amdgpu_waves_per_eu(7))) void ct_faces_kernel(CtArgs A) {
  constexpr int N2 = NT * NT, R = ring_cells(NT, NG);
  __shared__ double sB[2 * N2];
  if ((int)blockIdx.x >= A.nleaf) {
    const int w = blockIdx.x - A.nleaf, n = ct_tail_wgs<NT>(A.ntail);
    double* field = A.F.f[w & 1 ? kGG : kFF];
    if (w / 2 < n) ct_fill_tails<NT, 8>(A, field, w / 2);
    else ct_fill_fluxes<NT, NG>(A, field, !(w & 1), w / 2 - n);
    return;
  }
  const LeafItem L = A.leaves[blockIdx.x];
  const double dt = A.ip[L.inst].dt;
  const int last = A.step == A.rk, c = threadIdx.x;
  double* q = A.F.f[last ? kU : kUs] + (size_t)L.gs * 8 * N2;
  double q4 = 0., q5 = 0., q6 = 0.;
  if (c < N2) {
    const int r = ring_index(NT, NG, c % NT, c / NT);
    const uint64_t e = r < 0 ? 0 : A.ring[(size_t)L.gs * R + r];
    q4 = q[4 * N2 + c];
    q5 = q[5 * N2 + c];
    q6 = q[6 * N2 + c];
    A.F.f[kEMF][(size_t)L.gs * N2 + c] = A.emf[(size_t)L.gs * N2 + c];
    // the cell itself, the copied one, or the three of a face pair's restriction
    // (along j for component 0, along i for component 1: restrict_combine)
    int64_t g0 = L.gs, gx = 0, gy = 0;
    int a0 = c, ax = 0, ay = 0;
    bool pair = false;
    if ((e >> 40) == A.version) {
      const int op = (int)((e >> 38) & 3);
      g0 = gx = gy = (int64_t)(e & 0xfffffff);
      a0 = (int)((e >> 28) & 0x3ff);
      pair = op != kFillCopy;
      ax = a0 + NT;
      ay = a0 + 1;
      if (op == kFillGeneral) {
        const FillGen& G = A.gen[L.inst][g0];
        const int64_t r0 = G.ref[0], rx = G.ref[1], ry = G.ref[2];
        g0 = r0 >> 16;
        a0 = (int)(r0 & 0xffff);
        gx = rx >> 16;
        ax = (int)(rx & 0xffff);
        gy = ry >> 16;
        ay = (int)(ry & 0xffff);
      }
    }
    double v[2];
    face_values<NT>(A, dt, g0, a0, v);
    if (pair) {
      double x[2], y[2];
      face_values<NT>(A, dt, gx, ax, x);
      face_values<NT>(A, dt, gy, ay, y);
      v[0] = restrict_combine(kFillFace, 0, v[0], x[0], 0., 0.);
      v[1] = restrict_combine(kFillFace, 1, v[1], 0., y[1], 0.);
    }
    double* Bn = A.F.f[last ? kBi : kBis] + (size_t)L.gs * 2 * N2;
    sB[c] = Bn[c] = v[0];
    sB[N2 + c] = Bn[N2 + c] = v[1];
  }
  __syncthreads();
  if (c < N2) sync_cell<NT>(sB, q, c, q4, q5, q6);
}

// ------------------------------------------------------ CFL and criteria
// main.cpp:209-230 (per-leaf wave-speed bound, with the reference's
// |rho|+c_fx and |u|+c_fy terms) fused with criteria.cpp:6-44 (maximum of
// the max4diff/|w| ratio over p, rho, Bx, By on the interior).  One leaf, all
// TPB lanes (a power of two); sW: 8 NT^2 doubles and sRed: 2 TPB doubles of
// the workgroup's LDS.  The maxima never hold a NaN (std_max keeps its first
// operand against one), so the reduction order does not change them.
template <int NT, int NG, int TPB>
__device__ inline void cfl_block(const FieldPtrs& F, const double* __restrict__ Win, const LeafItem L, int leaf,
                                 const InstParams* __restrict__ ip, double* lam_grad, DevError* err, double* sW,
                                 double* sRed) {
  constexpr int N2 = NT * NT;
  constexpr int LO = NG, HI = NT - 1 - NG;
  const double g = ip[L.inst].gamma;
  const int tid = threadIdx.x;
  if (Win) {
    const double* W = Win + (size_t)leaf * 8 * N2;
    for (int q = tid; q < 8 * N2; q += TPB) sW[q] = W[q];
  } else {
    const double* U = F.f[kU] + (size_t)L.gs * 8 * N2;
    for (int c = tid; c < N2; c += TPB) {
      double u[8], w[8];
#pragma unroll
      for (int k = 0; k < 8; k++) u[k] = U[k * N2 + c];
      cons_to_prim(u, g, w);
#pragma unroll
      for (int k = 0; k < 8; k++) sW[k * N2 + c] = w[k];
      const int i = c % NT, j = c / NT;
      if (w[4] <= 0 && i > LO - 1 && i < HI + 1 && j > LO - 1 && j < HI + 1)
        report(err, L.inst, error_key(kOrdCfl, L.nb, 0, i, j, 0, L.nb, kErrPressure));
    }
  }
  __syncthreads();
  double lam = 0., grad = 0.;
  constexpr int NI = HI - LO + 1;
  for (int q = tid; q < NI * NI; q += TPB) {
    const int i = LO + q % NI, j = LO + q / NI, c = j * NT + i;
    double w[8];
#pragma unroll
    for (int k = 0; k < 8; k++) w[k] = sW[k * N2 + c];
    if (!Win) {
      lam = std_max(lam, fabs(w[0]) + fast_speed(w, g, 5));
      lam = std_max(lam, fabs(w[1]) + fast_speed(w, g, 6));
    }
    const int vars[4] = {4, 0, 5, 6};
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const double* Wk = sW + vars[v] * N2;
      const double x = Wk[c];
      double m = fabs(Wk[c + 1] - x);
      m = mac_max(m, fabs(Wk[c - 1] - x));
      m = mac_max(m, fabs(Wk[c + NT] - x));
      m = mac_max(m, fabs(Wk[c - NT] - x));
      grad = std_max(grad, m / mac_max(kEps, fabs(x)));
    }
  }
  sRed[tid] = lam;
  sRed[TPB + tid] = grad;
  __syncthreads();
  for (int w = TPB / 2; w > 0; w >>= 1) {
    if (tid < w) {
      sRed[tid] = std_max(sRed[tid], sRed[tid + w]);
      sRed[TPB + tid] = std_max(sRed[TPB + tid], sRed[TPB + tid + w]);
    }
    __syncthreads();
  }
  if (tid == 0) {
    const double dxl = ip[L.inst].dx[L.lev];
    lam_grad[2 * leaf] = std_min(dxl, dxl) / sRed[0];
    lam_grad[2 * leaf + 1] = sRed[TPB];
  }
}

template <int NT, int NG>
__global__ __launch_bounds__(kThreads) void cfl_criteria_kernel(FieldPtrs F, const double* __restrict__ Win,
                                                                const LeafItem* __restrict__ leaves,
                                                                const InstParams* __restrict__ ip, double* lam_grad,
                                                                DevError* err, const int32_t* __restrict__ counts) {
  __shared__ double sW[8 * NT * NT];
  __shared__ double sRed[2 * kThreads];
  if (counts && (int)blockIdx.x >= counts[kCountLeaves]) return;
  cfl_block<NT, NG, kThreads>(F, Win, leaves[blockIdx.x], blockIdx.x, ip, lam_grad, err, sW, sRed);
}

}  // namespace

}  // namespace amr
