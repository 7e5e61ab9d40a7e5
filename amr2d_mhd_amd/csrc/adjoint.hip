// Frozen-mesh step and its discrete adjoint on one uniform periodic N x N grid.
//
// Forward: the reference's RK2 step (main.cpp:128-247) restricted to one
// level with exact periodic halos -- cons->prim, minmod MUSCL edge states
// with the normal B from the faces, HLLE, stage update, CT (corner EMF, face
// update, cell sync with the energy fix).  The arithmetic is that of the
// engine's kernels (physics.hpp), so on a single-level mesh it reproduces the
// engine bit for bit.
//
// Adjoint: the exact reverse of that discrete map (branch-wise at the
// limiter and wave-speed switches), written as gather kernels so the result
// is deterministic: per-face reverse sweeps store their contributions to the
// four stencil cells, and per-cell kernels sum them.
//
// Layout: U[8][N][N] (row j, column i, i fastest); Bx[j][i] is the x-face
// between cells i-1 and i, By[j][i] the y-face between rows j-1 and j;
// fluxes follow the faces; E[j][i] sits at the corner (i-1/2, j-1/2).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <mutex>

#include "../../include/amr2d_mhd.h"
#include "abi_guard.hpp"
#include "adjoint_math.hpp"
#include "stage.hpp"

using namespace amr;

namespace {

constexpr int kT = 256;

__device__ inline int wrap(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }
// i mod n for any i (tiles can be wider than small grids)
__device__ inline int wrap_any(int i, int n) { return ((i % n) + n) % n; }

struct Grid {
  int n;
  double dx, g;
  size_t n2;
};

// -------------------------------------------------------------- forward
// A stage is two launches.  k_fwd_faces: primitives and face fluxes of a tile
// of kFx x kFy cells, whose lower x and y faces it owns -- the primitives of the
// tile and of the three more columns and rows its faces read go through LDS,
// with the AMR stage's reconstruction, solver and range flags (stage.hpp).
// k_fwd_update: everything that follows the fluxes, a lane a cell: the stage
// update, the four corner EMFs around the cell, its two faces and the far ones
// its field averages read (formed twice rather than stored and read back), and
// the cell sync.  (Primitives, fluxes, update, EMF, faces and sync as a launch
// each took 70 us a stage at 512 x 512, HLLD, and six launch gaps.)
// Tiles of 16 x 8 with a lane a face, the x faces on the first two wavefronts, the
// y faces on the others: bound by the flux arithmetic of the three wavefronts a
// SIMD its registers allow and by how evenly the last of them fill the card.  A
// step at 150, 300 and 512 cells a side, HLLD: 24.0, 42.0 and 80.5 us; 8 x 8 tiles of
// 128 lanes 27.7, 43.7 and 87.3, 16 x 16 tiles of 256 lanes (x then y faces) 30.3,
// 48.2 and 87.2, 32 x 4 tiles 24.2, 41.8 and 78.4 but 31.7 against 20.8 at 100.
constexpr int kFx = 16, kFy = 8, kFaceLanes = 2 * kFx * kFy;

template <int SOLVER>
__global__ __launch_bounds__(kFaceLanes) __attribute__((amdgpu_waves_per_eu(3))) void k_fwd_faces(
    Grid G, const double* __restrict__ Q, const double* __restrict__ Bx, const double* __restrict__ By,
    double* __restrict__ W, double* __restrict__ Fx, double* __restrict__ Fy) {
  constexpr int P = kFx + 3, VS = P * (kFy + 3);
  __shared__ double sW[8 * VS];
  __shared__ int sFlags;
  const int tid = threadIdx.x, i0 = blockIdx.x * kFx, j0 = blockIdx.y * kFy;
  if (tid == 0) sFlags = 0;
  __syncthreads();
  for (int c = tid; c < VS; c += kFaceLanes) {
    const int ti = c % P, tj = c / P;  // cell (i0 + ti - 2, j0 + tj - 2)
    const bool ci = ti >= 2 && ti < 2 + kFx, cj = tj >= 2 && tj < 2 + kFy;
    if (!ci && !cj) continue;  // no face reads the corners
    const size_t e = (size_t)wrap_any(j0 + tj - 2, G.n) * G.n + wrap_any(i0 + ti - 2, G.n);
    double u[8], w[8];
#pragma unroll
    for (int k = 0; k < 8; k++) u[k] = Q[k * G.n2 + e];
    const int tile = tile_prim(u, G.g, w);
    if (tile) atomicOr(&sFlags, tile);
#pragma unroll
    for (int k = 0; k < 8; k++) sW[k * VS + c] = w[k];
    if (ci && cj && i0 + ti - 2 < G.n && j0 + tj - 2 < G.n) {
#pragma unroll
      for (int k = 0; k < 8; k++) W[k * G.n2 + e] = w[k];
    }
  }
  __syncthreads();
  const int tile = sFlags;
  const int dir = tid >= kFx * kFy, r = tid - dir * kFx * kFy;
  const int ci = r % kFx, cj = r / kFx;
  if (i0 + ci >= G.n || j0 + cj >= G.n) return;
  const size_t f = (size_t)(j0 + cj) * G.n + i0 + ci;
  const double* Wl = sW + (cj + 2 - dir) * P + ci + 1 + dir;  // the cell below the face
  double fl[8];
  tile_face_flux<kStageHLLDMuscl>(Wl, VS, dir ? P : 1, kLimMinmod, SOLVER, G.g, 1., dir ? By[f] : Bx[f], tile, dir, fl);
  double* F = dir ? Fy : Fx;
#pragma unroll
  for (int k = 0; k < 8; k++) F[k * G.n2 + f] = fl[k];
}

constexpr int kUx = 64, kUy = 4;  // cells of one workgroup of the per-cell kernels

struct FwdFaces {
  const double *B0x, *B0y;  // the step's input faces
  const double *Bsx, *Bsy;  // the first stage's (stage 2)
  double *Bnx, *Bny;        // the stage's faces
  double *Bcx, *Bcy;        // a copy of them, or null
};

// STAGE 1: out = U - dt res, Bn = B0 - dt r; 2: out = 0.5 (U + Us - dt res),
// Bn = 0.5 (Bs + B0 - dt r).  pre: the cell B before the sync.  out may be U (a lane
// reads its cell before it writes it); the faces written may not be faces read,
// which neighbours read too.
template <int STAGE>
__global__ __launch_bounds__(kUx* kUy) void k_fwd_update(Grid G, const double* U, const double* __restrict__ Us,
                                                         const double* __restrict__ Fx, const double* __restrict__ Fy,
                                                         FwdFaces B, double dt, double* out,
                                                         double* __restrict__ pre) {
  const int i = blockIdx.x * kUx + threadIdx.x % kUx, j = blockIdx.y * kUy + threadIdx.x / kUx;
  if (i >= G.n || j >= G.n) return;
  const int n = G.n, ip = wrap(i + 1, n), im = wrap(i - 1, n), jp = wrap(j + 1, n), jm = wrap(j - 1, n);
  const size_t n2 = G.n2, c = (size_t)j * n + i, cx = (size_t)j * n + ip, cy = (size_t)jp * n + i;
  double dF[8], dG[8], u[8], us[8], res[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const size_t o = k * n2;
    u[k] = U[o + c];
    if (STAGE == 2) us[k] = Us[o + c];
    dF[k] = Fx[o + cx] - Fx[o + c];
    dG[k] = Fy[o + cy] - Fy[o + c];
  }
  // corner EMF at (i, j), (i + 1, j), (i, j + 1), (i + 1, j + 1)
  const double* gy5 = Fy + 5 * n2;
  const double* fx6 = Fx + 6 * n2;
  auto emf = [&](int a, int am, int b, int bm) {
    return 0.25 * ((gy5[(size_t)b * n + am] + gy5[(size_t)b * n + a]) - (fx6[(size_t)bm * n + a] + fx6[(size_t)b * n + a]));
  };
  const double E00 = emf(i, im, j, jm), E10 = emf(ip, i, j, jm), E01 = emf(i, im, jp, j), E11 = emf(ip, i, jp, j);
  const double rdx = 1. / G.dx;
  auto face = [&](const double* B0, const double* Bs, size_t f, double r) {
    return STAGE == 1 ? B0[f] - dt * r : 0.5 * (Bs[f] + B0[f] - dt * r);
  };
  const double bx = face(B.B0x, B.Bsx, c, rdx * (E01 - E00)), bxp = face(B.B0x, B.Bsx, cx, rdx * (E11 - E10));
  const double by = face(B.B0y, B.Bsy, c, -rdx * (E10 - E00)), byp = face(B.B0y, B.Bsy, cy, -rdx * (E11 - E01));
  stage_residual(dF, dG, G.dx, res);
  double q[8];
#pragma unroll
  for (int k = 0; k < 8; k++) q[k] = STAGE == 1 ? u[k] - dt * res[k] : 0.5 * (u[k] + us[k] - dt * res[k]);
  const double mx = 0.5 * (bxp + bx), my = 0.5 * (byp + by);
  pre[c] = q[5];
  pre[n2 + c] = q[6];
  q[4] = q[4] + 0.5 * ((mx * mx + my * my) - ((q[5] * q[5]) + (q[6] * q[6])));
  q[5] = mx;
  q[6] = my;
#pragma unroll
  for (int k = 0; k < 8; k++) out[k * n2 + c] = q[k];
  B.Bnx[c] = bx;
  B.Bny[c] = by;
  if (STAGE == 2 && B.Bcx) {
    B.Bcx[c] = bx;
    B.Bcy[c] = by;
  }
}

// -------------------------------------------------------------- adjoint
// Tape of one step (doubles, N2 = N*N each unless stated): the primitive
// states the two flux passes read (W1 = prim(U), W2 = prim(Us), 8 N2 each),
// the stage-1 faces (Bxs, Bys), the pre-sync cell B of both stages (2 N2
// each) and the output faces (Bxo, Byo).
struct Tape {
  double *W1, *W2, *Bxs, *Bys, *pre1, *pre2, *Bxo, *Byo;
};
constexpr size_t kTapePerCell = 24;

Tape tape_at(double* base, size_t n2) {
  Tape t;
  t.W1 = base;
  t.W2 = base + 8 * n2;
  t.Bxs = base + 16 * n2;
  t.Bys = base + 17 * n2;
  t.pre1 = base + 18 * n2;
  t.pre2 = base + 20 * n2;
  t.Bxo = base + 22 * n2;
  t.Byo = base + 23 * n2;
  return t;
}

// edge states of one face: x faces (dir 0) take Bx as the normal component,
// y faces (dir 1) By, and are returned in the rotated frame (swap_xy)
template <bool FAST>
__device__ AMR_INLINE void face_states(Rev<FAST>& A, const Grid& G, const double* W, const double* Bn, int dir, int i,
                                       int j, double* wl, double* wr, size_t* cell) {
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int o = s - 2;
    cell[s] = dir == 0 ? (size_t)j * G.n + wrap(i + o, G.n) : (size_t)wrap(j + o, G.n) * G.n + i;
  }
#pragma unroll
  for (int k = 0; k < 8; k++) {
    double v[4];
    if (k == 5 + dir) continue;
#pragma unroll
    for (int s = 0; s < 4; s++) v[s] = W[k * G.n2 + cell[s]];
    recon_minmod(A, v, wl[k], wr[k]);
  }
  const double b = Bn[(size_t)j * G.n + i];
  if (dir == 0) {
    wl[5] = b;
    wr[5] = b;
  } else {
    wl[6] = b;
    wr[6] = b;
    swap_xy(wl);
    swap_xy(wr);
  }
}

// Reverse of a stage, two launches: k_rev_faces takes the adjoint Q of the
// synced state and of the faces back through the cell sync and the face update
// to the corner EMF (adjoint Eb) and the earlier faces; the face reverse
// (k_stage_vjp, or k_flux_vjp and k_gather_prim_vjp) forms the flux adjoints it
// needs from Q and Eb as it goes and passes Q on to the stage's inputs.  (The
// sync, the faces, the EMF and the flux adjoints as launches of their own, with
// 16 flux adjoints a cell written and read back, took 37 us a stage at
// 512 x 512.)
//
// Cell sync: E += 0.5 ((bx^2 + by^2) - (q5^2 + q6^2)), q5 <- bx, q6 <- by, so the
// averages' adjoints are bb = (Q5 + Q4 bx, Q6 + Q4 by) and the pre-sync state's
// are Q but -Q4 pre in components 5 and 6.  Faces: the updated faces' adjoint
// Bb = Bin + 0.5 (bb of both adjacent cells); stage 2 (Bn = 0.5 (Bs + B0 - dt r))
// assigns B0b = Bsb = 0.5 Bb, stage 1 (Bn = B0 - dt r) adds Bb to B0b.  EMF:
// rx_b = -s dt Bbx, ry_b = -s dt Bby (s = 1 or 0.5), rx = (1/dx) (E[j+1] - E[j]),
// ry = -(1/dx) (E[i+1] - E[i]).  Face values a corner needs beside the cell's own
// are formed again from the inputs, which no lane writes.
template <int STAGE>
__global__ __launch_bounds__(kUx* kUy) void k_rev_faces(Grid G, const double* __restrict__ Q,
                                                        const double* __restrict__ Bx, const double* __restrict__ By,
                                                        const double* __restrict__ Binx,
                                                        const double* __restrict__ Biny, double dt,
                                                        double* __restrict__ B0bx, double* __restrict__ B0by,
                                                        double* __restrict__ Bsbx, double* __restrict__ Bsby,
                                                        double* __restrict__ Eb) {
  const int i = blockIdx.x * kUx + threadIdx.x % kUx, j = blockIdx.y * kUy + threadIdx.x / kUx;
  if (i >= G.n || j >= G.n) return;
  const int n = G.n, ip = wrap(i + 1, n), im = wrap(i - 1, n), jp = wrap(j + 1, n), jm = wrap(j - 1, n);
  const size_t n2 = G.n2;
  auto at = [n](int a, int b) { return (size_t)b * n + a; };
  auto bbx = [&](int a, int ap, int b) {  // adjoint of the x average of cell (a, b)
    const size_t c = at(a, b);
    return Q[5 * n2 + c] + Q[4 * n2 + c] * (0.5 * (Bx[at(ap, b)] + Bx[c]));
  };
  auto bby = [&](int a, int b, int bp) {
    const size_t c = at(a, b);
    return Q[6 * n2 + c] + Q[4 * n2 + c] * (0.5 * (By[at(a, bp)] + By[c]));
  };
  const size_t c = at(i, j);
  const double x = Binx[c] + 0.5 * (bbx(i, ip, j) + bbx(im, i, j));
  const double y = Biny[c] + 0.5 * (bby(i, j, jp) + bby(i, jm, j));
  const double x_jm = Binx[at(i, jm)] + 0.5 * (bbx(i, ip, jm) + bbx(im, i, jm));
  const double y_im = Biny[at(im, j)] + 0.5 * (bby(im, j, jp) + bby(im, jm, j));
  if (STAGE == 2) {
    B0bx[c] = 0.5 * x;
    B0by[c] = 0.5 * y;
    Bsbx[c] = 0.5 * x;
    Bsby[c] = 0.5 * y;
  } else {
    B0bx[c] += x;
    B0by[c] += y;
  }
  const double s = STAGE == 1 ? -dt : -0.5 * dt;
  const double rxb_jm = s * x_jm, rxb = s * x, ryb_im = s * y_im, ryb = s * y;
  Eb[c] = (1. / G.dx) * (rxb_jm - rxb) - (1. / G.dx) * (ryb_im - ryb);
}

// what the face reverse reads: the stage's synced-state adjoint, the cell B
// before the sync, the corner EMF's adjoint, and where Q goes on to -- stage 2
// (out = 0.5 (U + Us - dt res)) assigns Ub = 0.5 Q and Qb = 0.5 Q + ..., stage 1
// (out = U - dt res) adds Q and the face contributions to Qb = Ub
struct RevIn {
  const double *Q, *pre, *Eb;
  double s;  // residual adjoint = s Q: -dt, or -0.5 dt in stage 2
};

// pre-sync state adjoint, component k
__device__ inline double presync(const Grid& G, const RevIn& R, int k, size_t c) {
  return k == 5 || k == 6 ? -R.Q[4 * G.n2 + c] * R.pre[(k - 5) * G.n2 + c] : R.Q[k * G.n2 + c];
}

// adjoints of the fluxes through the lower face of cell (i, j) in direction
// DIR: from the update's residual and from the EMF (components 6 of x, 5 of y)
template <int DIR, bool FAST>
__device__ AMR_INLINE void flux_adjoint(Rev<FAST>& A, const Grid& G, const RevIn& R, int i, int j, double* fb) {
  const size_t f = (size_t)j * G.n + i;
  const size_t l = DIR == 0 ? (size_t)j * G.n + wrap(i - 1, G.n) : (size_t)wrap(j - 1, G.n) * G.n + i;
  A.note_den(G.dx);
  const Den<FAST> dx = A.den(G.dx);
#pragma unroll
  for (int k = 0; k < 8; k++) fb[k] = R.s * presync(G, R, k, l) - R.s * presync(G, R, k, f);
#pragma unroll
  for (int k = 0; k < 8; k += 2) {
    A.note(fb[k], fb[k + 1]);
    fb[k] = A.over(fb[k], dx);
    fb[k + 1] = A.over(fb[k + 1], dx);
  }
  if (DIR == 0) fb[6] -= 0.25 * (R.Eb[f] + R.Eb[(size_t)wrap(j + 1, G.n) * G.n + i]);
  else fb[5] += 0.25 * (R.Eb[f] + R.Eb[(size_t)j * G.n + wrap(i + 1, G.n)]);
}

// Q on to the stage's inputs, with the face contributions ub
template <int STAGE>
__device__ inline void pass_state(const Grid& G, const RevIn& R, size_t c, const double* ub, double* Ub, double* Qb) {
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const double q = presync(G, R, k, c);
    const size_t e = k * G.n2 + c;
    if (STAGE == 2) {
      Ub[e] = 0.5 * q;
      Qb[e] = 0.5 * q + ub[k];
    } else {
      Qb[e] = (Qb[e] + q) + ub[k];
    }
  }
}

// Reverse of reconstruction + flux at one face (i, j) of direction DIR: the
// adjoints (wlb, wrb) of its two edge states in the grid frame.  Returns whether
// they hold (Rev).
template <int DIR, int SOLVER, bool FAST>
__device__ AMR_INLINE bool face_reverse_as(const Grid& G, int i, int j, const double* __restrict__ W,
                                           const double* __restrict__ Bn, const RevIn& R, double* wlb, double* wrb) {
  Rev<FAST> A;
  double wl[8], wr[8], fb[8];
  size_t cell[4];
  face_states(A, G, W, Bn, DIR, i, j, wl, wr, cell);
  flux_adjoint<DIR>(A, G, R, i, j, fb);
  for (int k = 0; k < 8; k++) wlb[k] = wrb[k] = 0.;
  if (DIR) swap_xy(fb);  // adjoint of the output swap
  if (SOLVER == kFluxHLLD) hlld_vjp(A, wl, wr, G.g, fb, wlb, wrb);
  else hlle_vjp(A, wl, wr, G.g, fb, wlb, wrb);
  if (DIR) {
    swap_xy(wlb);  // adjoint of the input swap
    swap_xy(wrb);
  }
  return A.ok();
}

// the same with plain quotients, into out[q * stride], q = 0 .. 15 (wlb, then wrb);
// out of line, for its registers (inlined, the kernels below spilled 335 of them)
template <int DIR, int SOLVER>
__device__ __attribute__((noinline)) void face_reverse_plain(Grid G, int i, int j, const double* W, const double* Bn,
                                                             RevIn R, double* out, size_t stride) {
  double wlb[8], wrb[8];
  face_reverse_as<DIR, SOLVER, false>(G, i, j, W, Bn, R, wlb, wrb);
  for (int k = 0; k < 8; k++) {
    out[k * stride] = wlb[k];
    out[(8 + k) * stride] = wrb[k];
  }
}

// the same with the FAST quotients where they are exact; also the stencil cells
// (i-2 .. i+1 along the normal).  mem, stride: as face_reverse_plain's out, this
// lane's own memory
template <int DIR, int SOLVER>
__device__ AMR_INLINE void face_reverse(const Grid& G, int i, int j, const double* __restrict__ W,
                                        const double* __restrict__ Bn, const RevIn& R, double* mem, size_t stride,
                                        double* wlb, double* wrb, size_t* cell) {
  if (!face_reverse_as<DIR, SOLVER, true>(G, i, j, W, Bn, R, wlb, wrb)) {
    face_reverse_plain<DIR, SOLVER>(G, i, j, W, Bn, R, mem, stride);
    for (int k = 0; k < 8; k++) {
      wlb[k] = mem[k * stride];
      wrb[k] = mem[(8 + k) * stride];
    }
  }
  // Recompute the stencil cells from opaque copies of (i, j) rather than
  // keep the four 64-bit offsets alive across the solver reverse.
  int io = i, jo = j;
  asm volatile("" : "+v"(io), "+v"(jo));
  for (int s = 0; s < 4; s++)
    cell[s] = DIR == 0 ? (size_t)jo * G.n + wrap(io + s - 2, G.n) : (size_t)wrap(jo + s - 2, G.n) * G.n + io;
}

// stencil contributions vb[s] of variable k (zero for the normal B, which the
// face takes from Bn) from the edge-state adjoints; out(k, vb)
template <int DIR, class Out>
__device__ inline void stencil_reverse(const Grid& G, const double* __restrict__ W, const size_t* cell,
                                       const double* wlb, const double* wrb, Out out) {
  constexpr int nc = DIR ? 6 : 5;
  // Re-read the stencil for the reconstruction reverse rather than keep the
  // 28 values face_states loaded alive across the HLLE reverse: the opaque
  // copy of the pointer stops the compiler from reusing those loads, which
  // would cost ~60 VGPRs and push the kernel to one wave per SIMD.
  const double* Wr = W;
  asm volatile("" : "+s"(Wr));
  for (int k = 0; k < 8; k++) {
    double vb[4] = {0., 0., 0., 0.};
    if (k != nc) {
      double v[4];
      for (int s = 0; s < 4; s++) v[s] = Wr[k * G.n2 + cell[s]];
      Rev<true> A;
      recon_minmod_vjp(A, v, wlb[k], wrb[k], vb);
      if (!A.ok()) {
        Rev<false> plain;
        for (int s = 0; s < 4; s++) vb[s] = 0.;
        recon_minmod_vjp(plain, v, wlb[k], wrb[k], vb);
      }
    }
    out(k, vb);
  }
}

template <int DIR, int SOLVER>
__device__ inline void flux_vjp_face(const Grid& G, size_t f, const double* __restrict__ W,
                                     const double* __restrict__ Bn, const RevIn& R, double* __restrict__ S,
                                     double* __restrict__ Bnb) {
  const int i = (int)(f % G.n), j = (int)(f / G.n);
  double wlb[8], wrb[8];
  size_t cell[4];
  face_reverse<DIR, SOLVER>(G, i, j, W, Bn, R, S + f, G.n2, wlb, wrb, cell);
  constexpr int nc = DIR ? 6 : 5;
  Bnb[f] += wlb[nc] + wrb[nc];
  stencil_reverse<DIR>(G, W, cell, wlb, wrb, [&](int k, const double* vb) {
    for (int s = 0; s < 4; s++) S[((size_t)s * 8 + k) * G.n2 + f] = vb[s];
  });
}

template <int DIR, int SOLVER>
__global__ __launch_bounds__(kT) void k_flux_vjp(Grid G, const double* __restrict__ W, const double* __restrict__ Bn,
                                                 RevIn R, double* __restrict__ S, double* __restrict__ Bnb) {
  const size_t f = (size_t)blockIdx.x * kT + threadIdx.x;
  if (f >= G.n2) return;
  flux_vjp_face<DIR, SOLVER>(G, f, W, Bn, R, S, Bnb);
}

// per-cell sum of the stencil contributions, then the cons->prim reverse
// from the tape's primitive state: Qb += (dW/dQ)^T Wb
template <int STAGE>
__global__ __launch_bounds__(kT) void k_gather_prim_vjp(Grid G, const double* __restrict__ W,
                                                        const double* __restrict__ Sx, const double* __restrict__ Sy,
                                                        RevIn R, double* __restrict__ Ub, double* __restrict__ Qb) {
  const size_t c = (size_t)blockIdx.x * kT + threadIdx.x;
  if (c >= G.n2) return;
  const int i = (int)(c % G.n), j = (int)(c / G.n);
  double wb[8], w[8], ub[8];
  for (int k = 0; k < 8; k++) {
    double a = 0.;
    for (int s = 0; s < 4; s++) {
      // this cell is stencil position s of the x-face i + 2 - s and y-face j + 2 - s
      const size_t fx = (size_t)j * G.n + wrap(i + 2 - s, G.n), fy = (size_t)wrap(j + 2 - s, G.n) * G.n + i;
      a += Sx[((size_t)s * 8 + k) * G.n2 + fx];
      a += Sy[((size_t)s * 8 + k) * G.n2 + fy];
    }
    wb[k] = a;
    w[k] = W[k * G.n2 + c];
    ub[k] = 0.;
  }
  Rev<false> plain;
  prim_vjp_w(plain, w, G.g, wb, ub);
  pass_state<STAGE>(G, R, c, ub, Ub, Qb);
}

// Fused face reverse + stencil sum + cons->prim reverse over a tile of
// 16 x 13 cells, one workgroup: the x faces the tile's cells read (13 rows of 19)
// and the y faces (16 rows of 16) are reversed one per lane and leave their stencil
// contributions in LDS, from which, after a barrier, every cell sums its eight and
// adds (dW/dQ)^T Wb to Qb.  Faces next to the tile edge are reversed by both tiles
// that read them; the normal-B adjoint of a face is added only by the tile that
// owns the face.  Deterministic: fixed summation order, no atomics.
// Bound by the solver reverse's arithmetic at the two wavefronts a SIMD its 250
// registers allow (those of the plain quotients, out of line, within them).  Grids of no more tiles than CUs, which would be left half
// idle, take 512 lanes with the y faces beside the x faces (k_stage_vjp_both);
// others 256 lanes, the y faces after the x faces in the same LDS, two workgroups
// a CU (k_stage_vjp).  The reverse of a step, HLLD, as 512 lanes and as 256: 54.5
// and 67.5 us at 208 tiles (200 cells a side), 90.1 and 89.8 at 285, 98.0 and 95.9
// at 456, 230 and 215 at 1280 (512 a side).
constexpr int kVjpFaces = 256, kVjpW = 16, kVjpH = 13;
constexpr int kVjpBothTiles = 256;  // CUs

template <int SOLVER, int STAGE>
__global__ __launch_bounds__(kVjpFaces) void k_stage_vjp(Grid G, const double* __restrict__ W,
                                                  const double* __restrict__ Bx, const double* __restrict__ By, RevIn R,
                                                  double* __restrict__ Bnbx, double* __restrict__ Bnby,
                                                  double* __restrict__ Ub, double* __restrict__ Qb) {
  constexpr int TW = kVjpW, TH = kVjpH, TT = kVjpFaces;
  static_assert(TH * (TW + 3) <= TT && (TH + 3) * TW <= TT, "one face per lane and direction");
  __shared__ double S[8][4][TT];  // [variable][stencil position][face of the tile]
  // x-face sums of the tile's cells, kept in LDS across the y-face reverse
  // rather than in 16 VGPRs
  __shared__ double Sx[8][TW * TH];
  const int tid = threadIdx.x;
  const int i0 = blockIdx.x * TW, j0 = blockIdx.y * TH;
  // this lane's cell
  const int ci = tid % TW, cj = tid / TW;
  const int i = i0 + ci, j = j0 + cj;
  const bool has_cell = tid < TW * TH && i < G.n && j < G.n;
  // ---- x faces: tile row r, face column q -> face i0 - 1 + q
  if (tid < TH * (TW + 3)) {
    const int r = tid / (TW + 3), q = tid % (TW + 3);
    const int fj = j0 + r, fi = wrap_any(i0 - 1 + q, G.n);
    if (fj < G.n) {
      double wlb[8], wrb[8];
      size_t cell[4];
      face_reverse<0, SOLVER>(G, fi, fj, W, Bx, R, &S[0][0][tid], TT, wlb, wrb, cell);
      if (q >= 1 && q <= TW && i0 - 1 + q < G.n) Bnbx[(size_t)fj * G.n + fi] += wlb[5] + wrb[5];
      stencil_reverse<0>(G, W, cell, wlb, wrb, [&](int k, const double* vb) {
        for (int s = 0; s < 4; s++) S[k][s][tid] = vb[s];
      });
    }
  }
  __syncthreads();
  if (has_cell) {
    // this cell is stencil position s of the x face i + 2 - s: tile column ci + 3 - s
    for (int k = 0; k < 8; k++) {
      double a = 0.;
      for (int s = 0; s < 4; s++) a += S[k][s][cj * (TW + 3) + ci + 3 - s];
      Sx[k][tid] = a;
    }
  }
  __syncthreads();
  // ---- y faces: face row r -> face j0 - 1 + r, column q
  if (tid < (TH + 3) * TW) {
    const int r = tid / TW, q = tid % TW;
    const int fj = wrap_any(j0 - 1 + r, G.n), fi = i0 + q;
    if (fi < G.n) {
      double wlb[8], wrb[8];
      size_t cell[4];
      face_reverse<1, SOLVER>(G, fi, fj, W, By, R, &S[0][0][tid], TT, wlb, wrb, cell);
      if (r >= 1 && r <= TH && j0 - 1 + r < G.n) Bnby[(size_t)fj * G.n + fi] += wlb[6] + wrb[6];
      stencil_reverse<1>(G, W, cell, wlb, wrb, [&](int k, const double* vb) {
        for (int s = 0; s < 4; s++) S[k][s][tid] = vb[s];
      });
    }
  }
  __syncthreads();
  if (has_cell) {
    const size_t c = (size_t)j * G.n + i;
    double w[8], ub[8], wb[8];
    for (int k = 0; k < 8; k++) {
      double a = Sx[k][tid];
      for (int s = 0; s < 4; s++) a += S[k][s][(cj + 3 - s) * TW + ci];
      wb[k] = a;
      w[k] = W[k * G.n2 + c];
      ub[k] = 0.;
    }
    Rev<false> plain;
    prim_vjp_w(plain, w, G.g, wb, ub);
    pass_state<STAGE>(G, R, c, ub, Ub, Qb);
  }
}

// the same with the y faces beside the x faces
template <int SOLVER, int STAGE>
__global__ __launch_bounds__(2 * kVjpFaces) void k_stage_vjp_both(
    Grid G, const double* __restrict__ W, const double* __restrict__ Bx, const double* __restrict__ By, RevIn R,
    double* __restrict__ Bnbx, double* __restrict__ Bnby, double* __restrict__ Ub, double* __restrict__ Qb) {
  constexpr int TW = kVjpW, TH = kVjpH, TT = kVjpFaces;
  __shared__ double Sx[8][4][TT], Sy[8][4][TT];  // as k_stage_vjp's S, of the x faces and of the y faces
  const int tid = threadIdx.x, lane = tid % TT;
  const int i0 = blockIdx.x * TW, j0 = blockIdx.y * TH;
  double wlb[8], wrb[8];
  size_t cell[4];
  if (tid < TT) {
    const int r = lane / (TW + 3), q = lane % (TW + 3);
    const int fj = j0 + r, fi = wrap_any(i0 - 1 + q, G.n);
    if (r < TH && fj < G.n) {
      face_reverse<0, SOLVER>(G, fi, fj, W, Bx, R, &Sx[0][0][lane], TT, wlb, wrb, cell);
      if (q >= 1 && q <= TW && i0 - 1 + q < G.n) Bnbx[(size_t)fj * G.n + fi] += wlb[5] + wrb[5];
      stencil_reverse<0>(G, W, cell, wlb, wrb, [&](int k, const double* vb) {
        for (int s = 0; s < 4; s++) Sx[k][s][lane] = vb[s];
      });
    }
  } else {
    const int r = lane / TW, q = lane % TW;
    const int fj = wrap_any(j0 - 1 + r, G.n), fi = i0 + q;
    if (r < TH + 3 && fi < G.n) {
      face_reverse<1, SOLVER>(G, fi, fj, W, By, R, &Sy[0][0][lane], TT, wlb, wrb, cell);
      if (r >= 1 && r <= TH && j0 - 1 + r < G.n) Bnby[(size_t)fj * G.n + fi] += wlb[6] + wrb[6];
      stencil_reverse<1>(G, W, cell, wlb, wrb, [&](int k, const double* vb) {
        for (int s = 0; s < 4; s++) Sy[k][s][lane] = vb[s];
      });
    }
  }
  __syncthreads();
  const int ci = tid % TW, cj = tid / TW, i = i0 + ci, j = j0 + cj;
  if (tid >= TW * TH || i >= G.n || j >= G.n) return;
  const size_t c = (size_t)j * G.n + i;
  double w[8], ub[8], wb[8];
  for (int k = 0; k < 8; k++) {
    double a = 0.;
    for (int s = 0; s < 4; s++) a += Sx[k][s][cj * (TW + 3) + ci + 3 - s];
    for (int s = 0; s < 4; s++) a += Sy[k][s][(cj + 3 - s) * TW + ci];
    wb[k] = a;
    w[k] = W[k * G.n2 + c];
    ub[k] = 0.;
  }
  Rev<false> plain;
  prim_vjp_w(plain, w, G.g, wb, ub);
  pass_state<STAGE>(G, R, c, ub, Ub, Qb);
}

unsigned blocks(size_t n) { return (unsigned)((n + kT - 1) / kT); }

// In-place calls: a kernel, not a copy of the runtime's, as a caller may capture it
__global__ __launch_bounds__(kT) void k_copy(const double* __restrict__ from, double* __restrict__ to, size_t n) {
  const size_t e = (size_t)blockIdx.x * kT + threadIdx.x;
  if (e < n) to[e] = from[e];
}

struct Span {
  const double* p;
  size_t n;
};
bool overlap(std::initializer_list<Span> a, std::initializer_list<Span> b) {
  for (const Span& x : a)
    for (const Span& y : b)
      if ((uintptr_t)x.p < (uintptr_t)(y.p + y.n) && (uintptr_t)y.p < (uintptr_t)(x.p + x.n)) return true;
  return false;
}

}  // namespace

struct amr_adj {
  Grid G;
  int solver = kFluxHLLE;  // kFluxHLLE or kFluxHLLD
  int fused = 1;  // face reverse + gather in one tiled kernel: 1 by the number of tiles, 2 the y faces after the
                  // x faces; 0: per-face kernels and a gather
  // forward scratch
  double *Fx, *Fy, *Us, *Uo, *Bxo, *Byo, *tape;
  // adjoint work
  double *Usb, *Eb, *Bsbx, *Bsby, *Sx, *Sy;
};

namespace {

#define ADJ_CHK(x)                                                                             \
  do {                                                                                         \
    hipError_t e_ = (x);                                                                       \
    if (e_ != hipSuccess) {                                                                    \
      std::fprintf(stderr, "amr2d_mhd adjoint: HIP error %s at %s:%d\n", hipGetErrorString(e_), __FILE__, \
                   __LINE__);                                                                  \
      return AMR_ERR_HIP;                                                                      \
    }                                                                                          \
  } while (0)

template <int SOLVER>
void launch_faces(amr_adj* a, const double* Q, const double* Bx, const double* By, double* W, hipStream_t s) {
  const unsigned n = (unsigned)a->G.n;
  const dim3 grid((n + kFx - 1) / kFx, (n + kFy - 1) / kFy);
  k_fwd_faces<SOLVER><<<grid, kFaceLanes, 0, s>>>(a->G, Q, Bx, By, W, a->Fx, a->Fy);
}

dim3 cell_grid(const Grid& G) { return dim3((unsigned)((G.n + kUx - 1) / kUx), (unsigned)((G.n + kUy - 1) / kUy)); }

// forward stage sequence, writing the step's tape
template <int SOLVER>
int forward_of(amr_adj* a, const double* U, const double* Bx, const double* By, double dt, double* Uo, double* Bxo,
               double* Byo, const Tape& T, hipStream_t s) {
  const Grid& G = a->G;
  const dim3 cells = cell_grid(G);
  launch_faces<SOLVER>(a, U, Bx, By, T.W1, s);
  k_fwd_update<1><<<cells, kUx * kUy, 0, s>>>(G, U, nullptr, a->Fx, a->Fy,
                                              FwdFaces{Bx, By, nullptr, nullptr, T.Bxs, T.Bys, nullptr, nullptr}, dt,
                                              a->Us, T.pre1);
  launch_faces<SOLVER>(a, a->Us, T.Bxs, T.Bys, T.W2, s);
  // in place the faces go to the tape alone, and out of it when all are formed
  const size_t n2 = G.n2;
  const bool in_place = overlap({{Bxo, n2}, {Byo, n2}}, {{U, 8 * n2}, {Bx, n2}, {By, n2}});
  const FwdFaces faces = in_place ? FwdFaces{Bx, By, T.Bxs, T.Bys, T.Bxo, T.Byo, nullptr, nullptr}
                                  : FwdFaces{Bx, By, T.Bxs, T.Bys, Bxo, Byo, T.Bxo, T.Byo};
  k_fwd_update<2><<<cells, kUx * kUy, 0, s>>>(G, U, a->Us, a->Fx, a->Fy, faces, dt, Uo, T.pre2);
  if (in_place) {
    k_copy<<<blocks(n2), kT, 0, s>>>(T.Bxo, Bxo, n2);
    k_copy<<<blocks(n2), kT, 0, s>>>(T.Byo, Byo, n2);
  }
  ADJ_CHK(hipGetLastError());
  return 0;
}

int forward(amr_adj* a, const double* U, const double* Bx, const double* By, double dt, double* Uo, double* Bxo,
            double* Byo, const Tape& T, hipStream_t s) {
  return a->solver == kFluxHLLD ? forward_of<kFluxHLLD>(a, U, Bx, By, dt, Uo, Bxo, Byo, T, s)
                                : forward_of<kFluxHLLE>(a, U, Bx, By, dt, Uo, Bxo, Byo, T, s);
}

// face reverse of one stage: normal-B adjoints into Bnb*, cell adjoints to
// Ub (stage 2) and Qb
template <int SOLVER, int STAGE>
void face_and_gather(amr_adj* a, const double* W, const double* Bx, const double* By, const RevIn& R, double* Bnbx,
                     double* Bnby, double* Ub, double* Qb, hipStream_t s) {
  const Grid& G = a->G;
  if (a->fused) {
    const dim3 grid((unsigned)((G.n + kVjpW - 1) / kVjpW), (unsigned)((G.n + kVjpH - 1) / kVjpH));
    if (a->fused == 1 && grid.x * grid.y <= kVjpBothTiles)
      k_stage_vjp_both<SOLVER, STAGE><<<grid, 2 * kVjpFaces, 0, s>>>(G, W, Bx, By, R, Bnbx, Bnby, Ub, Qb);
    else k_stage_vjp<SOLVER, STAGE><<<grid, kVjpFaces, 0, s>>>(G, W, Bx, By, R, Bnbx, Bnby, Ub, Qb);
  } else {
    const unsigned b1 = blocks(G.n2);
    k_flux_vjp<0, SOLVER><<<b1, kT, 0, s>>>(G, W, Bx, R, a->Sx, Bnbx);
    k_flux_vjp<1, SOLVER><<<b1, kT, 0, s>>>(G, W, By, R, a->Sy, Bnby);
    k_gather_prim_vjp<STAGE><<<b1, kT, 0, s>>>(G, W, a->Sx, a->Sy, R, Ub, Qb);
  }
}

// reverse sweep of one step from its tape and input faces
template <int SOLVER>
int reverse_of(amr_adj* a, const Tape& T, const double* Bx, const double* By, double dt, const double* Uob,
               const double* Bxob, const double* Byob, double* Ub, double* Bxb, double* Byb, hipStream_t s) {
  const Grid& G = a->G;
  const dim3 cells = cell_grid(G);
  k_rev_faces<2><<<cells, kUx * kUy, 0, s>>>(G, Uob, T.Bxo, T.Byo, Bxob, Byob, dt, Bxb, Byb, a->Bsbx, a->Bsby, a->Eb);
  face_and_gather<SOLVER, 2>(a, T.W2, T.Bxs, T.Bys, RevIn{Uob, T.pre2, a->Eb, -0.5 * dt}, a->Bsbx, a->Bsby, Ub,
                             a->Usb, s);
  k_rev_faces<1><<<cells, kUx * kUy, 0, s>>>(G, a->Usb, T.Bxs, T.Bys, a->Bsbx, a->Bsby, dt, Bxb, Byb, nullptr, nullptr,
                                             a->Eb);
  face_and_gather<SOLVER, 1>(a, T.W1, Bx, By, RevIn{a->Usb, T.pre1, a->Eb, -dt}, Bxb, Byb, nullptr, Ub, s);
  ADJ_CHK(hipGetLastError());
  return 0;
}

int reverse(amr_adj* a, const Tape& T, const double* Bx, const double* By, double dt, const double* Uob,
            const double* Bxob, const double* Byob, double* Ub, double* Bxb, double* Byb, hipStream_t s) {
  // in place from a copy of the cotangents, in buffers that only amr_adj_step_vjp's
  // forward uses, before: the kernels read neighbours' while they write their own
  const size_t n2 = a->G.n2;
  if (overlap({{Ub, 8 * n2}, {Bxb, n2}, {Byb, n2}}, {{Uob, 8 * n2}, {Bxob, n2}, {Byob, n2}})) {
    k_copy<<<blocks(8 * n2), kT, 0, s>>>(Uob, a->Uo, 8 * n2);
    k_copy<<<blocks(n2), kT, 0, s>>>(Bxob, a->Bxo, n2);
    k_copy<<<blocks(n2), kT, 0, s>>>(Byob, a->Byo, n2);
    Uob = a->Uo;
    Bxob = a->Bxo;
    Byob = a->Byo;
  }
  return a->solver == kFluxHLLD ? reverse_of<kFluxHLLD>(a, T, Bx, By, dt, Uob, Bxob, Byob, Ub, Bxb, Byb, s)
                                : reverse_of<kFluxHLLE>(a, T, Bx, By, dt, Uob, Bxob, Byob, Ub, Bxb, Byb, s);
}

// ------------------------------------------------- allocation-free step
// Work memory of amr_adj_step_noalloc: the forward's face fluxes,
// stage state and tape (8 + 8 + 8 + kTapePerCell doubles per cell) for
// grids of up to kNoAllocMaxN^2 cells, in one file-scope device array that
// every GPU the library runs on holds until the process ends (25.2 MB).  Host
// code never passes the array's name to a kernel (a host-side stand-in):
// each device's address comes from hipGetSymbolAddress, taken once per
// device on its first call, and only that address is used.
constexpr int kNoAllocMaxN = 256;
constexpr size_t kNoAllocPerCell = 8 + 8 + 8 + kTapePerCell;
static __device__ __align__(256) double scratch[kNoAllocPerCell * kNoAllocMaxN * kNoAllocMaxN];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {nullptr};

// the current device's address of `scratch`
int scratch_address(double** out) {
  int dev = -1;
  ADJ_CHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return AMR_ERR_CONFIG;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    ADJ_CHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return AMR_ERR_HIP;
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

}  // namespace

extern "C" {

int amr_adj_step_noalloc(int n, double dx, double gamma, const char* flux, const double* U, const double* Bx,
                         const double* By, double dt, double* Uo, double* Bxo, double* Byo, void* stream) {
  AMR_TRY
  if (n < 4 || n > kNoAllocMaxN || dx <= 0 || !U || !Bx || !By || !Uo || !Bxo || !Byo) {
    if (n > kNoAllocMaxN)
      std::fprintf(stderr, "amr_adj_step_noalloc: n = %d exceeds the %d x %d cells of its static work memory\n", n,
                   kNoAllocMaxN, kNoAllocMaxN);
    return AMR_ERR_CONFIG;
  }
  int solver = kFluxHLLE;
  if (flux && std::strcmp(flux, "HLLD") == 0) solver = kFluxHLLD;
  else if (flux && std::strcmp(flux, "HLLE") != 0) return AMR_ERR_CONFIG;
  double* w = nullptr;
  if (int e = scratch_address(&w)) return e;
  // a context on the stack whose work buffers are views into the array
  amr_adj a{};
  a.G = Grid{n, dx, gamma, (size_t)n * n};
  a.solver = solver;
  const size_t n2 = a.G.n2;
  a.Fx = w;
  a.Fy = w + 8 * n2;
  a.Us = w + 16 * n2;
  a.tape = w + 24 * n2;
  return forward(&a, U, Bx, By, dt, Uo, Bxo, Byo, tape_at(a.tape, n2), (hipStream_t)stream);
  AMR_CATCH
}

int amr_adj_create(int n, double dx, double gamma, const char* flux, amr_adj** out) {
  AMR_TRY
  if (!out || n < 4 || dx <= 0) return AMR_ERR_CONFIG;
  int solver = kFluxHLLE;
  if (flux && std::strcmp(flux, "HLLD") == 0) solver = kFluxHLLD;
  else if (flux && std::strcmp(flux, "HLLE") != 0) return AMR_ERR_CONFIG;
  amr_adj* a = new amr_adj();
  a->solver = solver;
  a->G = Grid{n, dx, gamma, (size_t)n * n};
  const size_t n2 = a->G.n2;
  double** bufs8[] = {&a->Fx, &a->Fy, &a->Us, &a->Uo, &a->Usb};
  double** bufs1[] = {&a->Bxo, &a->Byo, &a->Eb, &a->Bsbx, &a->Bsby};
  bool ok = true;
  for (auto p : bufs8) ok = ok && hipMalloc((void**)p, 8 * n2 * sizeof(double)) == hipSuccess;
  for (auto p : bufs1) ok = ok && hipMalloc((void**)p, n2 * sizeof(double)) == hipSuccess;
  ok = ok && hipMalloc((void**)&a->tape, kTapePerCell * n2 * sizeof(double)) == hipSuccess;
  ok = ok && hipMalloc((void**)&a->Sx, 32 * n2 * sizeof(double)) == hipSuccess;
  ok = ok && hipMalloc((void**)&a->Sy, 32 * n2 * sizeof(double)) == hipSuccess;
  if (!ok) {
    amr_adj_destroy(a);
    return AMR_ERR_HIP;
  }
  *out = a;
  return AMR_OK;
  AMR_CATCH
}

int amr_adj_destroy(amr_adj* a) {
  AMR_TRY
  if (!a) return AMR_OK;
  double* all[] = {a->Fx,   a->Fy,   a->Us, a->Uo, a->Bxo, a->Byo, a->tape, a->Usb, a->Eb,
                   a->Bsbx, a->Bsby, a->Sx, a->Sy};
  for (double* p : all)
    if (p) hipFree(p);
  delete a;
  return AMR_OK;
  AMR_CATCH
}

int64_t amr_adj_tape_doubles(const amr_adj* a) { return a ? (int64_t)(kTapePerCell * a->G.n2) : 0; }

int amr_adj_step_tape(amr_adj* a, const double* U, const double* Bx, const double* By, double dt, double* Uo,
                      double* Bxo, double* Byo, double* tape, void* stream) {
  AMR_TRY
  if (!a || !U || !Bx || !By || !Uo || !Bxo || !Byo) return AMR_ERR_CONFIG;
  return forward(a, U, Bx, By, dt, Uo, Bxo, Byo, tape_at(tape ? tape : a->tape, a->G.n2), (hipStream_t)stream);
  AMR_CATCH
}

int amr_adj_step(amr_adj* a, const double* U, const double* Bx, const double* By, double dt, double* Uo, double* Bxo,
                 double* Byo, void* stream) {
  AMR_TRY
  return amr_adj_step_tape(a, U, Bx, By, dt, Uo, Bxo, Byo, nullptr, stream);
  AMR_CATCH
}

int amr_adj_vjp_tape(amr_adj* a, const double* tape, const double* Bx, const double* By, double dt,
                     const double* Uob, const double* Bxob, const double* Byob, double* Ub, double* Bxb, double* Byb,
                     void* stream) {
  AMR_TRY
  if (!a || !tape || !Bx || !By || !Uob || !Bxob || !Byob || !Ub || !Bxb || !Byb) return AMR_ERR_CONFIG;
  return reverse(a, tape_at(const_cast<double*>(tape), a->G.n2), Bx, By, dt, Uob, Bxob, Byob, Ub, Bxb, Byb,
                 (hipStream_t)stream);
  AMR_CATCH
}

int amr_adj_step_vjp(amr_adj* a, const double* U, const double* Bx, const double* By, double dt, const double* Uob,
                     const double* Bxob, const double* Byob, double* Ub, double* Bxb, double* Byb, void* stream) {
  AMR_TRY
  if (!a || !U || !Bx || !By || !Uob || !Bxob || !Byob || !Ub || !Bxb || !Byb) return AMR_ERR_CONFIG;
  hipStream_t s = (hipStream_t)stream;
  const Tape T = tape_at(a->tape, a->G.n2);
  // recompute the step into the context's own tape
  if (int e = forward(a, U, Bx, By, dt, a->Uo, a->Bxo, a->Byo, T, s)) return e;
  return reverse(a, T, Bx, By, dt, Uob, Bxob, Byob, Ub, Bxb, Byb, s);
  AMR_CATCH
}

// test hook: 1 = fused tiled face reverse, its form by the number of tiles
// (default), 2 = the y faces after the x faces, 0 = per-face kernels and a
// separate gather (same derivative, different summation order)
int amr_debug_adj_set_fused(amr_adj* a, int mode) {
  AMR_TRY
  if (!a || mode < 0 || mode > 2) return AMR_ERR_CONFIG;
  a->fused = mode;
  return AMR_OK;
  AMR_CATCH
}

// host entry points of the pointwise reverse pieces (CPU tests)
void amr_debug_hlle_vjp(const double* wL, const double* wR, double gamma, const double* fb, double* wLb, double* wRb) {
  for (int k = 0; k < 8; k++) wLb[k] = wRb[k] = 0.;
  Rev<false> A;
  hlle_vjp(A, wL, wR, gamma, fb, wLb, wRb);
}

void amr_debug_hlle(const double* wL, const double* wR, double gamma, double* f) { flux_hlle(wL, wR, gamma, f); }

// HLLD reverse on the host; f receives the flux its own forward computed
void amr_debug_hlld_vjp(const double* wL, const double* wR, double gamma, const double* fb, double* wLb, double* wRb,
                        double* f) {
  for (int k = 0; k < 8; k++) wLb[k] = wRb[k] = 0.;
  Rev<false> A;
  hlld_vjp(A, wL, wR, gamma, fb, wLb, wRb, f);
}

void amr_debug_hlld(const double* wL, const double* wR, double gamma, double* f) {
  for (int k = 0; k < 8; k++) f[k] = 0.;
  flux_hlld(wL, wR, gamma, f);
}

// forward values of the reverse's own forward pieces next to those of the
// engine's: out[0..7] = side_fwd (cf, e, H) of both sides and roe_fwd (lmin,
// lmax); ref[0..7] = the same from side_state / roe_bounds
void amr_debug_side_roe(const double* wL, const double* wR, double gamma, double* out, double* ref) {
  FastT fL, fR;
  double eL, HL, eR, HR, lmin, lmax;
  Rev<false> A;
  side_fwd(A, wL, gamma, fL, eL, HL);
  side_fwd(A, wR, gamma, fR, eR, HR);
  RoeT rt;
  roe_fwd(A, wL, wR, gamma, HL, HR, rt, lmin, lmax);
  const double o[] = {fL.cf, eL, HL, fR.cf, eR, HR, lmin, lmax};
  Side L, R;
  side_state(wL, gamma, L);
  side_state(wR, gamma, R);
  double u, rlmin, rlmax;
  roe_bounds(wL, wR, gamma, L.H, R.H, u, rlmin, rlmax);
  const double r[] = {L.cf, L.e, L.H, R.cf, R.e, R.H, rlmin, rlmax};
  for (int k = 0; k < 8; k++) {
    out[k] = o[k];
    ref[k] = r[k];
  }
}

void amr_debug_recon_minmod_vjp(const double* v, double wlb, double wrb, double* vb, double* wlr) {
  for (int s = 0; s < 4; s++) vb[s] = 0.;
  Rev<false> A;
  recon_minmod_vjp(A, v, wlb, wrb, vb);
  recon_minmod(A, v, wlr[0], wlr[1]);
}

void amr_debug_prim_vjp(const double* u, double gamma, const double* wb, double* ub, double* w) {
  for (int k = 0; k < 8; k++) ub[k] = 0.;
  Rev<false> A;
  prim_vjp(A, u, gamma, wb, ub);
  prim_of(A, u, gamma, w);
}

}  // extern "C"
