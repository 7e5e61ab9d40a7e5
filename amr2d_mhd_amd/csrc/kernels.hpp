// Launch interface of the AMR2D-MHD device kernels (kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "amr_types.hpp"

namespace amr {

struct FieldPtrs {
  double* f[kNumFields];
};

// up to four fields filled by one fill launch
struct FillSet {
  double* base[4];
  int32_t nv[4];
  int32_t kind[4];
  int32_t n;
  // optional: copy_words 8-byte words copy_src -> copy_dst done by the same
  // launch (the step's parameter upload from pinned host memory, so that it
  // costs no copy dispatch of its own); no fill op reads copy_dst
  int32_t copy_words;
  const double* copy_src;
  double* copy_dst;
};

// refine (4 sons from a parent) or coarsen (parent from 4 sons) operation
struct RegridOp {
  int32_t parent_gs;
  int32_t son_gs[4];
  int32_t inst;
  int32_t nb;      // parent (refine) or dad (coarsen) block id
  int32_t son_nb;  // first son's block id; the four sons are son_nb .. son_nb + 3
  int32_t seq;     // position among the instance's ops of this regrid, in the
                   // reference's order (all refinements, then all coarsenings)
};

bool tile_supported(int NT, int ng);

// Stage kernels (identical results), and the variant numbers of the interface
// that select them:
//   wide    768 lanes a leaf block, face fluxes in LDS (1, 2, 5): one pass over
//           the block's 578 faces, the shortest time of a single block
//   narrow  256 lanes, fluxes read back from ff/gg (0, 3, 4): 25.6 KB of LDS and
//           168 VGPRs, three blocks on a CU at a time whose load, face and
//           update phases overlap
//   strips  each block split into 4 row strips of 192 lanes (6, 7): four times
//           the workgroups where the blocks alone leave CUs idle
// Of the narrow and strip kernels the HLLD and HLLC ones with a MUSCL limiter hold
// their faces in the 168 VGPRs of three wavefronts a SIMD; the generic ones and
// WENO5's spill 103 to 119 more (416 to 456 B a lane; the generic narrow one for
// 12 x 12 tiles does not).  The wide ones take 137 to 146 and spill none.
// stage_rule chooses by the number of leaf blocks of the launch.  Microseconds a
// launch, rotor HLLD + MC (strips, wide, narrow): 52 blocks 10.9, 15.2, 19.3;
// 136: 16.2, 16.0, 20.5; 196: 17.2, 16.5, 20.4; 340: 24.4, 25.7, 27.4; 436: 28.5,
// 27.1, 28.3; 757: 41.2, 41.2, 34.3; 2352: 110, 117, 90.  HLLC + VanLeer at 100
// blocks 15.1, 17.0, 23.6, HLLE at 340 25.7, 27.1, 28.4, HLLD + WENO5 at 112 23.5,
// 24.4, 43.0 and at 925 70.9, 69.8, 60.9.  (Between the lines strips and wide lie
// within 6% of each other, either ahead as the blocks fill the 256 CUs.)  One rule for
// all tiles, though blocks of 8 x 8 cells leave 606 of the wide kernel's lanes without
// a face and do better with the narrow one from 160 blocks: 160 13.8, 11.1, 11.1; 340
// 18.1, 18.4, 15.3; 664 20.3, 25.4, 17.4; 1918 38.7, 54.9, 31.2.
enum { kStageWide, kStageNarrow, kStageStrips };
constexpr int stage_kernel_of(int variant) {
  return variant >= 6 ? kStageStrips : variant == 0 || variant == 3 || variant == 4 ? kStageNarrow : kStageWide;
}
constexpr int kVariantWide = 2, kVariantNarrow = 3, kVariantStrips = 7;
inline int stage_rule(int nleaf) { return nleaf < 128 ? kVariantStrips : nleaf < 512 ? kVariantWide : kVariantNarrow; }
constexpr int kStageVariants = 8;
// stage-kernel specialisations: generic (solver and limiter read per leaf), or
// HLLD with a MUSCL-family limiter, or HLLD with WENO5 (24x24 tiles, the only
// ones with the ghost depth WENO5 needs), fixed at compile time
// or HLLC with a MUSCL-family limiter.  The specialised kernels are 2-7% faster
// than the generic one with the same settings (rotor at 340 blocks: 25.7 and
// 26.7 us; WENO5 narrow at 925: 60.9 and 63.4).
enum { kStageGeneric = 0, kStageHLLDMuscl = 1, kStageHLLDWeno5 = 2, kStageHLLCMuscl = 3, kStageSpecs = 4 };
// Work-list counts on the device (counts[kCountLeaves], counts[kCountChunks]):
// a launch given `counts` may have a larger grid than its work (a captured
// step replayed over changing trees) and its surplus workgroups exit; with
// counts = null the grid is the work.
enum { kCountLeaves = 0, kCountChunks = 1 };
// one specialisation for one tile size (stage.hip, step.hip): 20 and 12 cells
// a side for every specialisation but HLLD + WENO5, 24 for all
template <int SPEC, int TILE>
void launch_stage_tile(int variant, const FieldPtrs& F, const LeafItem* leaves, int nleaf, const InstParams* ip,
                       int step, DevError* err, hipStream_t s, hipEvent_t ev_start, hipEvent_t ev_stop,
                       const int32_t* counts);
template <int SPEC, int TILE>
const void* step_kernel_tile(int lanes_idx);
void launch_stage(int NT, int ng, int variant, int spec, const FieldPtrs& F, const LeafItem* leaves, int nleaf,
                  const InstParams* ip, int step, DevError* err, hipStream_t s, hipEvent_t ev_start = nullptr,
                  hipEvent_t ev_stop = nullptr, const int32_t* counts = nullptr);
// corner EMF of RK stage `step` of an `rk`-stage scheme (CTtype per instance)
void launch_emf(int NT, const FieldPtrs& F, const LeafItem* leaves, int nleaf, const InstParams* ip, int step,
                int rk, DevError* err, hipStream_t s, const int32_t* counts = nullptr);
// face-B update of RK stage `step` of an `rk`-stage scheme; cell sync into U
// (last stage) or Us
void launch_bupdate(int NT, const FieldPtrs& F, const LeafItem* leaves, int nleaf, const InstParams* ip, int step,
                    int rk, hipStream_t s, const int32_t* counts = nullptr);
void launch_bsync(int NT, const FieldPtrs& F, const LeafItem* leaves, int nleaf, int last, hipStream_t s,
                  const int32_t* counts = nullptr);
// ghost fill of up to four fields through a program made of per-instance
// segments of whole kFillChunk-op chunks (device pointer tables
// inst_ops/inst_gen, cprefix[ninst+1] of chunk counts), one workgroup per chunk
// The fill programs by destination (amr_types.hpp) and the scratch fields of the
// fused CT launches; version: the entries that count
struct RingTable {
  uint64_t* entries = nullptr;  // [slot][ring_cells]
  double* emf = nullptr;        // [slot][N2]
  double* old = nullptr;        // [slot][2][N2]
  double* rdx = nullptr;        // [slot]
  uint32_t version = 0;
};
// enters the programs of the running instances into the table
void launch_ring_table(int NT, int ng, const FillOp* const* inst_ops, const int32_t* cprefix, int ninst, int nchunks,
                       const RingTable& ring, hipStream_t s);
// One instance whose fill program is compiled on the device (fillprog.hip): its
// tree, slots and leaves (rank: a block's place in the leaf list), the program
// (`main` ops, one per ring element of a leaf in order, padded to whole chunks,
// then up to cap_tail of the linked groups of up to max_group <= kFillChunk ops),
// scratch of `main` entries each (edges: cap_edges pairs) and the counters.
enum { kPullKinds = 0, kPullGen = 3, kPullLinked = 4, kPullEdges = 5, kPullFlags = 6, kPullTail = 7,
       kPullCount = 8, kPullNext = 20, kPullMeta = 32 };
// flags: a restriction of a restriction, out of space, a group larger than
// max_group (the host compiles instead); an op that reads its own destination
enum { kPullNested = 1, kPullSpace = 2, kPullGroup = 4, kPullSelf = 8 };
struct PullInst {
  const int32_t* lp;
  const uint8_t* leafs;
  const int32_t *gs, *leaf, *rank;
  FillOp* ops;
  FillGen* gen;
  int32_t *uf, *size, *linked, *root, *edges, *meta;
  int32_t nleaf, main, cap_tail, cap_gen, cap_edges, max_group;
};
// max_main, max_ops: the largest main and main + cap_tail of the n instances
void launch_pull(int NT, int ng, const PullInst* insts, int n, int max_main, int max_ops, hipStream_t s);

// a fill program's device tables (launch_fill)
struct FillTables {
  const FillOp* const* ops;
  const FillGen* const* gen;
  const int32_t* cprefix;
  int ninst, nchunks;
};
// the ghost fills of the fluxes and, in the first stage, of Bi, then
// CT2D.cpp:11-124 with its own, for trees whose programs (all: whole, tail: their
// linked tails) touch leaves only: two launches.  Bi comes filled from the step's
// first fill; of the fluxes of the stages before the last only what a later
// kernel reads is filled in memory (ct_fill_fluxes).
void launch_ct(int NT, int ng, const FieldPtrs& F, const LeafItem* leaves, int nleaf, const InstParams* ip, int step,
               int rk, const FillTables& all, const FillTables& tail, const RingTable& ring, DevError* err,
               hipStream_t s);
void launch_fill(int NT, const FillOp* const* inst_ops, const FillGen* const* inst_gen, const int32_t* cprefix,
                 int ninst, int nchunks, const FillSet& set, hipStream_t s, const int32_t* counts = nullptr);
// per-leaf CFL bound min(dx,dy)/lambda and refinement indicator, as pairs
// lam_grad[2 leaf], lam_grad[2 leaf + 1]; when W is non-null it supplies the
// primitives (initial regrid) instead of U.
void launch_cfl_criteria(int NT, int ng, const FieldPtrs& F, const double* W, const LeafItem* leaves, int nleaf,
                         const InstParams* ip, double* lam_grad, DevError* err, hipStream_t s,
                         const int32_t* counts = nullptr);
void launch_refine(int NT, int ng, const FieldPtrs& F, const RegridOp* ops, int nops, const InstParams* ip,
                   DevError* err, hipStream_t s);

// device copy of the quadtrees of a context: lp rows [block][8] and per-block
// flags; instance blocks from RegridInst::off on
struct DeviceTree {
  int32_t* lp;
  uint8_t* leafs;
  uint8_t* iref;
  uint8_t* icoarse;
  uint8_t* mark;
};
// regrid decision and tree surgery of every instance (regrid.hip), one
// workgroup per instance, from the per-leaf CFL bounds and indicators
void launch_regrid(const RegridInst* ri, int ninst, const LeafItem* leaves, const double* lam_grad,
                   const DeviceTree& tree, RegridOut* out, int32_t* oplog, hipStream_t s);
void launch_coarsen(int NT, int ng, const FieldPtrs& F, const RegridOp* ops, int nops, const int32_t* cmapU,
                    const int32_t* cmapB, const InstParams* ip, DevError* err, hipStream_t s);

// ---------------------------------------------------- persistent step kernel
// One launch runs the device work of a whole step (main.cpp:128-230): its
// phases -- ghost fills, RK stages, the CT kernels, CFL/criteria -- run in
// order over the device work lists, separated by grid-wide barriers, in a
// grid of workgroups that are all resident at once (cooperative launch).
enum { kPhaseFill = 0, kPhaseStage, kPhaseEmf, kPhaseBupdate, kPhaseBsync, kPhaseCfl };
struct StepPhase {
  int8_t kind;
  int8_t step;      // stage / face update: RK stage; cell sync: 1 = last stage
  int8_t nf;        // fill: number of fields
  int8_t pad;
  int8_t field[4];  // fill: slot fields and their combine kinds
  int8_t fkind[4];
};
constexpr int kMaxPhases = 32;

// grid barrier state: arrival count and generation in separate 128-byte
// lines; `fail` is set when a wait exceeds its bound (then every later wait
// returns at once, so the launch still ends)
struct GridSync {
  unsigned int arrive;
  unsigned int pad0[31];
  unsigned int gen;
  unsigned int pad1[31];
};

struct StepArgs {
  FieldPtrs F;
  const LeafItem* leaves;
  int nleaf;
  int nchunks;
  const FillOp* const* ops;  // fill program tables (see launch_fill)
  const FillGen* const* gen;
  const int32_t* cprefix;
  int ninst;
  int copy_words;            // parameter upload done by the first phase
  const double* copy_src;
  double* copy_dst;
  const InstParams* ip;
  double* lam_grad;
  DevError* err;
  GridSync* sync;
  int32_t* fail;
  unsigned long long* stamps;  // when non-null: device clock at the start and after every phase
  int nphases;
  StepPhase phase[kMaxPhases];
};

// lanes per workgroup of the step kernel
constexpr int kStepLanes[2] = {256, 512};
// largest co-resident grid of the step kernel for the tile, specialisation and
// lane count (0: it cannot run here)
int step_kernel_grid(int NT, int ng, int spec, int lanes_idx);
// cooperative launch of the step kernel; events (optional) bracket it on s
int launch_step(int NT, int ng, int spec, int lanes_idx, int grid, const StepArgs& A, hipStream_t s,
                hipEvent_t ev_start = nullptr, hipEvent_t ev_stop = nullptr);

// pointwise / tile-level parity entry points
void launch_riemann_batch(int solver, int dir, double gamma, int n, const double* wL, const double* wR, double* flux,
                          int32_t* status, hipStream_t s);
// fill: entries outside the reference's computed range are written as zeros
void launch_recon_batch(int NT, int ng, int lim, double dx, int nt, const double* W, double* out, bool fill,
                        hipStream_t s);

}  // namespace amr
