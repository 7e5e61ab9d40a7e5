// The persistent step kernel (one cooperative launch per step).
#pragma once
#include "phases.hpp"
#include "stage.hpp"

namespace amr {

namespace {

// ----------------------------------------------------- persistent step kernel
// Grid-wide barrier of a co-resident grid of nwg workgroups.  Lane 0 of each
// workgroup publishes the workgroup's writes (agent-scope release), arrives,
// and waits for the generation to move; the last to arrive resets the count
// and moves it.  The count is back at zero after every barrier, so the state
// serves every launch without a reset.  A wait is bounded by the device clock
// (100 MHz): past kBarrierTicks it sets *fail, and a set *fail makes every
// later wait return at once, so every workgroup reaches the end of the
// launch (the host then reports the failure and stops using this kernel).
constexpr unsigned long long kBarrierTicks = 200000000ull;  // 2 s

__device__ inline void grid_barrier(GridSync* b, unsigned nwg, int32_t* fail) {
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned g = __hip_atomic_load(&b->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    const unsigned old = __hip_atomic_fetch_add(&b->arrive, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    if (old == nwg - 1) {
      __hip_atomic_store(&b->arrive, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_add(&b->gen, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      const unsigned long long t0 = wall_clock64();
      while (__hip_atomic_load(&b->gen, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) == g) {
        if (__hip_atomic_load(fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
        if (wall_clock64() - t0 > kBarrierTicks) {
          __hip_atomic_store(fail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
}

template <int NT, int NG, int TPB>
struct StepLds {
  using S = StageLds<NT, NG, true>;
  static constexpr int kCfl = 8 * NT * NT + 2 * TPB;
  static constexpr int kDoubles = S::kDoubles > kCfl ? S::kDoubles : kCfl;
};

template <int NT, int NG, int TPB, int SPEC>
__global__ __launch_bounds__(TPB) void step_kernel(StepArgs A) {
  using S = StageLds<NT, NG, true>;
  constexpr int N2 = NT * NT;
  __shared__ double lds[StepLds<NT, NG, TPB>::kDoubles];
  __shared__ int sFlags;
  const int tid = threadIdx.x;
  const unsigned nwg = gridDim.x;
  const FillProgram prog{A.ops, A.gen, A.cprefix, A.ninst};
  if (A.stamps && blockIdx.x == 0 && tid == 0) A.stamps[0] = wall_clock64();
  for (int p = 0; p < A.nphases; p++) {
    const StepPhase ph = A.phase[p];
    if (ph.kind == kPhaseFill) {
      if (p == 0)  // the step's parameters (no fill op reads them)
        for (int i = blockIdx.x * TPB + tid; i < A.copy_words; i += nwg * TPB) A.copy_dst[i] = A.copy_src[i];
      // TPB / kFillChunk chunks side by side per workgroup
      constexpr int kPer = TPB / kFillChunk;
      const int lane = tid % kFillChunk, sub = tid / kFillChunk;
      for (int w0 = blockIdx.x * kPer; w0 < A.nchunks; w0 += nwg * kPer) {
        const int w = w0 + sub;
        FillOp op{};
        op.op = kFillNop;
        int q = 0;
        if (w < A.nchunks) {
          q = find_segment(prog, w);
          op = prog.ops[q][(w - prog.cprefix[q]) * kFillChunk + lane];
        }
        const bool live = op.op != kFillNop;
        const FillGen* gen = w < A.nchunks ? prog.gen[q] : nullptr;
        for (int f = 0; f < ph.nf; f++) {
          const int fld = ph.field[f];
          double* base = A.F.f[fld];
          if (fld == kBi || fld == kBis) fill_field<2>(FillCtx{base, 2, ph.fkind[f], N2, NT, gen}, base, op, live);
          else if (fld == kEMF) fill_field<1>(FillCtx{base, 1, ph.fkind[f], N2, NT, gen}, base, op, live);
          else fill_field<8>(FillCtx{base, 8, ph.fkind[f], N2, NT, gen}, base, op, live);
        }
      }
    } else if (ph.kind == kPhaseStage) {
      for (int l = blockIdx.x; l < A.nleaf; l += nwg) {
        __syncthreads();  // the previous leaf is done with the LDS
        stage_block<NT, NG, TPB, true, SPEC>(A.F, A.leaves[l], A.ip, ph.step, A.err, lds, lds + 8 * N2,
                                             lds + 8 * N2 + S::NFL, &sFlags);
      }
    } else if (ph.kind == kPhaseCfl) {
      for (int l = blockIdx.x; l < A.nleaf; l += nwg) {
        __syncthreads();
        cfl_block<NT, NG, TPB>(A.F, nullptr, A.leaves[l], l, A.ip, A.lam_grad, A.err, lds, lds + 8 * N2);
      }
    } else {
      // CT kernels: one lane per cell of every leaf
      const int total = A.nleaf * N2;
      for (int e = blockIdx.x * TPB + tid; e < total; e += nwg * TPB) {
        const LeafItem L = A.leaves[e / N2];
        const int c = e % N2;
        if (ph.kind == kPhaseEmf) emf_cell<NT>(A.F, L, A.ip, ph.step == A.ip[L.inst].rk, A.err, ph.step, c);
        else if (ph.kind == kPhaseBupdate) bupdate_cell<NT>(A.F, L, A.ip, ph.step, A.ip[L.inst].rk, c);
        else bsync_cell<NT>(A.F, L, ph.step, c);
      }
    }
    if (p + 1 < A.nphases) grid_barrier(A.sync, nwg, A.fail);
    if (A.stamps && blockIdx.x == 0 && tid == 0) A.stamps[p + 1] = wall_clock64();
  }
}

}  // namespace

}  // namespace amr
