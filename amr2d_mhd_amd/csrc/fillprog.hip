// The fill program of a tree compiled on the device (fill_pull.hpp): one lane a
// ring element finds its op, then the ops that read elements other ops write are
// grouped and laid out behind the rest.
//
// At every change of the tree the card waits for the program.  The sequential
// compile on the host (16 threads) takes 139 us for 196 leaves of 20x20 and 930 for
// 900 of 24x24, and several contexts at once share the threads; the launches here
// with their upload and the counters' download take 57 and 146.  pull_kernel, 14
// and 40 of them, is bound by chains of dependent loads of neighbour rows (a
// look-up is one to three strips); the others by launch and latency, each a pass
// that has to end before the next begins (as one workgroup of 1024 lanes the
// passes after pull_kernel took 490 us for the 900 leaves, and with an addition to
// a counter a lane instead of a workgroup pull_kernel took 4200).
#include <hip/hip_runtime.h>

#include "amr_types.hpp"
#include "device.hpp"
#include "fill_pull.hpp"
#include "kernels.hpp"

namespace amr {

namespace {

constexpr int kClasses = 9;  // group sizes 1, 2, 4 .. kFillChunk
static_assert(1 << (kClasses - 1) == kFillChunk, "a group fits a chunk");
static_assert(kPullNext + kClasses <= kPullMeta, "counters");

__device__ __forceinline__ int load_agent(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// place for each lane's n items in a list with one addition to its counter a
// workgroup (every lane calls this)
__device__ inline int wg_append(int n, int* counter) {
  __shared__ int sTotal, sBase;
  if (threadIdx.x == 0) sTotal = 0;
  __syncthreads();
  const int at = n ? atomicAdd(&sTotal, n) : 0;
  __syncthreads();
  if (threadIdx.x == 0 && sTotal) sBase = atomicAdd(counter, sTotal);
  __syncthreads();
  const int base = sTotal ? sBase : 0;
  __syncthreads();
  return base + at;
}

// union-find entries empty, padding everywhere past the leaves' ops, counters zero
__global__ __launch_bounds__(kThreads) void pull_init_kernel(const PullInst* __restrict__ insts) {
  const PullInst P = insts[blockIdx.y];
  const FillOp nop{0, 0, kFillNop, 0, 0, 0};
  const int e = blockIdx.x * kThreads + threadIdx.x;
  if (e < P.main + P.cap_tail) P.ops[e] = nop;
  if (e < P.main) {
    P.uf[e] = -1;
    P.size[e] = 0;
  }
  if (e < kPullMeta) P.meta[e] = 0;
}

// the op of each ring element, and the pairs of an op and another that writes
// one of its operands
template <int NT, int NG>
__global__ __launch_bounds__(kThreads) void pull_kernel(const PullInst* __restrict__ insts) {
  constexpr int R = ring_cells(NT, NG), W = NT - 2 * NG;
  const PullInst P = insts[blockIdx.y];
  if ((int)blockIdx.x * kThreads >= P.nleaf * R) return;
  const int e = blockIdx.x * kThreads + threadIdx.x;
  const PullTree T{P.lp, P.leafs};
  PullOp o;
  o.op = kFillNop;
  o.nref = 0;
  o.nested = false;
  int i = 0, j = 0, slot = 0;
  if (e < P.nleaf * R) {
    const int b = P.leaf[e / R];
    int r = e % R;  // ring_index backwards
    if (r < NG * NT) {
      j = r / NT;
      i = r % NT;
    } else if ((r -= NG * NT) < W * 2 * NG) {
      j = NG + r / (2 * NG);
      i = r % (2 * NG);
      i = i < NG ? i : i + W;
    } else {
      r -= W * 2 * NG;
      j = NT - NG + r / NT;
      i = r % NT;
    }
    slot = P.gs[b];
    o = pull_op(T, NT, NG, b, i, j);
  }
  int flags = o.nested ? kPullNested : 0;
  const int gen = wg_append(o.op == kFillGeneral, &P.meta[kPullGen]);
  int w[4], n = 0;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    w[q] = -1;
    if (q >= o.nref || !pull_filled(T, NT, NG, o.nb[q], o.i[q], o.j[q])) continue;
    const int rank = P.rank[o.nb[q]], p = rank * R + ring_index(NT, NG, o.i[q], o.j[q]);
    if (rank < 0) {  // no leaf: not a tree of pull_form
      flags |= kPullSpace;
    } else if (p == e) {
      flags |= kPullSelf;
    } else {
      w[q] = p;
      n++;
    }
  }
  int k = wg_append(n, &P.meta[kPullEdges]);
  if (o.op != kFillNop) {
    FillOp op{slot, (uint16_t)(j * NT + i), (int16_t)o.op, P.gs[o.nb[0]], (uint16_t)(o.j[0] * NT + o.i[0]), 0};
    if (o.op == kFillGeneral) {
      op.src_cell = 0;
      op.src = gen;
      if (gen < P.cap_gen) {
#pragma unroll
        for (int q = 0; q < 4; q++) P.gen[gen].ref[q] = src_ref(P.gs[o.nb[q]], o.j[q] * NT + o.i[q]);
      } else {
        flags |= kPullSpace;
        op.op = kFillNop;
      }
    }
    P.ops[e] = op;
  }
  if (n) P.uf[e] = e;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    if (w[q] < 0) continue;
    P.uf[w[q]] = w[q];
    if (k < P.cap_edges) {
      P.edges[2 * k] = e;
      P.edges[2 * k + 1] = w[q];
      k++;
    } else {
      flags |= kPullSpace;
    }
  }
  if (flags) atomicOr(&P.meta[kPullFlags], flags);
#pragma unroll
  for (int t = 0; t < 3; t++) wg_append(o.op == t, &P.meta[kPullKinds + t]);
}

// a root is hung under a smaller one, so the parents decrease along a path
__device__ inline int find_root(const int* uf, int x) {
  for (;;) {
    const int p = load_agent(uf + x);
    if (p == x) return x;
    x = p;
  }
}

// the linked ops' list and their groups: connected components of the pairs
__global__ __launch_bounds__(kThreads) void pull_link_kernel(const PullInst* __restrict__ insts) {
  const PullInst P = insts[blockIdx.y];
  if (P.meta[kPullFlags] & ~kPullSelf) return;
  const int e = blockIdx.x * kThreads + threadIdx.x;
  if ((int)blockIdx.x * kThreads < P.main) {
    const bool in = e < P.main && load_agent(P.uf + e) != -1;
    const int at = wg_append(in, &P.meta[kPullLinked]);
    if (in) P.linked[at] = e;
  }
  const int nedges = P.meta[kPullEdges];
  for (int k = e; k < nedges; k += gridDim.x * kThreads) {
    int a = P.edges[2 * k], b = P.edges[2 * k + 1];
    for (;;) {
      a = find_root(P.uf, a);
      b = find_root(P.uf, b);
      if (a == b) break;
      if (a < b) {
        const int t = a;
        a = b;
        b = t;
      }
      if (atomicCAS(P.uf + a, a, b) == a) break;
    }
  }
}

__global__ __launch_bounds__(kThreads) void pull_size_kernel(const PullInst* __restrict__ insts) {
  const PullInst P = insts[blockIdx.y];
  if (P.meta[kPullFlags] & ~kPullSelf) return;
  const int k = blockIdx.x * kThreads + threadIdx.x;
  if (k >= P.meta[kPullLinked]) return;
  const int r = find_root(P.uf, P.linked[k]);
  P.root[k] = r;
  atomicAdd(P.size + r, 1);
}

__device__ inline int size_class(int n) { return n <= 1 ? 0 : 32 - __clz(n - 1); }

// how many groups take room for each power of two.  (Other workgroups may set
// kPullGroup meanwhile: a check of it could part a workgroup before its barriers.
// The kernels after this one make it, or go by the flags of the ones before.)
__global__ __launch_bounds__(kThreads) void pull_classes_kernel(const PullInst* __restrict__ insts) {
  const PullInst P = insts[blockIdx.y];
  if (P.meta[kPullFlags] & ~(kPullSelf | kPullGroup)) return;
  __shared__ int sCount[kClasses];
  if (threadIdx.x < kClasses) sCount[threadIdx.x] = 0;
  __syncthreads();
  const int k = blockIdx.x * kThreads + threadIdx.x;
  if (k < P.meta[kPullLinked] && P.root[k] == P.linked[k]) {
    const int n = P.size[P.linked[k]];
    if (n > P.max_group) atomicOr(&P.meta[kPullFlags], kPullGroup);
    else atomicAdd(&sCount[size_class(n)], 1);
  }
  __syncthreads();
  if (threadIdx.x < kClasses && sCount[threadIdx.x]) atomicAdd(&P.meta[kPullCount + threadIdx.x], sCount[threadIdx.x]);
}

// each group's place behind the unlinked ops, inside one chunk: larger room first,
// so that none straddles two
__global__ __launch_bounds__(kThreads) void pull_place_kernel(const PullInst* __restrict__ insts) {
  const PullInst P = insts[blockIdx.y];
  __shared__ int sBase[kClasses], sCount[kClasses], sAt[kClasses], sTail;
  if (P.meta[kPullFlags] & ~(kPullSelf | kPullSpace)) return;
  if (threadIdx.x == 0) {
    int at = 0;
    for (int c = kClasses - 1; c >= 0; c--) {
      sBase[c] = at;
      at += P.meta[kPullCount + c] << c;
    }
    sTail = (at + kFillChunk - 1) / kFillChunk * kFillChunk;
  }
  if (threadIdx.x < kClasses) sCount[threadIdx.x] = 0;
  __syncthreads();
  if (blockIdx.x == 0 && threadIdx.x == 0) P.meta[kPullTail] = sTail;
  if (sTail > P.cap_tail) {
    if (threadIdx.x == 0) atomicOr(&P.meta[kPullFlags], kPullSpace);
    return;
  }
  const int k = blockIdx.x * kThreads + threadIdx.x;
  const bool is_root = k < P.meta[kPullLinked] && P.root[k] == P.linked[k];
  int c = 0, at = 0;
  if (is_root) {
    c = size_class(P.size[P.linked[k]]);
    at = atomicAdd(&sCount[c], 1);
  }
  __syncthreads();
  if (threadIdx.x < kClasses)
    sAt[threadIdx.x] = sCount[threadIdx.x] ? atomicAdd(&P.meta[kPullNext + threadIdx.x], sCount[threadIdx.x]) : 0;
  __syncthreads();
  if (is_root) P.size[P.linked[k]] = sBase[c] + ((sAt[c] + at) << c);
}

__global__ __launch_bounds__(kThreads) void pull_move_kernel(const PullInst* __restrict__ insts) {
  const PullInst P = insts[blockIdx.y];
  const int k = blockIdx.x * kThreads + threadIdx.x;
  if ((P.meta[kPullFlags] & ~kPullSelf) || k >= P.meta[kPullLinked]) return;
  const int p = P.linked[k], at = atomicAdd(P.size + P.root[k], 1);
  P.ops[P.main + at] = P.ops[p];
  P.ops[p].op = kFillNop;
}

}  // namespace

void launch_pull(int NT, int ng, const PullInst* insts, int n, int max_main, int max_ops, hipStream_t s) {
  if (n <= 0 || max_main <= 0) return;
  const dim3 grid((max_main + kThreads - 1) / kThreads, n), all((max_ops + kThreads - 1) / kThreads, n);
  pull_init_kernel<<<all, kThreads, 0, s>>>(insts);
  AMR_DISPATCH_TILE(NT, ng, (pull_kernel<T, G><<<grid, kThreads, 0, s>>>(insts)));
  pull_link_kernel<<<grid, kThreads, 0, s>>>(insts);
  pull_size_kernel<<<grid, kThreads, 0, s>>>(insts);
  pull_classes_kernel<<<grid, kThreads, 0, s>>>(insts);
  pull_place_kernel<<<grid, kThreads, 0, s>>>(insts);
  pull_move_kernel<<<grid, kThreads, 0, s>>>(insts);
}

}  // namespace amr
