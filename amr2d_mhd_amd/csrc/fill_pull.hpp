// The ghost fill by destination: what one ring element of a leaf holds after the
// sequential fill (boundary.cpp / boundaryfc.cpp / boundaryec.cpp,
// extboundary.cpp), found backwards from the element, on the host or the device.
//
// The reference's fill walks an ordered list of (block, side) entries
// (locate_bounds.cpp:35-208), the internal ones in block order, then those at
// the domain's boundary.  On a tree whose levels step by one with neighbour
// links that point back (pull_form) every side of a leaf belongs to exactly one
// entry, and an entry writes only the ghost strips of its sides.  So a ring
// element has at most two writers, the entries of the strips it lies in; the
// last of them before a given entry gives its value there: a copy of an element
// as that entry found it, which is looked up the same way, or a restriction of
// four such elements.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

#include "amr_types.hpp"

namespace amr {

// rows: level, father, first son, sibling id, left, right, bottom, top neighbour
struct PullTree {
  const int32_t* lp;
  const uint8_t* leafs;
};

// son offset of the first of the two finer blocks beyond a side, and the step to the second
inline __host__ __device__ int side_son(int s) { return s == 0 ? 1 : s == 2 ? 2 : 0; }
inline __host__ __device__ int side_stride(int s) { return s < 2 ? 2 : 1; }

// What the entry of side s of leaf b writes to element (i, j) of that side's
// ghost strip: a copy of (nb, i, j), or the restriction of the 2x2 elements from
// there; key orders the entries.
struct PullWrite {
  int64_t key;
  int nb, i, j;
  bool restricted;
};

inline __host__ __device__ bool pull_strip(const PullTree& T, int NT, int ng, int b, int s, int i, int j,
                                           PullWrite& w) {
  const int lo = ng, hi = NT - 1 - ng, top = hi + 1, lob = lo - 1, h2 = (NT - 1) / 2;
  const int32_t* row = T.lp + 8 * (size_t)b;
  const int n = row[4 + s];
  w.restricted = false;
  // distance into the strip from its outer edge (left, bottom) or the interior (right, top)
  const int g = s == 0 ? i : s == 1 ? i - top : s == 2 ? j : j - top;
  const bool low = !(s & 1), xs = s < 2;  // side at the low end; strip across x
  auto place = [&](int across, int along) {
    w.i = xs ? across : along;
    w.j = xs ? along : across;
  };
  if (n == -1) {
    // extboundary.cpp:5-61: mirror of the interior, after all internal entries
    w.key = ((int64_t)1 << 40) + 4 * b + s;
    w.nb = b;
    place(low ? lo + ng - 1 - g : hi - g, xs ? j : i);
    return true;
  }
  const int32_t* nrow = T.lp + 8 * (size_t)n;
  if (nrow[0] < row[0]) {
    // injection from the coarser leaf (boundary.cpp:97-107 and its siblings)
    const int o = s ^ 1;
    w.key = 4 * (int64_t)n + o;
    w.nb = n;
    const bool first = T.lp[8 * (size_t)nrow[4 + o] + 2] + side_son(o) == b;
    const int a = xs ? j : i;
    const int along = first ? (a + ng) / 2 : (a - ng + 2) / 2 + h2;
    // a low strip of b lies at the high end of n and the reverse
    place(low ? (g + 2) / 2 + hi - ng / 2 : (g + 1 + 2 * ng - 1) / 2, along);
    return true;
  }
  if (T.leafs[n]) {
    // the same level (boundary.cpp:17-35 and its siblings)
    w.key = b < n ? 4 * (int64_t)b + s : 4 * (int64_t)n + (s ^ 1);
    w.nb = n;
    place(low ? hi - (ng - 1) + g : lo + g, xs ? j : i);
    return true;
  }
  // finer neighbours (boundary.cpp:36-107, 128-197, 218-287, 308-377)
  w.key = 4 * (int64_t)b + s;
  const int n1 = nrow[2] + side_son(s), n2 = n1 + side_stride(s);
  const int a = xs ? j : i;  // position along the strip
  if (a >= lo && a <= hi) {
    // restriction: the first half of the rows from n1, the second from n2
    const bool first = a <= h2;
    w.nb = first ? n1 : n2;
    w.restricted = true;
    place(low ? 2 * (g - ng / 2) - ng / 2 + hi : 2 * (g + 1 + (ng / 2 - 1)),
          2 * (first ? a : a - h2 + ng - 1) - lo);
    return true;
  }
  // corners: the block diagonally beyond n1 (low end) or n2 (high end), found
  // through their father's neighbour; copied with same-level indices if it is a
  // leaf, else its designated son restricted if that is one
  const bool end = a > hi;
  const int cs = (xs ? 6 : 4) + end;
  const int cb = T.lp[8 * (size_t)T.lp[8 * (size_t)(end ? n2 : n1) + 1] + cs];
  if (cb == -1) return false;
  const int e = end ? NT - 1 - a : a;  // from the strip's end
  if (T.leafs[cb]) {
    w.nb = cb;
    place(low ? hi - ng + g + 1 : lob + g + 1, end ? lo + ng - (e + 1) : hi - ng + e + 1);
    return true;
  }
  // the son at the corner: nearest to b across, and to the strip's end along
  const int off = xs ? (low ? 1 : 0) + (end ? 0 : 2) : (low ? 2 : 0) + (end ? 0 : 1);
  const int fb = T.lp[8 * (size_t)cb + 2] + off;
  if (!T.leafs[fb]) return false;
  w.nb = fb;
  w.restricted = true;
  // beyond the top side's high end the reference does not mirror the position
  if (s == 3 && end) place(lob + 2 * (g + 1) - 1, lob + 2 * (a - hi) - 1);
  else place(low ? hi - 2 * ng + 2 * g + 1 : lob + 2 * (g + 1) - 1, end ? lo + 2 * ng - 2 * (e + 1) : hi - 2 * ng + 2 * e + 1);
  return true;
}

// An element's value before the entry `key`: another element's pre-fill value, or
// (restricted) the restriction of the 2x2 elements from (nb, i, j) as the entry
// `key` found them.  written: some entry wrote it before.
struct PullValue {
  int64_t key;
  int nb, i, j;
  bool restricted, written;
};

constexpr int64_t kPullEnd = INT64_MAX;

inline __host__ __device__ PullValue pull_value(const PullTree& T, int NT, int ng, int nb, int i, int j, int64_t key) {
  PullValue v{key, nb, i, j, false, false};
  const int hi = NT - 1 - ng;
  while (!v.restricted) {
    const int sx = v.i < ng ? 0 : v.i > hi ? 1 : -1, sy = v.j < ng ? 2 : v.j > hi ? 3 : -1;
    PullWrite w, y;
    bool found = sx >= 0 && pull_strip(T, NT, ng, v.nb, sx, v.i, v.j, w) && w.key < v.key;
    if (sy >= 0 && pull_strip(T, NT, ng, v.nb, sy, v.i, v.j, y) && y.key < v.key && !(found && w.key > y.key)) {
      w = y;
      found = true;
    }
    if (!found) break;
    v = PullValue{w.key, w.nb, w.i, w.j, w.restricted, true};
  }
  return v;
}

// The op of ring element (i, j) of leaf b: kFillNop where it keeps its value, else
// its operands, one element (copy) or four, in FillOp's order.  nested: an operand
// is itself a restriction.
struct PullOp {
  int op, nref;
  int nb[4], i[4], j[4];
  bool nested;
};

inline __host__ __device__ PullOp pull_op(const PullTree& T, int NT, int ng, int b, int i, int j) {
  PullOp o;
  o.nested = false;
  const PullValue v = pull_value(T, NT, ng, b, i, j, kPullEnd);
  if (!v.restricted) {
    o.op = v.nb == b && v.i == i && v.j == j ? kFillNop : kFillCopy;
    o.nref = o.op == kFillCopy;
    o.nb[0] = v.nb;
    o.i[0] = v.i;
    o.j[0] = v.j;
    return o;
  }
  o.op = kFillRestrict;
  o.nref = 4;
  for (int q = 0; q < 4; q++) {
    const PullValue e = pull_value(T, NT, ng, v.nb, v.i + (q >> 1), v.j + (q & 1), v.key);
    if (e.written) o.op = kFillGeneral;
    o.nested |= e.restricted;
    o.nb[q] = e.nb;
    o.i[q] = e.i;
    o.j[q] = e.j;
  }
  return o;
}

// whether some op of the fill writes element (i, j) of leaf b
inline __host__ __device__ bool pull_filled(const PullTree& T, int NT, int ng, int b, int i, int j) {
  if (i >= ng && i < NT - ng && j >= ng && j < NT - ng) return false;
  const PullValue v = pull_value(T, NT, ng, b, i, j, kPullEnd);
  return v.restricted || v.nb != b || v.i != i || v.j != j;
}

// Whether the fill of the tree is of this form: every side of a leaf is at the
// domain's boundary, beside a leaf of its level, beside one of the level above
// of whose two finer neighbours it is one, or beside two leaves of the level
// below; all pointing back.  All blocks that a fill reads or writes are leaves.
inline bool pull_form(const PullTree& T, int nblocks) {
  auto at = [&](int b, int k) { return T.lp[8 * (size_t)b + k]; };
  for (int b = 0; b < nblocks; b++) {
    if (!T.leafs[b]) continue;
    for (int s = 0; s < 4; s++) {
      const int n = at(b, 4 + s), o = s ^ 1;
      if (n == -1) continue;
      if (n == b) return false;
      if (at(n, 0) == at(b, 0)) {
        if (T.leafs[n]) {
          if (at(n, 4 + o) != b) return false;
          continue;
        }
        const int f1 = at(n, 2) + side_son(s), f2 = f1 + side_stride(s);
        for (int f : {f1, f2})
          if (!T.leafs[f] || at(f, 0) != at(b, 0) + 1 || at(f, 4 + o) != b) return false;
      } else if (at(n, 0) == at(b, 0) - 1 && T.leafs[n]) {
        const int m = at(n, 4 + o);
        if (m == -1 || T.leafs[m] || at(m, 0) != at(n, 0)) return false;
        const int f1 = at(m, 2) + side_son(o);
        if (b != f1 && b != f1 + side_stride(o)) return false;
      } else {
        return false;
      }
    }
  }
  return true;
}

}  // namespace amr
