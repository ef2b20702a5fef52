// csr_rows.hpp -- row loop of the passes over a full CSR list (drop-in Morse
// and EAM forces, force matching): kRowLanes neighbouring lanes per row.
#pragma once

#include <algorithm>

#include "pair_math.hpp"

namespace tdmd_hip {

// Lanes per row, and slots a lane takes at a time (kSlots of for_row). Rows of
// a solid have ~90-120 slots. us without / with the energy, by lanes x slots:
//   atoms                  4x4         8x1         8x2         8x4        16x2
//   EAM mixed   16,384   22 / 39     17 / 36     17 / 36     18 / 37     17 / 39
//   EAM mixed  131,072  110 / 112   116 / 117   108 / 110   101 / 105   105 / 110
//   EAM mixed  1M      1057 / 1037 1201 / 1231 1086 / 1100  961 / 951   996 / 1035
//   Morse FP64  16,384   14 / 34     12 / 36     12 / 36     12 / 37     12 / 40
//   Morse FP64 131,072   70 / 79     68 / 83     71 / 82     72 / 85     74 / 89
//   Morse FP64 1M       480 / 537   550 / 596   491 / 572   504 / 583   535 / 643
//   Morse, 1M atoms of a gas, rows of ~4 slots:
//                         38          46          49          66          91
// (one lane: EAM mixed 167, 368, 5445; Morse FP64 105, 216, 4515; gas 64).
// The passes are bound by their gathers (three 8-byte words of a position,
// one or two table quads, F' per slot: ~20 lines of L1 a wave and slot).
constexpr int kRowLanes = 8;
constexpr int kMorseSlots = 2;
constexpr int kEamSlots = 4;
constexpr int kEnergyBlock = 1024;  // with the energy: 256 atoms a workgroup, in turns

// Box of the pair geometry: half is infinite on an open axis.
struct PairBox {
  double size[3], half[3];
};

inline PairBox make_pair_box(const DevBox& b) {
  PairBox p;
  for (int a = 0; a < 3; ++a) {
    p.size[a] = b.size[a];
    p.half[a] = b.periodic[a] ? 0.5 * b.size[a] : __builtin_huge_val();
  }
  return p;
}

// min_image() (common.hpp) by one compare: the same values.
__device__ __forceinline__ double image(double d, double size, double half) {
  return d - (fabs(d) > half ? copysign(size, d) : 0.0);
}

// Sum over the kRowLanes lanes of a row, in every lane.
__device__ __forceinline__ double row_sum(double v) {
#pragma unroll
  for (int w = kRowLanes / 2; w > 0; w >>= 1) v += __shfl_xor(v, w, 64);
  return v;
}

// A neighbour as the passes read it: its position, and what else of it they
// want fetched with the position.
struct Neighbour {
  double x, y, z;
};
__device__ __forceinline__ Neighbour neighbour_at(const double* __restrict__ pos, int j) {
  const double* p = pos + 3 * static_cast<int64_t>(j);
  return Neighbour{p[0], p[1], p[2]};
}

// pair(j, load(j), dx, dy, dz, r2) for this lane's slots of a row, kSlots at
// a time: the indices of the next turn are loaded before this turn's loads
// are waited for, without a branch (past the row's end the last slot is read
// again and not evaluated).
template <int kSlots, class Load, class Pair>
__device__ __forceinline__ void for_row(const int32_t* __restrict__ nbrs, int off, int cnt,
                                        double xi, double yi, double zi, const PairBox& box,
                                        Load&& load, Pair&& pair) {
  if (cnt <= 0) return;
  const int32_t* row = nbrs + off;
  const int part = static_cast<int>(threadIdx.x) % kRowLanes;
  int j[kSlots];
#pragma unroll
  for (int u = 0; u < kSlots; ++u) j[u] = row[min(part + u * kRowLanes, cnt - 1)];
  for (int k = part; k < cnt; k += kSlots * kRowLanes) {
    decltype(load(0)) v[kSlots];
    double dx[kSlots], dy[kSlots], dz[kSlots], r2[kSlots];
    int jn[kSlots];
#pragma unroll
    for (int u = 0; u < kSlots; ++u) v[u] = load(j[u]);
#pragma unroll
    for (int u = 0; u < kSlots; ++u)
      jn[u] = row[min(k + (kSlots + u) * kRowLanes, cnt - 1)];
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
      dx[u] = image(xi - v[u].x, box.size[0], box.half[0]);
      dy[u] = image(yi - v[u].y, box.size[1], box.half[1]);
      dz[u] = image(zi - v[u].z, box.size[2], box.half[2]);
      r2[u] = dx[u] * dx[u] + dy[u] * dy[u] + dz[u] * dz[u];
    }
#pragma unroll
    for (int u = 0; u < kSlots; ++u)
      if (k + u * kRowLanes < cnt) pair(j[u], v[u], dx[u], dy[u], dz[u], r2[u]);
#pragma unroll
    for (int u = 0; u < kSlots; ++u) j[u] = jn[u];
  }
}

// Blocks are dealt round-robin to the 8 XCDs: block b of `n` takes piece
// piece_of(b, n) of the atoms, so that an XCD's pieces are consecutive and
// their rows' positions stay in its L2.
__device__ __forceinline__ int64_t piece_of(int b, int n) {
  const int per = n >> 3;
  return b < 8 * per ? static_cast<int64_t>(b & 7) * per + (b >> 3) : b;
}

// The workgroup's atoms [begin, end): kThreads / kRowLanes at a time. With
// the energy a workgroup takes 256 atoms, whose sum is partial piece_of(b);
// without, one turn's atoms (a grid of at most kMaxGrid strides over them).
constexpr int kMaxGrid = 1 << 22;

template <bool kEnergy, class Atom>
__device__ __forceinline__ void for_atoms(int count, Atom&& atom) {
  constexpr int kThreads = kEnergy ? kEnergyBlock : kBlock;
  constexpr int kTurn = kThreads / kRowLanes;
  const int64_t piece = piece_of(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
  const int sub = static_cast<int>(threadIdx.x) / kRowLanes;
  if (kEnergy) {
    for (int t = 0; t < kBlock; t += kTurn) {
      const int64_t i = piece * kBlock + t + sub;
      if (i < count) atom(static_cast<int>(i));
    }
  } else {
    for (int64_t i = piece * kTurn + sub; i < count;
         i += static_cast<int64_t>(gridDim.x) * kTurn)
      atom(static_cast<int>(i));
  }
}

inline int row_grid(int count, bool energy) {
  if (energy) return grid_for(count);
  return static_cast<int>(std::min<int64_t>(
      (static_cast<int64_t>(count) * kRowLanes + kBlock - 1) / kBlock, kMaxGrid));
}

// The tables' layout by value: the F splines share one grid, all r splines
// another (setfl: one Nrho, drho, Nr, dr), every table starts at 0.
struct EamLayout {
  SplineMeta F, r;  // offset of element 0's F and rho
  int ntypes;
  double rc_sq;
  __device__ __forceinline__ int f_at(int t) const { return t * (F.n - 1); }
  __device__ __forceinline__ int rho_at(int t) const { return r.offset + t * (r.n - 1); }
  __device__ __forceinline__ int phi_at(int p) const {
    return r.offset + (ntypes + p) * (r.n - 1);
  }
};

inline EamLayout eam_layout(const tdmd_eam_tables* t) {
  EamLayout e;
  e.F = SplineMeta{t->drho, 1.0 / t->drho, 0.0, t->nrho, 0};
  e.r = SplineMeta{t->dr, 1.0 / t->dr, 0.0, t->nr, t->ntypes * (t->nrho - 1)};
  e.ntypes = t->ntypes;
  e.rc_sq = t->cutoff * t->cutoff;
  return e;
}

// Derivative and value of one interval's cubic, spline_deriv's and
// spline_value's expressions.
template <class R, class Q>
__device__ __forceinline__ R quad_deriv(const Q& c, R dx) {
  return c.y + dx * (static_cast<R>(2) * c.z + dx * static_cast<R>(3) * c.w);
}
template <class R, class Q>
__device__ __forceinline__ R quad_value(const Q& c, R dx) {
  return c.x + dx * (c.y + dx * (c.z + dx * c.w));
}

}  // namespace tdmd_hip
