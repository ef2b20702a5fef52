// nlist_csr.cpp -- full CSR Verlet list for the DeviceNeighborList boundary
// (src/neighbors/device_neighbor_list.cu:26-139,158-278).
//
// Atom i's row holds the atoms of the 27 stencil cells (z, y, x outer to
// inner, single periodic wrap -- cell_list.hpp:47-56) that pass a test in
// FP64 exactly as the CPU half list does (neighbor_list.cpp:58-62):
// d = x_j - x_i, one conditional minimum image per axis, r2 = dx*dx + dy*dy
// + dz*dz rounded term by term, include iff r2 < r_list^2. Because
// (x_j - x_i) == -(x_i - x_j) exactly in IEEE arithmetic and the minimum
// image is odd, the GPU full list is exactly the symmetric closure of the
// CPU half list. The cell of atom i is the one the cell build assigned
// (computed once, not re-derived in a second precision as the reference's
// kernel does at :43-58).
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace tdmd_hip {

namespace {

// One lane per atom: the search of sparse systems (see nlist_csr below).
template <bool kFill>
__global__ void __launch_bounds__(kBlock)
nlist_csr_kernel(const double* __restrict__ pos, int natoms, DevBox box, double r_list_sq,
                 const int32_t* __restrict__ cell_counts, const int32_t* __restrict__ cell_offsets,
                 const int32_t* __restrict__ cell_atoms, const int32_t* __restrict__ atom_cells,
                 int ncx, int ncy, int ncz, const int32_t* __restrict__ offsets,
                 int32_t* __restrict__ neighbors, int32_t* __restrict__ counts, int max_neighbors,
                 int32_t* __restrict__ overflow) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= natoms) return;
  const double xi = pos[3 * i], yi = pos[3 * i + 1], zi = pos[3 * i + 2];
  const double hx = 0.5 * box.size[0], hy = 0.5 * box.size[1], hz = 0.5 * box.size[2];
  const int ci = atom_cells[i];
  const int iz = ci / (ncx * ncy);
  const int iy = (ci - iz * ncx * ncy) / ncx;
  const int ix = ci - iz * ncx * ncy - iy * ncx;
  const int off = kFill ? offsets[i] : 0;
  int count = 0;
  for (int dz = -1; dz <= 1; ++dz) {
    int nz = iz + dz;
    nz = nz < 0 ? nz + ncz : (nz >= ncz ? nz - ncz : nz);
    for (int dy = -1; dy <= 1; ++dy) {
      int ny = iy + dy;
      ny = ny < 0 ? ny + ncy : (ny >= ncy ? ny - ncy : ny);
      for (int dx = -1; dx <= 1; ++dx) {
        int nx = ix + dx;
        nx = nx < 0 ? nx + ncx : (nx >= ncx ? nx - ncx : nx);
        const int c = nz * ncx * ncy + ny * ncx + nx;
        const int start = cell_offsets[c], cnt = cell_counts[c];
        for (int k = 0; k < cnt; ++k) {
          const int j = cell_atoms[start + k];
          if (j == i) continue;
          const double ddx = min_image(pos[3 * j] - xi, box.size[0], hx, box.periodic[0]);
          const double ddy = min_image(pos[3 * j + 1] - yi, box.size[1], hy, box.periodic[1]);
          const double ddz = min_image(pos[3 * j + 2] - zi, box.size[2], hz, box.periodic[2]);
          if (r2_unfused(ddx, ddy, ddz) < r_list_sq) {
            if (kFill) {
              if (count < max_neighbors)
                neighbors[off + count] = j;
              else
                atomicMax(overflow, count + 1);
            }
            ++count;
          }
        }
      }
    }
  }
  counts[i] = count;
}


// One workgroup per cell (or, for crowded cells among sparse ones, several, each
// with its share of the cell's atoms), for cells that hold a few atoms or more.
//
// The candidates of a cell -- the atoms of its 27 stencil cells, in stencil
// order (z, y, x outer to inner, then cell order), the order of the rows --
// are staged in LDS once for all atoms of the cell, as FP32 offsets from the
// cell's centre with their index. A wavefront takes two atoms at a time and
// tests 64 candidates a turn against both: FP32 r^2 decides outside a narrow
// band around r_list^2, nlist_csr_kernel's FP64 test on the caller's
// positions inside it (a few candidates per million). Hits are written side
// by side at their rank (ballot, prefix count).
//
// What FP32 may decide. Offsets are of the periodic image nearest the
// centre, k box lengths from where the atom is. Take an atom i with k = 0
// that reaches less than half a box from the centre on every periodic axis:
// a candidate with k in {-1, 0, 1} that comes out near i does so in the image
// that the single minimum image picks. Candidates with a larger k get a NaN
// offset (undecided); for an i with k != 0 FP32 only rejects; where r_list
// reaches further (boxes of under 3 r_list) differences are folded again,
// which leaves them no longer than any single image, and FP32 only rejects.
// Rounding: offsets to 2^-24 of at most 4 r_list for a candidate that could
// be near, i within 2 r_list of the centre, so r^2 is within 2e-6 of its
// value where the margin is 1e-5; an i further out (open axes) asks the FP64
// test about every candidate.
//
// Bound by VALU issue, ~9 (count) and ~13 (fill) instructions per atom and 64
// candidates. One lane per atom instead walks ~650 candidates in turn, each
// a dependent index load, three 8-byte gathers and ~45 FP64 instructions.
constexpr double kPreMargin = 1e-5;
constexpr int kHomeMax = 64;  // atoms of a cell staged at a time

__device__ __forceinline__ int rank_below(unsigned long long mask) {
  return static_cast<int>(__builtin_amdgcn_mbcnt_hi(
      static_cast<unsigned>(mask >> 32),
      __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0u)));
}

template <bool kFill, int kThreads>
__global__ void __launch_bounds__(kThreads)
nlist_csr_cell_kernel(const double* __restrict__ pos, int ncells, DevBox box, double r_list,
                      const int32_t* __restrict__ cell_counts,
                      const int32_t* __restrict__ cell_offsets,
                      const int32_t* __restrict__ cell_atoms, int ncx, int ncy, int ncz,
                      const int32_t* __restrict__ offsets, int32_t* __restrict__ neighbors,
                      int32_t* counts, int max_neighbors, int32_t* __restrict__ overflow) {
  constexpr int kWaves = kThreads / kWave;
  constexpr int kCandMax = kThreads >= 256 ? 1024 : 256;  // candidates staged at a time
  __shared__ float4 cand[kCandMax];
  __shared__ float4 home_at[kHomeMax];  // an atom's FP32 offset and index
  __shared__ int home_how[kHomeMax];    // 0: FP32 decides, 1: rejects, 2: neither; 4: fold
  __shared__ int run_start[27], run_end[27];  // run t: candidates [run_end[t-1], run_end[t])
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const double L[3] = {box.size[0], box.size[1], box.size[2]};
  const double inv[3] = {box.periodic[0] ? 1.0 / L[0] : 0.0, box.periodic[1] ? 1.0 / L[1] : 0.0,
                         box.periodic[2] ? 1.0 / L[2] : 0.0};
  const double r_list_sq = r_list * r_list;
  const float sure = static_cast<float>(r_list_sq * (1.0 - kPreMargin));
  const float out = static_cast<float>(r_list_sq * (1.0 + kPreMargin));
  // each XCD takes a contiguous run of cells (the grid is a multiple of 8)
  const int per = (ncells + 7) >> 3;
  for (int b = static_cast<int>(blockIdx.x) >> 3; b < per; b += static_cast<int>(gridDim.x) >> 3) {
    const int c = (static_cast<int>(blockIdx.x) & 7) * per + b;
    if (c >= ncells) return;
    const int n_home = cell_counts[c];
    // (a cell's atoms go to gridDim.y workgroups, kHomeMax at a time)
    if (n_home <= kHomeMax * static_cast<int>(blockIdx.y)) continue;
    const int home = cell_offsets[c];
    const int iz = c / (ncx * ncy);
    const int iy = (c - iz * ncx * ncy) / ncx;
    const int ix = c - iz * ncx * ncy - iy * ncx;
    __syncthreads();  // the LDS of the previous cell is done with
    if (w == 0) {
      int cnt = 0;
      if (lane < 27) {
        int nz = iz + lane / 9 - 1, ny = iy + (lane / 3) % 3 - 1, nx = ix + lane % 3 - 1;
        nz = nz < 0 ? nz + ncz : (nz >= ncz ? nz - ncz : nz);
        ny = ny < 0 ? ny + ncy : (ny >= ncy ? ny - ncy : ny);
        nx = nx < 0 ? nx + ncx : (nx >= ncx ? nx - ncx : nx);
        const int nc = nz * ncx * ncy + ny * ncx + nx;
        cnt = cell_counts[nc];
        run_start[lane] = cell_offsets[nc];
      }
      int incl = cnt;
      for (int off = 1; off < 32; off <<= 1) {
        const int o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
      }
      if (lane < 27) run_end[lane] = incl;
    }
    __syncthreads();
    const int total = run_end[26];
    const double ctr[3] = {box.lo[0] + (ix + 0.5) * (L[0] / ncx),
                           box.lo[1] + (iy + 0.5) * (L[1] / ncy),
                           box.lo[2] + (iz + 0.5) * (L[2] / ncz)};
    // offset from the centre in the nearest image, *k box lengths away
    auto rel = [&](int a, double x, double* k) {
      const double d = x - ctr[a];
      *k = rint(d * inv[a]);
      return d - L[a] * *k;
    };
    for (int c0 = 0; c0 < total; c0 += kCandMax) {
      const int m = min(kCandMax, total - c0);
      const int m64 = (m + 63) & ~63;
      if (c0 > 0) __syncthreads();  // the previous chunk is done with
      for (int q = threadIdx.x; q < m64; q += kThreads) {
        // (padding: beyond every radius)
        float4 v = make_float4(__builtin_huge_valf(), 0.0f, 0.0f, __int_as_float(-1));
        if (q < m) {
          // the run that candidate c0 + q lies in: the first that ends beyond it
          int t = 0;
#pragma unroll
          for (int step = 16; step > 0; step >>= 1)
            if (t + step <= 26 && run_end[t + step - 1] <= c0 + q) t += step;
          const int j = cell_atoms[run_start[t] + (c0 + q - (t > 0 ? run_end[t - 1] : 0))];
          const double* p = pos + 3 * static_cast<int64_t>(j);
          double kx, ky, kz;
          const double x = rel(0, p[0], &kx), y = rel(1, p[1], &ky), z = rel(2, p[2], &kz);
          const bool ok = fabs(kx) <= 1.0 && fabs(ky) <= 1.0 && fabs(kz) <= 1.0;
          v = make_float4(ok ? static_cast<float>(x) : __builtin_nanf(""), static_cast<float>(y),
                          static_cast<float>(z), __int_as_float(j));
        }
        cand[q] = v;
      }
      const int first = kHomeMax * static_cast<int>(blockIdx.y);
      for (int h0 = first; h0 < n_home; h0 += kHomeMax * static_cast<int>(gridDim.y)) {
        const int nh = min(kHomeMax, n_home - h0);
        if (h0 > first) __syncthreads();  // the previous atoms are done with
        if (static_cast<int>(threadIdx.x) < nh) {
          const int i = cell_atoms[home + h0 + static_cast<int>(threadIdx.x)];
          const double* p = pos + 3 * static_cast<int64_t>(i);
          double kx, ky, kz;
          const double x = rel(0, p[0], &kx), y = rel(1, p[1], &ky), z = rel(2, p[2], &kz);
          const double reach = r_list * (1.0 + kPreMargin);
          const bool fold = (box.periodic[0] && !(fabs(x) + reach <= 0.5 * L[0])) ||
                            (box.periodic[1] && !(fabs(y) + reach <= 0.5 * L[1])) ||
                            (box.periodic[2] && !(fabs(z) + reach <= 0.5 * L[2]));
          const bool near =
              fabs(x) <= 2.0 * r_list && fabs(y) <= 2.0 * r_list && fabs(z) <= 2.0 * r_list;
          const bool put = kx == 0.0 && ky == 0.0 && kz == 0.0;
          home_at[threadIdx.x] = make_float4(static_cast<float>(x), static_cast<float>(y),
                                             static_cast<float>(z), __int_as_float(i));
          home_how[threadIdx.x] = !near ? 2 : fold ? 5 : put ? 0 : 1;
        }
        __syncthreads();
        for (int a0 = 2 * w; a0 < nh; a0 += 2 * kWaves) {
          // two atoms a wavefront (the second repeats the first in an odd cell)
          const float4 at[2] = {home_at[a0], home_at[min(a0 + 1, nh - 1)]};
          const int i[2] = {__builtin_amdgcn_readfirstlane(__float_as_int(at[0].w)),
                            __builtin_amdgcn_readfirstlane(__float_as_int(at[1].w))};
          const int how = __builtin_amdgcn_readfirstlane(home_how[a0]) |
                          __builtin_amdgcn_readfirstlane(home_how[min(a0 + 1, nh - 1)]);
          const float lo2 = how ? -1.0f : sure;
          const float hi2 = (how & 2) ? __builtin_huge_valf() : out;
          int off[2], count[2] = {0, 0};
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            off[u] = kFill ? __builtin_amdgcn_readfirstlane(offsets[i[u]]) : 0;
            // hits of earlier chunks: stored by this wave's lane 0
            if (c0 > 0) count[u] = __builtin_amdgcn_readfirstlane(counts[i[u]]);
          }
          const bool two = a0 + 1 < nh;
          auto turn = [&](int k, auto folds) {
            const float4 p = cand[k + lane];
            const int j = __float_as_int(p.w);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              float dx = p.x - at[u].x, dy = p.y - at[u].y, dz = p.z - at[u].z;
              if constexpr (decltype(folds)::value) {
                dx -= static_cast<float>(L[0]) * rintf(dx * static_cast<float>(inv[0]));
                dy -= static_cast<float>(L[1]) * rintf(dy * static_cast<float>(inv[1]));
                dz -= static_cast<float>(L[2]) * rintf(dz * static_cast<float>(inv[2]));
              }
              const float r2 = dx * dx + dy * dy + dz * dz;
              unsigned long long mask = __builtin_amdgcn_ballot_w64(r2 < lo2);
              const unsigned long long ask = __builtin_amdgcn_ballot_w64(!(r2 > hi2)) & ~mask;
              if (ask != 0) {
                bool hit = false;
                if (((ask >> lane) & 1ull) && j >= 0) {
                  const double* pi = pos + 3 * static_cast<int64_t>(i[u]);
                  const double* pj = pos + 3 * static_cast<int64_t>(j);
                  const double ddx = min_image(pj[0] - pi[0], L[0], 0.5 * L[0], box.periodic[0]);
                  const double ddy = min_image(pj[1] - pi[1], L[1], 0.5 * L[1], box.periodic[1]);
                  const double ddz = min_image(pj[2] - pi[2], L[2], 0.5 * L[2], box.periodic[2]);
                  hit = r2_unfused(ddx, ddy, ddz) < r_list_sq;
                }
                mask |= __builtin_amdgcn_ballot_w64(hit);
              }
              mask &= ~__builtin_amdgcn_ballot_w64(j == i[u]);
              const int n = __popcll(mask);
              if constexpr (kFill) {
                if (u == 0 || two) {
                  const int rank = rank_below(mask);
                  int32_t* row = neighbors + off[u] + count[u];
                  if (((mask >> lane) & 1ull) && rank < max_neighbors - count[u]) row[rank] = j;
                }
              }
              count[u] += n;
            }
          };
          if (how & 4) {
            for (int k = 0; k < m; k += kWave) turn(k, std::true_type{});
          } else {
            for (int k = 0; k < m; k += kWave) turn(k, std::false_type{});
          }
          if (lane == 0) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              if (u == 1 && !two) break;
              counts[i[u]] = count[u];
              if (kFill && count[u] > max_neighbors && c0 + kCandMax >= total)
                atomicMax(overflow, count[u]);
            }
          }
        }
      }
    }
  }
}

template <bool kFill>
int launch_cells(int threads, int parts, const double* pos, int64_t ncells, const DevBox& box,
                 double r_list, const int32_t* cc, const int32_t* co, const int32_t* ca,
                 const int32_t n[3], const int32_t* offsets, int32_t* nbrs, int32_t* counts, int32_t max_nb,
                 int32_t* overflow, hipStream_t stream) {
  const int grid = static_cast<int>(std::min<int64_t>((ncells + 7) / 8 * 8, 1 << 20));
  auto go = [&](auto kernel) {
    kernel<<<dim3(grid, parts), threads, 0, stream>>>(
        pos, static_cast<int>(ncells), box, r_list, cc, co, ca, n[0], n[1], n[2], offsets, nbrs,
        counts, max_nb, overflow);
  };
  switch (threads) {
    case 64: go(&nlist_csr_cell_kernel<kFill, 64>); break;
    case 256: go(&nlist_csr_cell_kernel<kFill, 256>); break;
    case 512: go(&nlist_csr_cell_kernel<kFill, 512>); break;
    default: go(&nlist_csr_cell_kernel<kFill, 1024>); break;
  }
  TDMD_LAUNCH_CHECK();
  return TDMD_OK;
}

}  // namespace

int nlist_csr(bool fill, const double* d_pos, int64_t natoms, const tdmd_box& box, double r_list,
              const int32_t* cc, const int32_t* co, const int32_t* ca, const int32_t* ac,
              const int32_t n[3], const int32_t* offsets, int32_t* nbrs, int32_t* counts,
              int32_t max_nb, int32_t* overflow, hipStream_t stream) {
  if (natoms == 0) return TDMD_OK;
  const DevBox db = make_devbox(box);
  const double r_list_sq = r_list * r_list;
  const int na = static_cast<int>(natoms);
  // A workgroup per cell where cells hold two atoms or more on average (or
  // half an atom, in at most 65,536 cells); a lane per atom in sparser
  // systems. Workgroup size by how many cells there are to fill the chip with
  // and how many atoms share a cell's candidates. Count / fill, us, random
  // atoms, r_list 6.5 A:
  //   atoms, cells (per cell)   lane        64       256       512       1024
  //   4,000      125 (32)     616 / 763   96 / 142  22 / 33   13 / 20   10 / 14
  //   16,384     512 (32)     643 / 774   96 / 141  21 / 34   15 / 23   16 / 24
  //   65,536    2744 (24)     520 / 646   69 / 103  35 / 53   45 / 65   59 / 82
  //   268,960 10,648 (25)    1315 / 1591 147 / 219 110 / 169 162 / 237 219 / 307
  //   2,000      343 (6)      138 / 173    9 / 13    6 / 7     7 / 6     9 / 10
  //   1M         250k (4)    1257 / 1417 241 / 291 643 / 764
  //   65,536    64,000 (1)     74 / 83    37 / 43  125 / 136
  //   65,536   125,000 (0.5)   56 / 60    56 / 62  196 / 210
  //   1M          1M (1)      433 / 468  483 / 557
  // Where a cell's workgroup is a wavefront, up to four share a cell of more than
  // 64 atoms, for droplets with long cutoffs; the idle ones of other cells cost
  // ~1 us per 4,000 cells each. Parts 1, 2, 4 against a lane per atom:
  //   10,976 atoms, r_list 20 A, 8,000 cells    11151 / 17784  5673 / 9047
  //                                  3034 / 4837; lane 8936 / 11347
  //   32,768 atoms in as many cells  21 / 24  26 / 30  41 / 47; lane 75 / 84
  //   64,000 atoms in as many cells  36 / 41  48 / 55  78 / 88; lane 75 / 83
  const int64_t ncells = static_cast<int64_t>(n[0]) * n[1] * n[2];
  if (natoms >= 2 * ncells || (ncells <= 65536 && 2 * natoms >= ncells)) {
    const bool dense = natoms >= 8 * ncells;
    const int threads = dense ? (ncells >= 2048 ? 256 : ncells >= 216 ? 512 : 1024)
                              : (ncells >= 1024 ? 64 : 256);
    const int parts = threads > 64 ? 1 : ncells <= 32768 ? 4 : ncells <= 65536 ? 2 : 1;
    return fill ? launch_cells<true>(threads, parts, d_pos, ncells, db, r_list, cc, co, ca, n,
                                     offsets, nbrs, counts, max_nb, overflow, stream)
                : launch_cells<false>(threads, parts, d_pos, ncells, db, r_list, cc, co, ca, n,
                                      nullptr, nullptr, counts, 0, nullptr, stream);
  }
  if (fill) {
    nlist_csr_kernel<true><<<grid_for(natoms), kBlock, 0, stream>>>(
        d_pos, na, db, r_list_sq, cc, co, ca, ac, n[0], n[1], n[2], offsets, nbrs, counts,
        max_nb, overflow);
  } else {
    nlist_csr_kernel<false><<<grid_for(natoms), kBlock, 0, stream>>>(
        d_pos, na, db, r_list_sq, cc, co, ca, ac, n[0], n[1], n[2], nullptr, nullptr, counts, 0,
        nullptr);
  }
  TDMD_LAUNCH_CHECK();
  return TDMD_OK;
}

}  // namespace tdmd_hip

using namespace tdmd_hip;

extern "C" {

int tdmd_nlist_count(const double* d_pos, int64_t natoms, const tdmd_box* box, double r_list,
                     const int32_t* d_cell_counts, const int32_t* d_cell_offsets,
                     const int32_t* d_cell_atoms, const int32_t* d_atom_cells,
                     const int32_t ncells[3], int32_t* d_counts, void* stream) {
  if (!box || !ncells || !(r_list > 0.0) || natoms < 0 || natoms > INT32_MAX)
    return fail(TDMD_E_INVALID, "nlist_count: bad arguments");
  if (natoms > 0 && (!d_pos || !d_cell_counts || !d_cell_offsets || !d_cell_atoms ||
                     !d_atom_cells || !d_counts))
    return fail(TDMD_E_INVALID, "nlist_count: null pointer");
  return nlist_csr(false, d_pos, natoms, *box, r_list, d_cell_counts, d_cell_offsets,
                   d_cell_atoms, d_atom_cells, ncells, nullptr, nullptr, d_counts, 0, nullptr,
                   as_stream(stream));
}

int tdmd_nlist_fill(const double* d_pos, int64_t natoms, const tdmd_box* box, double r_list,
                    const int32_t* d_cell_counts, const int32_t* d_cell_offsets,
                    const int32_t* d_cell_atoms, const int32_t* d_atom_cells,
                    const int32_t ncells[3], const int32_t* d_offsets, int32_t* d_neighbors,
                    int32_t* d_counts, int32_t max_neighbors, int32_t* d_overflow,
                    void* stream) {
  if (!box || !ncells || !(r_list > 0.0) || natoms < 0 || natoms > INT32_MAX ||
      max_neighbors < 0)
    return fail(TDMD_E_INVALID, "nlist_fill: bad arguments");
  if (natoms > 0 && (!d_pos || !d_cell_counts || !d_cell_offsets || !d_cell_atoms ||
                     !d_atom_cells || !d_offsets || !d_counts || !d_overflow ||
                     (max_neighbors > 0 && !d_neighbors)))
    return fail(TDMD_E_INVALID, "nlist_fill: null pointer");
  return nlist_csr(true, d_pos, natoms, *box, r_list, d_cell_counts, d_cell_offsets,
                   d_cell_atoms, d_atom_cells, ncells, d_offsets, d_neighbors, d_counts,
                   max_neighbors, d_overflow, as_stream(stream));
}

}  // extern "C"
