// fm.cpp -- force matching on the GPU: the loss L = sum_i |F_i - T_i|^2
// over a fixed set of configurations (snapshots) and its adjoint gradient
// with respect to the Morse parameters (D, alpha, r0) or the knot values of a
// single-element EAM (F(rho), rho(r), phi(r) as EamAlloy holds them). No
// reference counterpart: this is the fitting path built on the same pair
// arithmetic as the force kernels (pair_math.hpp).
//
// Layout: the snapshots are one concatenated system of nsnap * natoms atoms
// (AoS FP64 positions) sharing one box; each snapshot's full CSR list is
// built once at creation with global indices, so every pass is a single launch
// over all snapshots. The half list (neighbours j > i) beside it and the EAM
// adjoint's records are built by the first call whose passes read them.
// Rows are read by eight lanes side by side (csr_rows.hpp).
//
// Adjoint (ordered pairs i -> j, d = x_i - x_j, u = d / r, g = F - T):
//   Morse:  dL/dtheta = sum 2 (g_i . d) dfpair/dtheta        (one pass)
//   EAM:    w_ij = -2 (g_i - g_j) . u_ij
//           phi'  coefficients  (b,c,d)[k(r)] += w/2 * (1, 2t, 3t^2)     per ordered pair,
//           rho'  coefficients  (b,c,d)[k(r)] += w/2 (Fp_i+Fp_j) (1, 2t, 3t^2),
//           lam_i = sum_j w_ij rho'(r_ij),
//           F     coefficients  (b,c,d)[k(rho_i)] += lam_i (1, 2t, 3t^2),
//           mu_i = lam_i F''(rho_i),
//           rho   coefficients  (a,b,c,d)[k(r)] += mu_i (1, t, t^2, t^3).
//   (w/2 per ordered pair: the two orderings of a pair give w in total, and
//   mu_i + mu_j: the histogram pass takes each pair once.)
// Coefficient gradients go back to knot values through the transpose of the
// FD-Hermite construction (eam_alloy.cpp:19-50).
//
// FP64 (and mixed tables of more points than seven FP32 histograms fit the
// LDS for) takes three passes: lam_i over full rows; the F coefficients and
// mu_i per atom; the phi and rho coefficients per unordered pair, seven adds
// each, in FP64 histograms in LDS where they fit. (One pass over ordered
// pairs, ten global FP64 atomics each: 21.3 ms an evaluation of 100 x 4,000
// atoms, 5000 points, 0.8 ms so.)
//
// Mixed precision: pair geometry and r in FP64, spline and Morse arithmetic
// in FP32 (as the forward kernels), per-atom sums FP64; the r histograms are
// accumulated in FP32 in LDS per workgroup and flushed with FP64 atomics, so
// the gradient is reproducible to FP32 rounding of the per-workgroup partial
// sums, not bit for bit (in FP64 to FP64 rounding).
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "csr_rows.hpp"

struct tdmd_fm {
  int precision = TDMD_MIXED;
  int natoms = 0, nsnap = 0, ntot = 0;
  tdmd_box box{};
  double r_list = 0;
  int64_t npairs = 0;          // listed, ordered
  double r_min = 0;            // shortest listed pair (with the half list)
  double* d_pos = nullptr;     // [ntot][3]
  int32_t* d_cnt = nullptr;    // [ntot]
  int32_t* d_off = nullptr;    // [ntot]
  int32_t* d_hcnt = nullptr;   // [ntot] half list: neighbours j > i (fm_half_list)
  int32_t* d_hoff = nullptr;   // [ntot]
  int32_t* d_hnbr = nullptr;   // [npairs / 2]
  int32_t* d_nbr = nullptr;    // [total]
  int32_t* d_types = nullptr;  // [ntot], all 1
  double* d_target = nullptr;  // [ntot][3]
  double* d_rec = nullptr;     // [ntot] FmRec, what the adjoint passes gather
  void* d_force = nullptr;     // [ntot][3] in R
  double* d_rho = nullptr;     // [ntot]
  void* d_fp = nullptr;        // [ntot] in R
  double* d_partials = nullptr;
  int nparts = 0;
  int ncu = 0, lds_max = 0;  // compute units, LDS bytes of a workgroup
  double* d_scalars = nullptr;  // [8]
  bool has_target = false;
  // EAM scratch
  tdmd_eam_tables* tables = nullptr;  // geometry + quads rewritten per call
  double* d_gcoef = nullptr;          // [4 niF + 8 niR]
  int nrho = 0, nr = 0;
  double drho = 0, dr = 0, cutoff = 0;
};

namespace tdmd_hip {

namespace {

// Slots a lane takes at a time; us at 1, 2, 4 (55M ordered pairs, FP32 pair
// functions): the lambda pass 422, 373, 338; phi's FP64 histograms 233, 202,
// 219; rho's 238, 226, 258. Bound by their 48- and 64-byte gathers from L2.
constexpr int kLambdaSlots = 4;
constexpr int kHistSlots = 2;
constexpr int kFmBlock = 1024;  // workgroup of the histogram passes
constexpr int kFmGrid = 2048;   // workgroups (and partials) of the Morse pass, at most

// What the adjoint passes gather of an atom, 64 bytes: half a cache line; the
// lambda and phi passes want the first 48 (three 16-byte loads).
struct alignas(64) FmRec {
  double x, y, z;     // position
  double gx, gy, gz;  // residual F - T
  double fp, mu;      // F'(rho); lam, then mu
};

template <class R>
__device__ __forceinline__ R fm_exp(R x);
template <>
__device__ __forceinline__ float fm_exp<float>(float x) {
  return expf(x);
}
template <>
__device__ __forceinline__ double fm_exp<double>(double x) {
  return exp(x);
}

// ---------------------------------------------------------------------------
// Morse: forces, residual, loss and dL/d(D, alpha, r0) in one sweep of the
// rows: dL/dtheta = 2 g_i . sum_j d_ij dfpair/dtheta, so the three vectors are
// summed beside the force and meet g_i at the row's end.
// partials[blk * 4 + {0: L, 1: dD, 2: dalpha, 3: dr0}]
// ---------------------------------------------------------------------------
template <class R, bool kTarget>
__global__ void __launch_bounds__(kBlock)
k_fm_morse(const double* __restrict__ pos, const int32_t* __restrict__ nbr,
           const int32_t* __restrict__ off, const int32_t* __restrict__ cnt, int ntot, PairBox box,
           MorseCoef p, const double* __restrict__ target, double* __restrict__ forces_out,
           double* __restrict__ partials) {
  double l = 0.0, gD = 0.0, ga = 0.0, gr = 0.0;
  const R D = static_cast<R>(p.D), al = static_cast<R>(p.alpha);
  for_atoms<false>(ntot, [&](int i) {
    const Neighbour a = neighbour_at(pos, i);
    double fx = 0.0, fy = 0.0, fz = 0.0;
    double vD[3] = {0.0, 0.0, 0.0}, va[3] = {0.0, 0.0, 0.0}, vr[3] = {0.0, 0.0, 0.0};
    auto load = [&](int j) { return neighbour_at(pos, j); };
    for_row<kMorseSlots>(nbr, off[i], cnt[i], a.x, a.y, a.z, box, load,
                         [&](int, const Neighbour&, double dx, double dy, double dz, double r2) {
      if (r2 < p.rc_sq) {
        const PairR<R> pr = pair_r<R>(r2);
        R en;
        const double fpair = static_cast<double>(morse_fpair<R>(p, pr, &en));
        fx = fma(fpair, dx, fx);
        fy = fma(fpair, dy, fy);
        fz = fma(fpair, dz, fz);
        if (kTarget) {
          const R x = static_cast<R>(pr.r - p.r0);
          const R e = fm_exp<R>(-al * x);
          const R one = static_cast<R>(1), two = static_cast<R>(2);
          const R ome = one - e, o2e = one - two * e;
          const double dfdD = static_cast<double>(-two * al * ome * e * pr.rinv);
          const double dfda = static_cast<double>(-two * D * e * (ome - al * o2e * x) * pr.rinv);
          const double dfdr = static_cast<double>(-two * D * al * al * o2e * e * pr.rinv);
          const double d[3] = {dx, dy, dz};
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            vD[c] = fma(dfdD, d[c], vD[c]);
            va[c] = fma(dfda, d[c], va[c]);
            vr[c] = fma(dfdr, d[c], vr[c]);
          }
        }
      }
    });
    // forces as the product path stores them (R)
    const double F[3] = {static_cast<double>(static_cast<R>(row_sum(fx))),
                         static_cast<double>(static_cast<R>(row_sum(fy))),
                         static_cast<double>(static_cast<R>(row_sum(fz)))};
    const bool first = threadIdx.x % kRowLanes == 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const size_t at = 3 * static_cast<size_t>(i) + c;
      if (forces_out && first) forces_out[at] = F[c];
      if (kTarget) {
        const double g = F[c] - target[at];
        if (first) l += g * g;
        gD = fma(2.0 * g, vD[c], gD);
        ga = fma(2.0 * g, va[c], ga);
        gr = fma(2.0 * g, vr[c], gr);
      }
    }
  });
  if (!kTarget) return;
  const double s0 = block_sum<kBlock>(l);
  const double s1 = block_sum<kBlock>(gD);
  const double s2 = block_sum<kBlock>(ga);
  const double s3 = block_sum<kBlock>(gr);
  if (threadIdx.x == 0) {
    partials[4 * blockIdx.x] = s0;
    partials[4 * blockIdx.x + 1] = s1;
    partials[4 * blockIdx.x + 2] = s2;
    partials[4 * blockIdx.x + 3] = s3;
  }
}

// Fixed-order sum of `ncomp` interleaved partial streams, one per workgroup.
__global__ void k_fm_reduce(const double* __restrict__ partials, int nblk, int ncomp,
                            double* __restrict__ out) {
  __shared__ double s[256];
  const int c = blockIdx.x;
  double t = 0.0;
  for (int b = threadIdx.x; b < nblk; b += 256) t += partials[b * ncomp + c];
  s[threadIdx.x] = t;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (static_cast<int>(threadIdx.x) < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[c] = s[0];
}

// ---------------------------------------------------------------------------
// EAM
// ---------------------------------------------------------------------------

// FD-Hermite coefficients from knot values (build_fd_hermite on the device,
// same operation order, no contraction): spline s = 0 F, 1 rho, 2 phi; quads:
// F, rho, phi intervals in a row. Clears the coefficient gradients (blocks
// [spline][4][ni]) for an adjoint that follows; null: they stay.
template <class R>
__global__ void k_fm_build_coeffs(const double* __restrict__ vals, int nrho, double drho, int nr,
                                  double dr, double* __restrict__ gcoef,
                                  typename Quad<R>::type* __restrict__ quads) {
#pragma clang fp contract(off)
  const int s = blockIdx.y;
  const int n = s == 0 ? nrho : nr;
  const double h = s == 0 ? drho : dr;
  const double* v = vals + (s == 0 ? 0 : (s == 1 ? nrho : nrho + nr));
  const int ni = n - 1;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ni) return;
  const double slope_left = (i > 0) ? (v[i] - v[i - 1]) / h : 0.0;
  const double slope_right = (v[i + 1] - v[i]) / h;
  const double slope_next = (i + 2 < n) ? (v[i + 2] - v[i + 1]) / h : slope_right;
  double m0 = (slope_left + slope_right) * 0.5;
  double m1 = (slope_right + slope_next) * 0.5;
  if (i == 0) m0 = slope_right;
  if (i == n - 2) m1 = slope_right;
  const double a = v[i], b = m0, c = (3.0 * slope_right - 2.0 * m0 - m1) / h,
               d = (m0 + m1 - 2.0 * slope_right) / (h * h);
  const int niF = nrho - 1, niR = nr - 1;
  const size_t base = s == 0 ? 0 : (s == 1 ? 4 * static_cast<size_t>(niF)
                                           : 4 * static_cast<size_t>(niF) + 4 * niR);
  if (gcoef)
    for (int k = 0; k < 4; ++k) gcoef[base + static_cast<size_t>(k) * ni + i] = 0.0;
  const int qo = s == 0 ? 0 : (s == 1 ? niF : niF + niR);
  typename Quad<R>::type q;
  q.x = static_cast<R>(a);
  q.y = static_cast<R>(b);
  q.z = static_cast<R>(c);
  q.w = static_cast<R>(d);
  quads[qo + i] = q;
}

// Residual g = F - T (F as stored, in R), loss partials (one per block).
template <class R>
__global__ void __launch_bounds__(kBlock)
k_fm_residual(const R* __restrict__ f, const R* __restrict__ fp, const double* __restrict__ target,
              int ntot, FmRec* __restrict__ rec, double* __restrict__ forces_out,
              double* __restrict__ partials, int has_target) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  double l = 0.0;
  if (i < ntot) {
    double g[3] = {0.0, 0.0, 0.0};
    for (int c = 0; c < 3; ++c) {
      const size_t at = 3 * static_cast<size_t>(i) + c;
      const double F = static_cast<double>(f[at]);
      if (forces_out) forces_out[at] = F;
      if (has_target) {
        g[c] = F - target[at];
        l += g[c] * g[c];
      }
    }
    rec[i].fp = static_cast<double>(fp[i]);
    rec[i].gx = g[0];
    rec[i].gy = g[1];
    rec[i].gz = g[2];
  }
  const double s = block_sum<kBlock>(l);
  if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// w_ij = -2 (g_i - g_j) . d_ij / r_ij
__device__ __forceinline__ double fm_weight(const FmRec& a, const FmRec& b, double dx, double dy,
                                            double dz, double r) {
  return -2.0 * ((a.gx - b.gx) * dx + (a.gy - b.gy) * dy + (a.gz - b.gz) * dz) / r;
}

// lam_i = sum_j w_ij rho'(r_ij) over full rows, left in rec[i].mu.
template <class R>
__global__ void __launch_bounds__(kBlock)
k_fm_eam_lambda(FmRec* rec, const int32_t* __restrict__ nbr, const int32_t* __restrict__ off,
                const int32_t* __restrict__ cnt, int ntot, PairBox box, EamLayout t,
                const typename Quad<R>::type* __restrict__ quads) {
  for_atoms<false>(ntot, [&](int i) {
    FmRec a = rec[i];
    double lam = 0.0;
    auto load = [&](int j) {
      FmRec b;  // all but fp and mu, which other workgroups write
      const FmRec* p = rec + j;
      b.x = p->x;
      b.y = p->y;
      b.z = p->z;
      b.gx = p->gx;
      b.gy = p->gy;
      b.gz = p->gz;
      return b;
    };
    for_row<kLambdaSlots>(nbr, off[i], cnt[i], a.x, a.y, a.z, box, load,
                         [&](int, const FmRec& b, double dx, double dy, double dz, double r2) {
      if (r2 < t.rc_sq) {
        const PairR<R> pr = pair_r<R>(r2);
        R x;
        const int k = spline_locate<R>(t.r, pr.r, &x);
        const R drho = quad_deriv<R>(quads[t.rho_at(0) + k], x);
        lam = fma(fm_weight(a, b, dx, dy, dz, pr.r), static_cast<double>(drho), lam);
      }
    });
    lam = row_sum(lam);
    if (threadIdx.x % kRowLanes == 0) rec[i].mu = lam;
  });
}

// F coefficients at rho_i and mu_i = lam_i F''(rho_i) (rec[i].mu: lam to mu).
// The densities of a solid fall on a few hundred of F's intervals, so the
// three adds an atom go to an LDS histogram first where it fits (kLds).
template <class R, bool kLds>
__global__ void __launch_bounds__(kFmBlock)
k_fm_eam_embed(FmRec* __restrict__ rec, const double* __restrict__ rho, int ntot, EamLayout t,
               const typename Quad<R>::type* __restrict__ quads, double* __restrict__ gF) {
  extern __shared__ __align__(16) unsigned char fm_smem[];
  double* hist = reinterpret_cast<double*>(fm_smem);  // b, c, d
  const int ni = t.F.n - 1;
  if (kLds) {
    for (int q = threadIdx.x; q < 3 * ni; q += kFmBlock) hist[q] = 0.0;
    __syncthreads();
  }
  double* out = kLds ? hist : gF + ni;  // gF[0, ni): the a block, untouched
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kFmBlock + threadIdx.x; i < ntot;
       i += static_cast<int64_t>(gridDim.x) * kFmBlock) {
    const double lam = rec[i].mu;
    R x;
    const int k = spline_locate<R>(t.F, rho[i], &x);
    const double xd = static_cast<double>(x);
    atomicAdd(&out[k], lam);
    atomicAdd(&out[ni + k], 2.0 * xd * lam);
    atomicAdd(&out[2 * ni + k], 3.0 * xd * xd * lam);
    const auto c = quads[t.f_at(0) + k];
    rec[i].mu = lam * static_cast<double>(static_cast<R>(2) * c.z + static_cast<R>(6) * c.w * x);
  }
  if (kLds) {
    __syncthreads();
    for (int q = threadIdx.x; q < 3 * ni; q += kFmBlock)
      if (hist[q] != 0.0) atomicAdd(&gF[ni + q], hist[q]);
  }
}

// phi (b, c, d) and rho (a, b, c, d) coefficients over unordered pairs, the
// half list. kPhi / kRho: which of them this launch adds (both, or
// one each where seven histograms do not fit the LDS together). kLds: in
// LDS, intervals k_lo (that of the set's shortest pair) and up, flushed at
// the end; else straight to gcoef. Workgroups are persistent, each over a
// contiguous run of rows.
template <class R, bool kPhi, bool kRho, bool kLds>
__global__ void __launch_bounds__(kFmBlock)
k_fm_eam_hist(const FmRec* __restrict__ rec, const int32_t* __restrict__ nbr,
              const int32_t* __restrict__ off, const int32_t* __restrict__ cnt, int ntot,
              PairBox box, EamLayout t, int k_lo, double* __restrict__ gcoef) {
  extern __shared__ __align__(16) unsigned char fm_smem[];
  double* hist = reinterpret_cast<double*>(fm_smem);
  const int ni = t.r.n - 1, nw = ni - k_lo;
  constexpr int kN = (kPhi ? 3 : 0) + (kRho ? 4 : 0);
  constexpr int kRhoAt = kPhi ? 3 : 0;
  // gcoef after the F block: rho {a,b,c,d}, phi {a,b,c,d}
  double* g = gcoef + 4 * static_cast<size_t>(t.F.n - 1);
  auto home = [](int which) { return which < kRhoAt ? 5 + which : which - kRhoAt; };
  if (kLds) {
    for (int q = threadIdx.x; q < kN * nw; q += kFmBlock) hist[q] = 0.0;
    __syncthreads();
  }
  auto add = [&](int which, int k, double v) {
    if (kLds)
      atomicAdd(&hist[which * nw + (k - k_lo)], v);
    else
      atomicAdd(&g[static_cast<size_t>(home(which)) * ni + k], v);
  };
  constexpr int kTurn = kFmBlock / kRowLanes;
  const int64_t piece = piece_of(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
  const int64_t turns = (static_cast<int64_t>(ntot) + kTurn - 1) / kTurn;
  const int64_t t1 = turns * (piece + 1) / gridDim.x;
  for (int64_t tt = turns * piece / gridDim.x; tt < t1; ++tt) {
    const int64_t ii = tt * kTurn + static_cast<int>(threadIdx.x) / kRowLanes;
    if (ii >= ntot) continue;
    const int i = static_cast<int>(ii);
    const FmRec a = rec[i];
    auto load = [&](int j) { return rec[j]; };
    for_row<kHistSlots>(nbr, off[i], cnt[i], a.x, a.y, a.z, box, load,
                         [&](int, const FmRec& b, double dx, double dy, double dz, double r2) {
      if (r2 < t.rc_sq) {
        const PairR<R> pr = pair_r<R>(r2);
        R x;
        const int k = spline_locate<R>(t.r, pr.r, &x);
        const double w = fm_weight(a, b, dx, dy, dz, pr.r);
        const double td = static_cast<double>(x);
        if (kPhi) {
          add(0, k, w);
          add(1, k, 2.0 * td * w);
          add(2, k, 3.0 * td * td * w);
        }
        if (kRho) {
          const double m = a.mu + b.mu;
          const double wp =
              w * static_cast<double>(static_cast<R>(a.fp) + static_cast<R>(b.fp));
          add(kRhoAt, k, m);
          add(kRhoAt + 1, k, wp + m * td);
          add(kRhoAt + 2, k, td * (2.0 * wp + m * td));
          add(kRhoAt + 3, k, td * td * (3.0 * wp + m * td));
        }
      }
    });
  }
  if (kLds) {
    __syncthreads();
    for (int which = 0; which < kN; ++which)
      for (int k = threadIdx.x; k < nw; k += kFmBlock) {
        const double v = hist[which * nw + k];
        if (v != 0.0) atomicAdd(&g[static_cast<size_t>(home(which)) * ni + k_lo + k], v);
      }
  }
}

// Mixed precision where seven FP32 histograms fit the LDS: the whole adjoint
// in one pass over ordered pairs, one lane per atom. An FP32 sum of ~100 terms
// of either sign a bin carries a rounding error that its order decides
// (1.5e-6 of the gradient), and the adds bound this pass so evenly that two
// runs differ by less than half of that (0.6e-6): sums in another type or
// order would move the gradients of existing mixed fits by more than they
// move from run to run. ~200 cycles per ds_add_f32 of a wavefront, ten a pair,
// are all of its time (2865 us at 55M ordered pairs of 1M atoms, 5000 points;
// the FP64 passes take 800).
__global__ void __launch_bounds__(kFmBlock)
k_fm_eam_adjoint_f32(const FmRec* __restrict__ rec, const int32_t* __restrict__ nbr,
                     const int32_t* __restrict__ off, const int32_t* __restrict__ cnt, int ntot,
                     PairBox box, EamLayout tab, const float4* __restrict__ quads,
                     const double* __restrict__ rho, double* __restrict__ gcoef) {
  extern __shared__ __align__(16) unsigned char fm_smem[];
  float* hist = reinterpret_cast<float*>(fm_smem);  // phi b,c,d; rho a,b,c,d
  const int niF = tab.F.n - 1, niR = tab.r.n - 1;
  double* gF = gcoef;                                  // [4][niF]
  double* gRP = gcoef + 4 * static_cast<size_t>(niF);  // rho[4][niR], phi[4][niR]
  for (int q = threadIdx.x; q < 7 * niR; q += kFmBlock) hist[q] = 0.0f;
  __syncthreads();
  auto add = [&](int which, int k, double v) {
    atomicAdd(&hist[which * niR + k], static_cast<float>(v));
  };
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kFmBlock + threadIdx.x; i < ntot;
       i += static_cast<int64_t>(gridDim.x) * kFmBlock) {
    const FmRec a = rec[i];
    const int32_t* row = nbr + off[i];
    const int c = cnt[i];
    double lam = 0.0;
    for (int k = 0; k < c; ++k) {
      const FmRec b = rec[row[k]];
      const double dx = image(a.x - b.x, box.size[0], box.half[0]);
      const double dy = image(a.y - b.y, box.size[1], box.half[1]);
      const double dz = image(a.z - b.z, box.size[2], box.half[2]);
      const double r2 = dx * dx + dy * dy + dz * dz;
      if (r2 < tab.rc_sq) {
        const PairR<float> pr = pair_r<float>(r2);
        float t;
        const int q = spline_locate<float>(tab.r, pr.r, &t);
        const float drho = quad_deriv<float>(quads[tab.rho_at(0) + q], t);
        const double w = fm_weight(a, b, dx, dy, dz, pr.r);
        const double hw = 0.5 * w;  // the two orderings of the pair give w
        const double P = static_cast<double>(static_cast<float>(a.fp) + static_cast<float>(b.fp));
        const double td = static_cast<double>(t);
        add(0, q, hw);
        add(1, q, 2.0 * td * hw);
        add(2, q, 3.0 * td * td * hw);
        add(4, q, hw * P);
        add(5, q, 2.0 * td * hw * P);
        add(6, q, 3.0 * td * td * hw * P);
        lam = fma(w, static_cast<double>(drho), lam);
      }
    }
    float tF;
    const int qF = spline_locate<float>(tab.F, rho[i], &tF);
    const double tFd = static_cast<double>(tF);
    atomicAdd(&gF[niF + qF], lam);
    atomicAdd(&gF[2 * niF + qF], 2.0 * tFd * lam);
    atomicAdd(&gF[3 * niF + qF], 3.0 * tFd * tFd * lam);
    const float4 cF = quads[tab.f_at(0) + qF];
    const double mu = lam * static_cast<double>(2.0f * cF.z + 6.0f * cF.w * tF);
    for (int k = 0; k < c; ++k) {
      const FmRec* b = rec + row[k];
      const double dx = image(a.x - b->x, box.size[0], box.half[0]);
      const double dy = image(a.y - b->y, box.size[1], box.half[1]);
      const double dz = image(a.z - b->z, box.size[2], box.half[2]);
      const double r2 = dx * dx + dy * dy + dz * dz;
      if (r2 < tab.rc_sq) {
        float t;
        const int q = spline_locate<float>(tab.r, pair_r<float>(r2).r, &t);
        const double td = static_cast<double>(t);
        add(3, q, mu);
        add(4, q, mu * td);
        add(5, q, mu * td * td);
        add(6, q, mu * td * td * td);
      }
    }
  }
  __syncthreads();
  for (int q = threadIdx.x; q < 7 * niR; q += kFmBlock) {
    const float v = hist[q];
    if (v != 0.0f) {
      const int which = q / niR, k = q - which * niR;
      atomicAdd(&gRP[static_cast<size_t>(which < 3 ? 5 + which : which - 3) * niR + k],
                static_cast<double>(v));
    }
  }
}

// Transpose of the FD-Hermite map: the knot-value gradient from the
// coefficient gradients, through S[k], the gradient of interval k's slope.
__device__ __forceinline__ double fm_slope_grad(const double* __restrict__ gb,
                                                const double* __restrict__ gc,
                                                const double* __restrict__ gd, int k, int ni,
                                                double h) {
  auto gm0 = [&](int q) { return gb[q] - 2.0 * gc[q] / h + gd[q] / (h * h); };
  auto gm1 = [&](int q) { return -gc[q] / h + gd[q] / (h * h); };
  double v = 3.0 * gc[k] / h - 2.0 * gd[k] / (h * h);
  v += (k == 0) ? gm0(0) : 0.5 * gm0(k);
  if (k + 1 <= ni - 1) v += 0.5 * gm0(k + 1);
  v += (k == ni - 1) ? gm1(k) : 0.5 * gm1(k);
  if (k >= 1) v += 0.5 * gm1(k - 1);
  return v;
}

__global__ void k_fm_coef_grad(const double* __restrict__ gcoef, int nrho, double drho, int nr,
                               double dr, double* __restrict__ gv) {
  const int s = blockIdx.y;
  const int niF = nrho - 1, niR = nr - 1;
  const int n = s == 0 ? nrho : nr, ni = n - 1;
  const double h = s == 0 ? drho : dr;
  const double* ga = gcoef + (s == 0 ? 0 : (s == 1 ? 4 * static_cast<size_t>(niF)
                                                   : 4 * static_cast<size_t>(niF) + 4 * niR));
  const double *gb = ga + ni, *gc = ga + 2 * ni, *gd = ga + 3 * ni;
  double* out = gv + (s == 0 ? 0 : (s == 1 ? nrho : nrho + nr));
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= n) return;
  double v = 0.0;
  if (m <= ni - 1) v += ga[m] - fm_slope_grad(gb, gc, gd, m, ni, h) / h;
  if (m >= 1) v += fm_slope_grad(gb, gc, gd, m - 1, ni, h) / h;
  out[m] = v;
}

// Rows from the snapshots' local indices to global ones. One wavefront per row.
__global__ void __launch_bounds__(kBlock)
k_fm_rows(int32_t* __restrict__ nbr, const int32_t* __restrict__ off,
          const int32_t* __restrict__ cnt, int ntot, int natoms) {
  const int64_t row = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) >> 6;
  if (row >= ntot) return;
  const int i = static_cast<int>(row);
  const int shift = i / natoms * natoms;
  const int o = off[i], c = cnt[i];
  for (int q = threadIdx.x & 63; q < c; q += kWave) nbr[o + q] += shift;
}

// The half list's counts, and *r2_min: the shortest pair's r^2 (non-negative
// doubles order as their bits). One wavefront per row.
__global__ void __launch_bounds__(kBlock)
k_fm_half_counts(const int32_t* __restrict__ nbr, const int32_t* __restrict__ off,
                 const int32_t* __restrict__ cnt, int ntot, const double* __restrict__ pos,
                 PairBox box, int32_t* __restrict__ hcnt, unsigned long long* r2_min) {
  const int64_t row = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) >> 6;
  if (row >= ntot) return;
  const int lane = threadIdx.x & 63;
  const int i = static_cast<int>(row);
  const int o = off[i], c = cnt[i];
  const Neighbour a = neighbour_at(pos, i);
  int nh = 0;
  double r2 = __builtin_huge_val();
  for (int q = lane; q < c; q += kWave) {
    const int j = nbr[o + q];
    nh += j > i ? 1 : 0;
    const Neighbour b = neighbour_at(pos, j);
    const double dx = image(a.x - b.x, box.size[0], box.half[0]);
    const double dy = image(a.y - b.y, box.size[1], box.half[1]);
    const double dz = image(a.z - b.z, box.size[2], box.half[2]);
    r2 = fmin(r2, dx * dx + dy * dy + dz * dz);
  }
  for (int w = 32; w > 0; w >>= 1) {
    nh += __shfl_xor(nh, w, 64);
    r2 = fmin(r2, __shfl_xor(r2, w, 64));
  }
  if (lane == 0) {
    hcnt[i] = nh;
    const auto bits = static_cast<unsigned long long>(__double_as_longlong(r2));
    if (bits < __hip_atomic_load(r2_min, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMin(r2_min, bits);
  }
}

// The half list, each row's neighbours j > i in the row's order.
__global__ void __launch_bounds__(kBlock)
k_fm_half(const int32_t* __restrict__ nbr, const int32_t* __restrict__ off,
          const int32_t* __restrict__ cnt, int ntot, const int32_t* __restrict__ hoff,
          int32_t* __restrict__ hnbr) {
  const int64_t row = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) >> 6;
  if (row >= ntot) return;
  const int lane = threadIdx.x & 63;
  const int i = static_cast<int>(row);
  const int o = off[i], c = cnt[i];
  int at = hoff[i];
  for (int k = 0; k < c; k += kWave) {
    const int j = k + lane < c ? nbr[o + k + lane] : -1;
    const unsigned long long m = __ballot(j > i);
    if (j > i) hnbr[at + __popcll(m & ((1ull << lane) - 1ull))] = j;
    at += __popcll(m);
  }
}

__global__ void __launch_bounds__(kBlock)
k_fm_records(const double* __restrict__ pos, int ntot, FmRec* __restrict__ rec) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= ntot) return;
  rec[i] = FmRec{pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], 0.0, 0.0, 0.0, 0.0, 0.0};
}

int fm_free(tdmd_fm* F) {
  void* ptrs[] = {F->d_pos,  F->d_cnt, F->d_off, F->d_nbr, F->d_hcnt, F->d_hoff, F->d_hnbr, F->d_types,
                  F->d_target, F->d_rec, F->d_force, F->d_rho, F->d_fp, F->d_partials, F->d_scalars, F->d_gcoef};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  if (F->tables) eam_tables_destroy(F->tables);
  delete F;
  return TDMD_OK;
}

template <class T>
int fm_alloc(T** p, size_t n) {
  void* q = nullptr;
  const int rc = tdmd_malloc(&q, std::max<size_t>(n, 1) * sizeof(T));
  *p = static_cast<T*>(q);
  return rc;
}

// The half list and the shortest pair, for the passes over unordered pairs.
int fm_half_list(tdmd_fm* F, hipStream_t s) {
  if (F->d_hnbr) return TDMD_OK;
  const int N = F->ntot;
  int32_t *cnt = nullptr, *off = nullptr, *nbr = nullptr;
  char* work = nullptr;
  size_t sb = 0;
  double r2 = __builtin_huge_val();
  auto build = [&]() -> int {
    int rc = tdmd_scan_workspace_bytes(N, &sb);
    if (rc || (rc = fm_alloc(&cnt, N)) || (rc = fm_alloc(&off, N)) ||
        (rc = fm_alloc(&nbr, static_cast<size_t>(F->npairs / 2 + 1))) ||
        (rc = fm_alloc(&work, sb)))
      return rc;
    const int rows = grid_for(N, kBlock / kWave);
    TDMD_HIP_TRY(hipMemcpyAsync(F->d_scalars, &r2, sizeof(r2), hipMemcpyHostToDevice, s));
    k_fm_half_counts<<<rows, kBlock, 0, s>>>(F->d_nbr, F->d_off, F->d_cnt, N, F->d_pos,
                                             make_pair_box(make_devbox(F->box)), cnt,
                                             reinterpret_cast<unsigned long long*>(F->d_scalars));
    TDMD_LAUNCH_CHECK();
    if ((rc = tdmd_scan_exclusive_i32(cnt, off, N, nullptr, work, s))) return rc;
    k_fm_half<<<rows, kBlock, 0, s>>>(F->d_nbr, F->d_off, F->d_cnt, N, off, nbr);
    TDMD_LAUNCH_CHECK();
    TDMD_HIP_TRY(hipMemcpyAsync(&r2, F->d_scalars, sizeof(r2), hipMemcpyDeviceToHost, s));
    TDMD_HIP_TRY(hipStreamSynchronize(s));
    return TDMD_OK;
  };
  const int rc = build();
  if (rc) (void)hipStreamSynchronize(s);
  if (work) (void)hipFree(work);
  if (rc) {
    for (int32_t* p : {cnt, off, nbr})
      if (p) (void)hipFree(p);
    return rc;
  }
  F->r_min = r2 < F->r_list * F->r_list ? std::sqrt(r2) : 0.0;
  F->d_hcnt = cnt;
  F->d_hoff = off;
  F->d_hnbr = nbr;
  return TDMD_OK;
}

// The adjoint passes: coefficient gradients in F->d_gcoef (cleared before).
template <class R>
int fm_eam_adjoint(tdmd_fm* F, hipStream_t s) {
  const int N = F->ntot;
  const size_t niF = static_cast<size_t>(F->nrho - 1), niR = static_cast<size_t>(F->nr - 1);
  const size_t lmax = static_cast<size_t>(F->lds_max);
  const PairBox box = make_pair_box(make_devbox(F->box));
  const EamLayout t = eam_layout(F->tables);
  const auto* quads = static_cast<const typename Quad<R>::type*>(F->tables->d_coeff);
  auto* rec = reinterpret_cast<FmRec*>(F->d_rec);
  // Persistent workgroups of `lds` bytes: as many as the CUs hold (two of
  // 1024 threads at most), no more than there is work for.
  auto persistent = [&](size_t lds, int64_t threads) {
    const int64_t per_cu = 2 * lds <= lmax ? 2 : 1;
    return static_cast<int>(std::max<int64_t>(
        1, std::min<int64_t>(per_cu * F->ncu, (threads + kFmBlock - 1) / kFmBlock)));
  };
  // (the same limit for every handle: no call lowers another's)
  auto allow = [&](const void* kernel, size_t lds) -> int {
    if (lds <= 65536) return TDMD_OK;
    TDMD_HIP_TRY(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     F->lds_max));
    return TDMD_OK;
  };
  if constexpr (std::is_same_v<R, float>) {
    const size_t lds = 7 * niR * sizeof(float);
    if (lds + 1024 <= lmax) {
      if (const int r = allow(reinterpret_cast<const void*>(&k_fm_eam_adjoint_f32), lds)) return r;
      k_fm_eam_adjoint_f32<<<std::max(1, std::min(grid_for(N, kFmBlock), F->ncu)), kFmBlock, lds,
                             s>>>(rec, F->d_nbr, F->d_off, F->d_cnt, N, box, t, quads, F->d_rho,
                                  F->d_gcoef);
      TDMD_LAUNCH_CHECK();
      return TDMD_OK;
    }
  }
  int rc = fm_half_list(F, s);
  if (rc) return rc;
  k_fm_eam_lambda<R><<<row_grid(N, false), kBlock, 0, s>>>(rec, F->d_nbr, F->d_off, F->d_cnt, N,
                                                           box, t, quads);
  TDMD_LAUNCH_CHECK();
  const size_t lf = 3 * niF * sizeof(double);
  if (lf <= lmax) {
    if ((rc = allow(reinterpret_cast<const void*>(&k_fm_eam_embed<R, true>), lf))) return rc;
    k_fm_eam_embed<R, true><<<persistent(lf, N), kFmBlock, lf, s>>>(rec, F->d_rho, N, t, quads,
                                                                    F->d_gcoef);
  } else {
    k_fm_eam_embed<R, false><<<persistent(0, N), kFmBlock, 0, s>>>(rec, F->d_rho, N, t, quads,
                                                                   F->d_gcoef);
  }
  TDMD_LAUNCH_CHECK();
  // no pair of the set lies below interval k_lo (r is exact to rounding; one
  // interval of margin)
  const int k_lo = std::max(0, std::min(static_cast<int>(F->r_min / F->dr) - 1, F->nr - 2));
  const size_t nw = niR - static_cast<size_t>(k_lo);
  const int64_t threads = static_cast<int64_t>(N) * kRowLanes;
  auto hist = [&](auto* kernel, size_t lds) -> int {
    const int r = allow(reinterpret_cast<const void*>(kernel), lds);
    if (r) return r;
    kernel<<<persistent(lds, threads), kFmBlock, lds, s>>>(
        rec, F->d_hnbr, F->d_hoff, F->d_hcnt, N, box, t, k_lo, F->d_gcoef);
    TDMD_LAUNCH_CHECK();
    return TDMD_OK;
  };
  constexpr size_t d = sizeof(double);
  if (7 * nw * d <= lmax) return hist(&k_fm_eam_hist<R, true, true, true>, 7 * nw * d);
  if (4 * nw * d <= lmax) {  // phi's three histograms, then rho's four
    rc = hist(&k_fm_eam_hist<R, true, false, true>, 3 * nw * d);
    return rc ? rc : hist(&k_fm_eam_hist<R, false, true, true>, 4 * nw * d);
  }
  return hist(&k_fm_eam_hist<R, true, true, false>, 0);
}

}  // namespace
}  // namespace tdmd_hip

using namespace tdmd_hip;

extern "C" {

int tdmd_fm_create(tdmd_fm** out, int32_t precision, const tdmd_box* box, int32_t natoms,
                   int32_t nsnap, const double* pos, double r_cut) {
  if (!out || !box || !pos || natoms <= 0 || nsnap <= 0 || !(r_cut > 0))
    return fail(TDMD_E_INVALID, "fm_create: bad arguments");
  if (precision != TDMD_MIXED && precision != TDMD_FP64)
    return fail(TDMD_E_INVALID, "fm_create: bad precision");
  const int64_t ntot64 = static_cast<int64_t>(natoms) * nsnap;
  if (ntot64 > (1LL << 30)) return fail(TDMD_E_INVALID, "fm_create: too many atoms");
  auto* F = new tdmd_fm();
  F->precision = precision;
  F->natoms = natoms;
  F->nsnap = nsnap;
  F->ntot = static_cast<int>(ntot64);
  F->box = *box;
  F->r_list = r_cut;
  const int N = F->ntot;
  const size_t rsz = precision == TDMD_MIXED ? 4 : 8;
  int rc = 0;
  if ((rc = fm_alloc(&F->d_pos, 3 * static_cast<size_t>(N))) ||
      (rc = fm_alloc(&F->d_cnt, N)) || (rc = fm_alloc(&F->d_off, N)) ||
      (rc = fm_alloc(&F->d_types, N)) || (rc = fm_alloc(&F->d_target, 3 * static_cast<size_t>(N))) ||
      (rc = fm_alloc(reinterpret_cast<char**>(&F->d_force), 3 * rsz * N)) ||
      (rc = fm_alloc(&F->d_rho, N)) ||
      (rc = fm_alloc(reinterpret_cast<char**>(&F->d_fp), rsz * N)) ||
      (rc = fm_alloc(&F->d_scalars, 8))) {
    fm_free(F);
    return rc;
  }
  F->nparts = (N + kBlock - 1) / kBlock;
  if ((rc = fm_alloc(&F->d_partials, std::max(4 * static_cast<size_t>(kFmGrid),
                                              static_cast<size_t>(F->nparts))))) {
    fm_free(F);
    return rc;
  }
  hipError_t e = hipMemcpy(F->d_pos, pos, 3 * sizeof(double) * N, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    fm_free(F);
    return hip_fail(e, "hipMemcpy", __FILE__, __LINE__);
  }
  std::vector<int32_t> ones(static_cast<size_t>(N), 1);
  e = hipMemcpy(F->d_types, ones.data(), 4 * static_cast<size_t>(N), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    fm_free(F);
    return hip_fail(e, "hipMemcpy", __FILE__, __LINE__);
  }
  int dev = 0;
  e = hipGetDevice(&dev);
  if (e == hipSuccess)
    e = hipDeviceGetAttribute(&F->ncu, hipDeviceAttributeMultiprocessorCount, dev);
  if (e == hipSuccess)
    e = hipDeviceGetAttribute(&F->lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
  if (e != hipSuccess) {
    fm_free(F);
    return hip_fail(e, "hipDeviceGetAttribute", __FILE__, __LINE__);
  }
  // Per-snapshot full lists (cell build + count), one global scan, fill,
  // then all rows to their global form at once.
  int32_t ncells[3];
  double cs[3];
  if ((rc = tdmd_cell_grid(box, r_cut, ncells, cs))) {
    fm_free(F);
    return rc;
  }
  const int nc = ncells[0] * ncells[1] * ncells[2];
  size_t wb = 0, sb = 0;
  tdmd_cell_workspace_bytes(natoms, nc, &wb);
  tdmd_scan_workspace_bytes(N, &sb);
  const size_t S = static_cast<size_t>(nsnap);
  int32_t *cc = nullptr, *co = nullptr, *ca = nullptr, *ac = nullptr, *meta = nullptr;
  char *work = nullptr, *swork = nullptr;
  if (!(rc = fm_alloc(&cc, S * nc)) && !(rc = fm_alloc(&co, S * nc)) && !(rc = fm_alloc(&ca, N)) &&
      !(rc = fm_alloc(&ac, N)) && !(rc = fm_alloc(&meta, 4)) && !(rc = fm_alloc(&work, wb)))
    rc = fm_alloc(&swork, sb);
  auto cells = [&](int s, auto&& call) {  // call(positions, first atom, cells of snapshot s)
    const size_t a0 = static_cast<size_t>(s) * natoms, c0 = static_cast<size_t>(s) * nc;
    return call(F->d_pos + 3 * a0, a0, cc + c0, co + c0, ca + a0, ac + a0);
  };
  for (int s = 0; s < nsnap && !rc; ++s)
    rc = cells(s, [&](const double* ps, size_t a0, int32_t* c, int32_t* o, int32_t* a, int32_t* k) {
      const int r = tdmd_cell_build(ps, natoms, box, r_cut, c, o, a, k, work, nullptr);
      return r ? r
               : tdmd_nlist_count(ps, natoms, box, r_cut, c, o, a, k, ncells, F->d_cnt + a0,
                                  nullptr);
    });
  if (!rc) rc = tdmd_scan_exclusive_i32(F->d_cnt, F->d_off, N, meta, swork, nullptr);
  int32_t hm[2] = {0, 0};
  if (!rc) {
    e = hipMemcpy(hm, meta, 8, hipMemcpyDeviceToHost);
    if (e != hipSuccess) rc = hip_fail(e, "hipMemcpy", __FILE__, __LINE__);
  }
  F->npairs = hm[0];
  if (!rc && !(rc = fm_alloc(&F->d_nbr, static_cast<size_t>(std::max(hm[0], 1))))) {
    (void)hipMemset(meta + 2, 0, 4);  // overflow: cannot happen, the rows were counted
    for (int s = 0; s < nsnap && !rc; ++s)
      rc = cells(s, [&](const double* ps, size_t a0, int32_t* c, int32_t* o, int32_t* a, int32_t* k) {
        return tdmd_nlist_fill(ps, natoms, box, r_cut, c, o, a, k, ncells, F->d_off + a0, F->d_nbr,
                               F->d_cnt + a0, hm[1], meta + 2, nullptr);
      });
    if (!rc) {
      k_fm_rows<<<grid_for(N, kBlock / kWave), kBlock>>>(F->d_nbr, F->d_off, F->d_cnt, N, natoms);
      e = hipGetLastError();
      if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
      if (e != hipSuccess) rc = hip_fail(e, "fm_create rows", __FILE__, __LINE__);
    }
  }
  for (void* p : {static_cast<void*>(cc), static_cast<void*>(co), static_cast<void*>(ca),
                  static_cast<void*>(ac), static_cast<void*>(meta),
                  static_cast<void*>(work), static_cast<void*>(swork)})
    if (p) (void)hipFree(p);
  if (rc) {
    fm_free(F);
    return rc;
  }
  *out = F;
  return TDMD_OK;
}

int tdmd_fm_destroy(tdmd_fm* F) {
  if (!F) return TDMD_OK;
  (void)hipDeviceSynchronize();
  return fm_free(F);
}

int tdmd_fm_info(const tdmd_fm* F, int32_t* ntot, int64_t* npairs) {
  if (!F) return fail(TDMD_E_INVALID, "fm_info: null");
  if (ntot) *ntot = F->ntot;
  if (npairs) {
    int32_t last[2];
    TDMD_HIP_TRY(hipMemcpy(&last[0], F->d_off + F->ntot - 1, 4, hipMemcpyDeviceToHost));
    TDMD_HIP_TRY(hipMemcpy(&last[1], F->d_cnt + F->ntot - 1, 4, hipMemcpyDeviceToHost));
    *npairs = static_cast<int64_t>(last[0]) + last[1];
  }
  return TDMD_OK;
}

int tdmd_fm_set_targets(tdmd_fm* F, const double* forces) {
  if (!F || !forces) return fail(TDMD_E_INVALID, "fm_set_targets: null");
  TDMD_HIP_TRY(hipMemcpy(F->d_target, forces, 3 * sizeof(double) * F->ntot,
                         hipMemcpyHostToDevice));
  F->has_target = true;
  return TDMD_OK;
}

int tdmd_fm_morse(tdmd_fm* F, const double params[3], double rc, double* loss, double grad[3],
                  double* forces_out) {
  if (!F || !params || !(rc > 0)) return fail(TDMD_E_INVALID, "fm_morse: bad arguments");
  if (rc > F->r_list) return fail(TDMD_E_INVALID, "fm_morse: cutoff beyond the list cutoff");
  if ((loss || grad) && !F->has_target) return fail(TDMD_E_STATE, "fm_morse: no targets set");
  const int N = F->ntot;
  const PairBox box = make_pair_box(make_devbox(F->box));
  const MorseCoef p{params[0], params[1], params[2], rc * rc};
  double* d_fout = nullptr;
  if (forces_out) {
    const int rc2 = fm_alloc(&d_fout, 3 * static_cast<size_t>(N));
    if (rc2) return rc2;
  }
  const int nb = std::min(row_grid(N, false), kFmGrid);
  const bool want = F->has_target && (loss || grad);
  auto go = [&](auto kernel) {
    kernel<<<nb, kBlock>>>(F->d_pos, F->d_nbr, F->d_off, F->d_cnt, N, box, p, F->d_target, d_fout,
                           F->d_partials);
  };
  if (F->precision == TDMD_MIXED)
    want ? go(&k_fm_morse<float, true>) : go(&k_fm_morse<float, false>);
  else
    want ? go(&k_fm_morse<double, true>) : go(&k_fm_morse<double, false>);
  TDMD_LAUNCH_CHECK();
  if (want) {
    k_fm_reduce<<<4, 256>>>(F->d_partials, nb, 4, F->d_scalars);
    TDMD_LAUNCH_CHECK();
  }
  double h[4] = {0.0, 0.0, 0.0, 0.0};
  if (want) TDMD_HIP_TRY(hipMemcpy(h, F->d_scalars, sizeof(h), hipMemcpyDeviceToHost));
  if (loss) *loss = h[0];
  if (grad) {
    grad[0] = h[1];
    grad[1] = h[2];
    grad[2] = h[3];
  }
  if (forces_out) {
    TDMD_HIP_TRY(hipMemcpy(forces_out, d_fout, 3 * sizeof(double) * N, hipMemcpyDeviceToHost));
    TDMD_HIP_TRY(hipFree(d_fout));
  }
  return TDMD_OK;
}

int tdmd_fm_eam(tdmd_fm* F, int32_t nrho, double drho, int32_t nr, double dr, double cutoff,
                const double* d_values, double* d_loss, double* d_grad, double* d_forces,
                void* stream) {
  if (!F || !d_values || nrho < 3 || nr < 3 || !(drho > 0) || !(dr > 0) || !(cutoff > 0))
    return fail(TDMD_E_INVALID, "fm_eam: bad arguments");
  if (cutoff > F->r_list) return fail(TDMD_E_INVALID, "fm_eam: cutoff beyond the list cutoff");
  if ((d_loss || d_grad) && !F->has_target) return fail(TDMD_E_STATE, "fm_eam: no targets set");
  hipStream_t s = as_stream(stream);
  const int N = F->ntot;
  const int niF = nrho - 1, niR = nr - 1;
  if (!F->tables || F->nrho != nrho || F->nr != nr || F->drho != drho || F->dr != dr ||
      F->cutoff != cutoff) {
    if (F->tables) eam_tables_destroy(F->tables);
    F->tables = nullptr;
    if (F->d_gcoef) (void)hipFree(F->d_gcoef);
    F->d_gcoef = nullptr;
    SetflData sd;
    sd.ntypes = 1;
    sd.nrho = nrho;
    sd.nr = nr;
    sd.drho = drho;
    sd.dr = dr;
    sd.cutoff = cutoff;
    sd.phi_values = true;
    sd.F.assign(static_cast<size_t>(nrho), 0.0);
    sd.rho.assign(static_cast<size_t>(nr), 0.0);
    sd.rphi.assign(static_cast<size_t>(nr), 0.0);
    int rc = eam_tables_create(&F->tables, F->precision, sd);
    if (rc) return rc;
    const size_t ng = 4 * static_cast<size_t>(niF) + 8 * static_cast<size_t>(niR);
    if ((rc = fm_alloc(&F->d_gcoef, ng))) return rc;
    if ((rc = tdmd_fill_u32(F->d_gcoef, 0u, 2 * ng, stream))) return rc;
    F->nrho = nrho;
    F->nr = nr;
    F->drho = drho;
    F->dr = dr;
    F->cutoff = cutoff;
  }
  if (!F->d_rec) {
    const int rc = fm_alloc(&F->d_rec, 8 * static_cast<size_t>(N));
    if (rc) return rc;
    k_fm_records<<<grid_for(N), kBlock, 0, s>>>(F->d_pos, N, reinterpret_cast<FmRec*>(F->d_rec));
    TDMD_LAUNCH_CHECK();
  }
  const bool mixed = F->precision == TDMD_MIXED;
  // FD-Hermite coefficients from the knot values, and the kernels' quads
  const dim3 gc((std::max(niF, niR) + 255) / 256, 3);
  double* const clear = d_grad ? F->d_gcoef : nullptr;
  if (mixed)
    k_fm_build_coeffs<float><<<gc, 256, 0, s>>>(d_values, nrho, drho, nr, dr, clear,
                                                static_cast<float4*>(F->tables->d_coeff));
  else
    k_fm_build_coeffs<double><<<gc, 256, 0, s>>>(d_values, nrho, drho, nr, dr, clear,
                                                 static_cast<double4*>(F->tables->d_coeff));
  TDMD_LAUNCH_CHECK();
  // forward: density, embedding, forces (the drop-in EAM path)
  int rc = tdmd_eam_compute(F->tables, F->d_pos, F->d_force, F->d_types, F->d_nbr, F->d_off,
                            F->d_cnt, N, &F->box, F->d_rho, F->d_fp, nullptr, nullptr, stream);
  if (rc) return rc;
  const int nb = F->nparts;
  auto* rec = reinterpret_cast<FmRec*>(F->d_rec);
  if (mixed)
    k_fm_residual<float><<<nb, kBlock, 0, s>>>(
        static_cast<const float*>(F->d_force), static_cast<const float*>(F->d_fp), F->d_target, N,
        rec, d_forces, F->d_partials, F->has_target ? 1 : 0);
  else
    k_fm_residual<double><<<nb, kBlock, 0, s>>>(
        static_cast<const double*>(F->d_force), static_cast<const double*>(F->d_fp), F->d_target,
        N, rec, d_forces, F->d_partials, F->has_target ? 1 : 0);
  TDMD_LAUNCH_CHECK();
  if (d_loss) {
    k_fm_reduce<<<1, 256, 0, s>>>(F->d_partials, nb, 1, d_loss);
    TDMD_LAUNCH_CHECK();
  }
  if (d_grad) {
    rc = mixed ? fm_eam_adjoint<float>(F, s) : fm_eam_adjoint<double>(F, s);
    if (rc) return rc;
    const dim3 gv((std::max(nrho, nr) + 255) / 256, 3);
    k_fm_coef_grad<<<gv, 256, 0, s>>>(F->d_gcoef, nrho, drho, nr, dr, d_grad);
    TDMD_LAUNCH_CHECK();
  }
  TDMD_HIP_TRY(hipStreamSynchronize(s));
  return TDMD_OK;
}

int tdmd_fm_eam_coef_grad(const tdmd_fm* F, double* gcoef) {
  if (!F || !gcoef || !F->d_gcoef) return fail(TDMD_E_STATE, "fm_eam_coef_grad: no gradient yet");
  const size_t n = 4 * static_cast<size_t>(F->nrho - 1) + 8 * static_cast<size_t>(F->nr - 1);
  TDMD_HIP_TRY(hipMemcpy(gcoef, F->d_gcoef, n * sizeof(double), hipMemcpyDeviceToHost));
  return TDMD_OK;
}

}  // extern "C"
