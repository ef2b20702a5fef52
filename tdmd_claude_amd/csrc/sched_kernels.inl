// sched_kernels.inl -- kernels of the FastPipelineScheduler fast path
// (src/scheduler/fast_pipeline_scheduler.cu:87-232 re-designed for gfx950).
//
// Per NVE step (the reference's kick-drift / force pair,
// fast_pipeline_scheduler.cu:101-166):
//   [rebuild: bin, scan, scatter, order, permute, copy-back, list]
//   EAM density pass        M  -> M2 (rho, F'(rho) fused: reference passes
//                                 1+2, device_eam.cu:72-162)
//   force pass + epilogue   M2 -> F, then the cross-step kick and drift of
//                                 the next step in registers (the
//                                 reference's fused_full_kick_drift,
//                                 device_velocity_verlet.cu:88-130), which
//                                 writes the next M and tests the skin.
// The density pass reads M and writes M2; the force pass reads M2 and writes
// M, so no pass reads a record another thread of the same pass writes.
#pragma once

#include "nhc.hpp"
#include "sched_kernels.hpp"

namespace tdmd_hip {
namespace sched {

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------

__device__ __forceinline__ double wrap1(double x, double lo, double L, int periodic) {
  // device_velocity_verlet.cu:49-61
  if (periodic) {
    if (x < lo)
      x += L;
    else if (x >= lo + L)
      x -= L;
  }
  return x;
}

template <class Mir>
__device__ __forceinline__ typename Mir::T encode_type(const MirrorParams& mp, double x,
                                                       double y, double z, int ti) {
  return Mir::encode(mp, x, y, z, ti);
}

template <class R>
__device__ __forceinline__ R* rp(void* p) {
  return static_cast<R*>(p);
}

template <int BLOCK = kBlock>
__device__ __forceinline__ void emit_partial(double v, double* partials, int slot) {
  const double t = block_sum<BLOCK>(v);
  if (threadIdx.x == 0) partials[slot] = t;
}

// Kick-and-drift for atom i with a given kick factor and an optional pre
// scale of v (NHC). Writes x, v and the gather record (into `rec`: M, or the
// Morse pass's other record buffer); sets the rebuild flag when the atom has
// moved more than skin/2 since the last build (minimum image).
// Streaming accesses of the integrator (positions, velocities, forces, build
// positions, types): each element is touched once per step, so they are
// loaded and stored non-temporally and leave the caches (L2, and MALL in
// front of HBM) to the neighbour rows and gather records that both passes
// re-read every step (1M-atom NVT step 286.6 -> 280.0 us).
template <class T>
__device__ __forceinline__ T ntl(const T* p) {
  return __builtin_nontemporal_load(p);
}
template <class T>
__device__ __forceinline__ void nts(T v, T* p) {
  __builtin_nontemporal_store(v, p);
}

// kKick2: the stored v lacks the previous step's closing half kick (its
// force pass only summed the KE of the kicked velocity, epilogue kKe); it is
// applied here first, as v + (dt/2) F / (m mvv2e), the epilogue's expression.
template <class R, class Mir, bool kKick2 = false>
__device__ __forceinline__ void kick_drift(const StepArgs& a, int i, double vscale,
                                           double kick_dt, double f0, double f1, double f2,
                                           void* rec) {
  const int ti = a.one_type ? 0 : ntl(&a.types[i]) - 1;
  const double mass = a.masses[ti + 1];
  double ux = ntl(&a.vx[i]), uy = ntl(&a.vy[i]), uz = ntl(&a.vz[i]);
  if constexpr (kKick2) {
    const double half = (0.5 * a.dt) / (mass * kMvv2e);
    ux = __fma_rn(half, f0, ux);
    uy = __fma_rn(half, f1, uy);
    uz = __fma_rn(half, f2, uz);
  }
  // explicit fused operations: the same roundings whether the half kick
  // above was applied here or by the force pass (kick 2 stored)
  const double factor = kick_dt / (mass * kMvv2e);
  const double vx = __fma_rn(factor, f0, vscale * ux);
  const double vy = __fma_rn(factor, f1, vscale * uy);
  const double vz = __fma_rn(factor, f2, vscale * uz);
  const MirrorParams& mp = mp_of<Mir>(a, i);
  const double x = wrap1(ntl(&a.px[i]) + a.dt * vx, mp.lo[0], mp.L[0], mp.periodic[0]);
  const double y = wrap1(ntl(&a.py[i]) + a.dt * vy, mp.lo[1], mp.L[1], mp.periodic[1]);
  const double z = wrap1(ntl(&a.pz[i]) + a.dt * vz, mp.lo[2], mp.L[2], mp.periodic[2]);
  nts(vx, &a.vx[i]);
  nts(vy, &a.vy[i]);
  nts(vz, &a.vz[i]);
  nts(x, &a.px[i]);
  nts(y, &a.py[i]);
  nts(z, &a.pz[i]);
  const typename Mir::T m = encode_type<Mir>(mp, x, y, z, ti);
  static_cast<typename Mir::T*>(rec)[i] = m;
  double dx, dy, dz;
  if constexpr (Mir::kFixed) {
    // displacement since the build from the 32-bit coordinates: the
    // wrapping difference is the minimum image on a periodic axis
    dx = static_cast<double>(Mir::wdiff(m.x, ntl(&reinterpret_cast<const int32_t*>(a.bx)[i]))) * mp.unit[0];
    dy = static_cast<double>(Mir::wdiff(m.y, ntl(&reinterpret_cast<const int32_t*>(a.by)[i]))) * mp.unit[1];
    dz = static_cast<double>(Mir::wdiff(m.z, ntl(&reinterpret_cast<const int32_t*>(a.bz)[i]))) * mp.unit[2];
  } else {
    dx = min_image(x - a.bx[i], mp.L[0], mp.hL[0], mp.periodic[0]);
    dy = min_image(y - a.by[i], mp.L[1], mp.hL[1], mp.periodic[1]);
    dz = min_image(z - a.bz[i], mp.L[2], mp.hL[2], mp.periodic[2]);
  }
  if (dx * dx + dy * dy + dz * dz > a.skin_half_sq) a.flags[0] = 1;
  if (!(isfinite(x) && isfinite(y) && isfinite(z) && Mir::representable(mp, x, y, z)))
    a.flags[2] = 1;
}

// Force-pass epilogue. The full kick-drift writes the next step's records
// into `rec` (M for the EAM passes, which gather M2; the other buffer of the
// pair for the Morse pass, which gathers M).
template <class R, class Mir, int kEpi>
__device__ __forceinline__ double epilogue(const StepArgs& a, int i, double fx, double fy,
                                           double fz, void* rec = nullptr) {
  const R f0 = static_cast<R>(fx), f1 = static_cast<R>(fy), f2 = static_cast<R>(fz);
  if (kEpi == kFullKickDrift) {
    kick_drift<R, Mir>(a, i, 1.0, a.dt, static_cast<double>(f0), static_cast<double>(f1),
                       static_cast<double>(f2), rec ? rec : a.M);
    return 0.0;
  }
  nts(f0, &rp<R>(a.fx)[i]);
  nts(f1, &rp<R>(a.fy)[i]);
  nts(f2, &rp<R>(a.fz)[i]);
  if (kEpi == kForceOnly) return 0.0;
  // kHalfKick / kKick2Ke: v += (dt/2) F / (m mvv2e)  (half_kick_kernel,
  // device_velocity_verlet.cu:14-32)
  const int ti = a.one_type ? 0 : ntl(&a.types[i]) - 1;
  const double mass = a.masses[ti + 1];
  const double factor = (0.5 * a.dt) / (mass * kMvv2e);
  const double vx = __fma_rn(factor, static_cast<double>(f0), ntl(&a.vx[i]));
  const double vy = __fma_rn(factor, static_cast<double>(f1), ntl(&a.vy[i]));
  const double vz = __fma_rn(factor, static_cast<double>(f2), ntl(&a.vz[i]));
  if (kEpi != kKe) {
    nts(vx, &a.vx[i]);
    nts(vy, &a.vy[i]);
    nts(vz, &a.vz[i]);
  }
  if (emits_ke(kEpi)) return 0.5 * mass * kMvv2e * (vx * vx + vy * vy + vz * vz);
  return 0.0;
}

// ---------------------------------------------------------------------------
// integrate-only kernels
// ---------------------------------------------------------------------------

// Window bootstrap (fused_half_kick_drift) and the NVT first kick: kick by
// dt/2 with the stored forces, drift, write M. NVT scales v by the chain's
// pending factor first.
template <class R, class Mir, bool kNvt, bool kFull, bool kKick2 = false>
__global__ void __launch_bounds__(kBlock) k_kick_drift(StepArgs a) {
  const int i = xcd_block(a.nblocks) * kBlock + threadIdx.x;
  if (i >= a.natoms) return;
  const double s = kNvt ? a.nhc[26] : 1.0;
  kick_drift<R, Mir, kKick2>(a, i, s, kFull ? a.dt : 0.5 * a.dt,
                             static_cast<double>(ntl(&rp<R>(a.fx)[i])),
                             static_cast<double>(ntl(&rp<R>(a.fy)[i])),
                             static_cast<double>(ntl(&rp<R>(a.fz)[i])), a.M);
}

// Mirror refresh (after upload or restore): M[i] = {x, type}.
template <class Mir>
__global__ void __launch_bounds__(kBlock) k_write_mirror(StepArgs a) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.natoms) return;
  static_cast<typename Mir::T*>(a.M)[i] =
      encode_type<Mir>(mp_of<Mir>(a, i), a.px[i], a.py[i], a.pz[i], a.types[i] - 1);
}

template <class R>
__global__ void __launch_bounds__(kBlock) k_ke_partials(StepArgs a) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  double e = 0.0;
  if (i < a.natoms) {
    const double mass = a.masses[a.types[i]];
    e = 0.5 * mass * kMvv2e * (a.vx[i] * a.vx[i] + a.vy[i] * a.vy[i] + a.vz[i] * a.vz[i]);
  }
  emit_partial(e, a.partials, blockIdx.x);
}

static __global__ void k_scale_v(StepArgs a) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.natoms) return;
  const double s = a.nhc[24];
  a.vx[i] *= s;
  a.vy[i] *= s;
  a.vz[i] *= s;
}

// ---------------------------------------------------------------------------
// NHC chain (one thread; device_nose_hoover.cu:206-289 on device state)
//   nhc[0..7] eta, [8..15] eta_v, [16..23] eta_m, [24] vscale (pending
//   factor not yet applied to v), [25] KE of the stored v, [26] kick scale,
//   [27] reduced sum scratch
// ---------------------------------------------------------------------------

// Before the VV step: half-step on the KE of the actual velocities
// (vscale^2 * stored KE), kick scale = s1 * vscale.
static __global__ void k_nhc_pre(double* nhc, NhcParams p) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const double ke = nhc[24] * nhc[24] * nhc[25];
  const double s1 = nhc_half_step(p.M, nhc, nhc + 8, nhc + 16, p.t_target, p.t_period, p.dt,
                                  p.n_dof, ke);
  nhc[26] = s1 * nhc[24];
  nhc[24] = 1.0;
}

// After the VV step: KE from the per-block partials of the kick-2 epilogue,
// half-step, pending scale = s2. kPre: the next step's k_nhc_pre follows in
// the same thread (same operations, one launch less per step).
template <bool kPre>
__global__ void k_nhc_post(double* nhc, const double* partials, int n, NhcParams p) {
  __shared__ double s[256];
  double t = 0.0;
  for (int k = threadIdx.x; k < n; k += 256) t += partials[k];
  s[threadIdx.x] = t;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (static_cast<int>(threadIdx.x) < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double ke = s[0];
    const double s2 = nhc_half_step(p.M, nhc, nhc + 8, nhc + 16, p.t_target, p.t_period, p.dt,
                                    p.n_dof, ke);
    nhc[25] = ke;
    nhc[24] = s2;
    if (kPre) {
      const double ke1 = nhc[24] * nhc[24] * nhc[25];
      const double s1 = nhc_half_step(p.M, nhc, nhc + 8, nhc + 16, p.t_target, p.t_period, p.dt,
                                      p.n_dof, ke1);
      nhc[26] = s1 * nhc[24];
      nhc[24] = 1.0;
    }
  }
}

// Stored-KE refresh (after upload, or after the pending scale was applied).
static __global__ void k_nhc_set_ke(double* nhc, const double* partials, int n, int commit_scale) {
  __shared__ double s[256];
  double t = 0.0;
  for (int k = threadIdx.x; k < n; k += 256) t += partials[k];
  s[threadIdx.x] = t;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (static_cast<int>(threadIdx.x) < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    nhc[25] = s[0];
    if (commit_scale) nhc[24] = 1.0;
  }
}

// Window end: the pending factor has been applied to v by k_scale_v.
static __global__ void k_nhc_commit(double* nhc) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  nhc[25] *= nhc[24] * nhc[24];
  nhc[24] = 1.0;
}

// ---------------------------------------------------------------------------
// Neighbour loop shared by the force passes.
//
// Slots are visited in groups of kU. The indices of the next group are
// loaded while the current group's records are gathered and evaluated, so an
// index load (a coalesced 256-byte line per slot and wave, from HBM) overlaps
// a whole group of pair work instead of heading a dependent load chain. Rows
// are padded to a multiple of kRowPad slots with the atom itself, so group
// loads need no predicate; padded slots arrive with in_row = false.
// ---------------------------------------------------------------------------

constexpr int kRowPad = 8;  // rows padded to a multiple of this (cap too)
constexpr int kPairUnroll = 8;

// Slots k..k+kU-1 of atom i (k a multiple of 4): one 16-byte load per quad.
template <int kU>
__device__ __forceinline__ void load_slots(const StepArgs& a, int i, int k, int4 (&q)[kU / 4]) {
  const int4* __restrict__ q4 = reinterpret_cast<const int4*>(a.nbr);
#pragma unroll
  for (int h = 0; h < kU / 4; ++h) q[h] = q4[ell(i, k + 4 * h, a.cap) >> 2];
}

// Record j of a gather array, addressed as the array base plus an unsigned
// 32-bit byte offset (the host keeps natoms x record size below 4 GiB), so
// the index stays one 32-bit register instead of a sign-extended pair.
template <class T>
__device__ __forceinline__ T gather(const T* __restrict__ rec, int j) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(rec) +
                                     static_cast<uint32_t>(j) * static_cast<uint32_t>(sizeof(T)));
}

// The loop carries the next group's slots as the loaded quads and unpacks
// them at the top of the next iteration: registers the loads write are not
// copied before this group's pair work, so that work overlaps their latency
// (and the records' gathers) instead of waiting for them.
template <class T, int kU, class Pair>
__device__ __forceinline__ void for_neighbours(const StepArgs& a, int i, int n,
                                               const T* __restrict__ rec, Pair&& pair) {
  static_assert(kRowPad % kU == 0 && kU % 4 == 0, "groups must tile the padded row in quads");
  int4 q[kU / 4];
  if (n > 0) {
    load_slots<kU>(a, i, 0, q);
  } else {
#pragma unroll
    for (int h = 0; h < kU / 4; ++h) q[h] = make_int4(i, i, i, i);
  }
  for (int k = 0; k < n; k += kU) {
    int j[kU];
#pragma unroll
    for (int h = 0; h < kU / 4; ++h) {
      j[4 * h] = q[h].x;
      j[4 * h + 1] = q[h].y;
      j[4 * h + 2] = q[h].z;
      j[4 * h + 3] = q[h].w;
    }
    T mj[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) mj[u] = gather(rec, j[u]);
    if (k + kU < n) load_slots<kU>(a, i, k + kU, q);
#pragma unroll
    for (int u = 0; u < kU; ++u) pair(j[u], mj[u], k + u < n);
  }
}

// Packed 16-bit slots of one group: eight slots in a uint4, four in a uint2.
template <int kU>
struct Slots16;
template <>
struct Slots16<8> {
  using type = uint4;
};
template <>
struct Slots16<4> {
  using type = uint2;
};

// The packed slots k..k+kU-1 of atom i in 16-bit rows (k a multiple of kU).
template <int kU>
__device__ __forceinline__ typename Slots16<kU>::type load_local(const uint16_t* rows, int cap,
                                                                 int i, int k) {
  static_assert(kU == 4 || kU == 8, "four or eight slots per group");
  using P = typename Slots16<kU>::type;
  return reinterpret_cast<const P*>(rows)[ell16(i, k, cap) / kU];
}

__device__ __forceinline__ void unpack_local(const uint4& v, int (&ln)[8]) {
  const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    ln[2 * q] = static_cast<int>(w[q] & 0xffffu);
    ln[2 * q + 1] = static_cast<int>(w[q] >> 16);
  }
}
__device__ __forceinline__ void unpack_local(const uint2& v, int (&ln)[4]) {
  ln[0] = static_cast<int>(v.x & 0xffffu);
  ln[1] = static_cast<int>(v.x >> 16);
  ln[2] = static_cast<int>(v.y & 0xffffu);
  ln[3] = static_cast<int>(v.y >> 16);
}

// for_neighbours over a block whose halo records sit in LDS (`hrec`): the
// 16-bit rows index the halo, and the records come from LDS. The next
// group's slots stay packed until the top of the next iteration, so their
// load is waited for only after this group's pair work. pair(l, record,
// in_row, slot). kGuard: slots past n hold no valid index (read slot 0's
// record instead).
template <class T, int kU, bool kGuard = false, class Pair>
__device__ __forceinline__ void for_neighbours_staged(const StepArgs& a, const uint16_t* rows,
                                                      int i, int n, const T* hrec, Pair&& pair) {
  typename Slots16<kU>::type raw{};
  if (n > 0) raw = load_local<kU>(rows, a.cap, i, 0);
  for (int k = 0; k < n; k += kU) {
    int ln[kU];
    unpack_local(raw, ln);
    if (kGuard) {
#pragma unroll
      for (int u = 0; u < kU; ++u) ln[u] = k + u < n ? ln[u] : 0;
    }
    T mj[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) mj[u] = hrec[ln[u]];
    if (k + kU < n) raw = load_local<kU>(rows, a.cap, i, k + kU);
#pragma unroll
    for (int u = 0; u < kU; ++u) pair(ln[u], mj[u], k + u < n, k + u);
  }
}

// ---------------------------------------------------------------------------
// EAM passes (global tables; any number of elements)
// ---------------------------------------------------------------------------

__device__ __forceinline__ void load_meta(SplineMeta* sm, const SplineMeta* meta, int ns) {
  for (int k = threadIdx.x; k < ns; k += blockDim.x) sm[k] = meta[k];
  __syncthreads();
}

// A row split over kLanes neighbouring lanes (small systems, where one lane
// per atom leaves most of the chip idle): lane `part` takes quads part,
// part + kLanes, ... of the padded row; the four records of a quad are
// gathered before its pairs are evaluated.
template <class T, int kLanes, class Pair>
__device__ __forceinline__ void for_neighbours_split(const StepArgs& a, int i, int n, int part,
                                                     const T* __restrict__ rec, Pair&& pair) {
  const int4* __restrict__ q4 = reinterpret_cast<const int4*>(a.nbr);
  const int nq = (n + 3) >> 2;  // rows are padded to 8 slots: whole quads
  for (int q = part; q < nq; q += kLanes) {
    const int4 s = q4[ell(i, 4 * q, a.cap) >> 2];
    const T r0 = gather(rec, s.x), r1 = gather(rec, s.y), r2 = gather(rec, s.z),
            r3 = gather(rec, s.w);
    const int k = 4 * q;
    pair(s.x, r0, k < n);
    pair(s.y, r1, k + 1 < n);
    pair(s.z, r2, k + 2 < n);
    pair(s.w, r3, k + 3 < n);
  }
}

// for_neighbours_split for few wavefronts (kFew passes: one a SIMD, with nothing
// to hide a load or a chain of arithmetic behind). The next quad's
// records and the slots of the one after are loaded before a quad's pairs are
// evaluated (past the row's end the last quad again), and pairs go side by side,
// kB at a time: batch(records[kB], in_row[kB]) takes all distances, then all
// table loads, then the sums in slot order. A branch around each pair would put
// its load after the one before it.
template <class R>
constexpr int kFewBatch = sizeof(R) == 4 ? 4 : 2;

template <class T, int kLanes, int kB, class Batch>
__device__ __forceinline__ void for_neighbours_few(const StepArgs& a, int i, int n, int part,
                                                   const T* __restrict__ rec, Batch&& batch) {
  static_assert(4 % kB == 0, "batches tile a quad");
  const int4* __restrict__ q4 = reinterpret_cast<const int4*>(a.nbr);
  const int nq = (n + 3) >> 2;
  if (part >= nq) return;
  auto slots = [&](int q) { return q4[ell(i, 4 * min(q, nq - 1), a.cap) >> 2]; };
  const int4 s = slots(part);
  int4 s1 = slots(part + kLanes);
  T r[4] = {gather(rec, s.x), gather(rec, s.y), gather(rec, s.z), gather(rec, s.w)};
  for (int q = part; q < nq; q += kLanes) {
    const T r1[4] = {gather(rec, s1.x), gather(rec, s1.y), gather(rec, s1.z), gather(rec, s1.w)};
    s1 = slots(q + 2 * kLanes);
#pragma unroll
    for (int u = 0; u < 4; u += kB) {
      T bm[kB];
      bool br[kB];
#pragma unroll
      for (int v = 0; v < kB; ++v) {
        bm[v] = r[u + v];
        br[v] = 4 * q + u + v < n;
      }
      batch(bm, br);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) r[u] = r1[u];
  }
}

// Sum over the kLanes lanes of one atom (butterfly; every lane ends with
// the same bits, so the order is fixed).
template <int kLanes>
__device__ __forceinline__ double lane_sum(double v) {
#pragma unroll
  for (int w = kLanes / 2; w > 0; w >>= 1) v += __shfl_xor(v, w, 64);
  return v;
}

// Global-table EAM passes (several elements, or systems small enough that
// one workgroup per 1024 atoms would leave most CUs idle). kLanes > 1: the
// row of atom i is split over kLanes neighbouring lanes (quads p, p + kLanes,
// ... to lane p) and the lanes' partial sums are combined by a butterfly in
// a fixed order, so the result is run-to-run identical; the grid is kLanes
// times the one-lane grid and emits one energy / KE partial per 256 threads.
template <class R, class Mir, bool kEnergy, int kLanes, bool kFew = false>
__global__ void __launch_bounds__(kBlock)
k_eam_density(StepArgs a, const SplineMeta* __restrict__ meta,
              const typename Quad<R>::type* __restrict__ coeff, double rc_sq) {
  static_assert(kLanes >= 1 && 64 % kLanes == 0, "an atom's lanes share a wavefront");
  using T = typename Mir::T;
  pass_clock_begin(a.pclock);
  __shared__ SplineMeta sm[kMaxSplines];
  load_meta(sm, meta, 2 * a.ntypes);
  const int blk = xcd_block(gridDim.x);
  const int g = blk * kBlock + threadIdx.x;
  const int i = g / kLanes;
  const int part = g % kLanes;
  const T* __restrict__ M = static_cast<const T*>(a.M);
  double e = 0.0, rho = 0.0;
  T mi{};
  if (i < a.natoms) {
    mi = M[i];
    const MirrorParams& mpi = mp_of<Mir>(a, i);
    const int n = a.cnt[i];
    auto pair = [&](int, const T& mj, bool in_row) {
      double dx, dy, dz;
      const double r2 = Mir::delta(mi, mj, mpi, &dx, &dy, &dz);
      if (in_row && r2 < rc_sq) {
        const SplineMeta& m = sm[a.ntypes + Mir::type_of(mj)];
        if constexpr (std::is_same_v<R, float>) {
          float t;
          const auto c = coeff[m.offset + locate_f32(meta_f32(m), r2, &t)];
          rho += static_cast<double>(c.x + t * (c.y + t * (c.z + t * c.w)));
        } else {
          rho += spline_value<R>(m, coeff, pair_r<R>(r2).r);
        }
      }
    };
    if constexpr (kFew) {
      constexpr int kB = kFewBatch<R>;
      for_neighbours_few<T, kLanes, kB>(
          a, i, n, part, M, [&](const T (&mj)[kB], const bool (&in_row)[kB]) {
            double r2[kB];
            bool ok[kB], any = false;
#pragma unroll
            for (int u = 0; u < kB; ++u) {
              double dx, dy, dz;
              r2[u] = Mir::delta(mi, mj[u], mpi, &dx, &dy, &dz);
              ok[u] = in_row[u] && r2[u] < rc_sq;
              r2[u] = ok[u] ? r2[u] : 0.25 * rc_sq;  // any place in the table
              any = any || ok[u];
            }
            if (!any) return;
            typename Quad<R>::type c[kB];
            R t[kB];
#pragma unroll
            for (int u = 0; u < kB; ++u) {
              const SplineMeta& m = sm[a.ntypes + Mir::type_of(mj[u])];
              int idx;
              if constexpr (std::is_same_v<R, float>)
                idx = locate_f32(meta_f32(m), r2[u], &t[u]);
              else
                idx = spline_locate<R>(m, pair_r<R>(r2[u]).r, &t[u]);
              c[u] = coeff[m.offset + idx];
            }
#pragma unroll
            for (int u = 0; u < kB; ++u) {
              const R v = c[u].x + t[u] * (c[u].y + t[u] * (c[u].z + t[u] * c[u].w));
              rho = ok[u] ? rho + static_cast<double>(v) : rho;
            }
          });
    } else if constexpr (kLanes == 1) {
      for_neighbours<T, kPairUnroll>(a, i, n, M, pair);
    } else {
      for_neighbours_split<T, kLanes>(a, i, n, part, M, pair);
    }
  }
  if constexpr (kLanes > 1) rho = lane_sum<kLanes>(rho);  // every lane takes part
  if (i < a.natoms && part == 0) {
    const int ti = Mir::type_of(mi);
    const SplineVal<R> F = spline_both<R>(sm[ti], coeff, rho);
    // two to kPackedTypes elements: the force pass reads a neighbour's
    // element from F'(rho)'s two lowest mantissa bits
    const bool typed = a.ntypes > 1 && a.ntypes <= kPackedTypes;
    static_cast<T*>(a.M2)[i] = Mir::with_w(mi, typed ? Mir::template pack_typed<R>(F.df, ti)
                                                     : Mir::template pack_real<R>(F.df));
    e = static_cast<double>(F.f);
  }
  if (kEnergy) emit_partial(e, a.partials, blk);
  pass_clock_end(a.pclock);
}

template <class R, class Mir, int kEpi, bool kEnergy, bool kMulti, int kLanes, bool kFew = false>
__global__ void __launch_bounds__(kBlock)
k_eam_force(StepArgs a, const SplineMeta* __restrict__ meta,
            const typename Quad<R>::type* __restrict__ coeff, double rc_sq) {
  static_assert(kLanes >= 1 && 64 % kLanes == 0, "an atom's lanes share a wavefront");
  using T = typename Mir::T;
  unsigned long long* const pclk = a.pclock ? a.pclock + 4 : nullptr;
  pass_clock_begin(pclk);
  __shared__ SplineMeta sm[kMaxSplines];
  const int nt = a.ntypes;
  load_meta(sm, meta, 2 * nt + nt * (nt + 1) / 2);
  const int blk = xcd_block(gridDim.x);
  const int g = blk * kBlock + threadIdx.x;
  const int i = g / kLanes;
  const int part = g % kLanes;
  const T* __restrict__ M2 = static_cast<const T*>(a.M2);
  using Q = typename Quad<R>::type;
  constexpr bool kF32 = std::is_same_v<R, float>;
  double red = 0.0, vir = 0.0, fx = 0.0, fy = 0.0, fz = 0.0, pe = 0.0;
  if (i < a.natoms) {
    const T mi = M2[i];
    const MirrorParams& mpi = mp_of<Mir>(a, i);
    const R fpi = Mir::template w_real<R>(mi);
    const int ti = kMulti ? a.types[i] - 1 : 0;
    const int n = a.cnt[i];
    const ForceLocF floc = force_loc_f32(sm[nt]);  // every r spline's grid
    auto pair = [&](int j, const T& mj, bool in_row) {
      double dx, dy, dz;
      const double r2 = Mir::delta(mi, mj, mpi, &dx, &dy, &dz);
      if (in_row && r2 < rc_sq) {
        const int tj = kMulti ? (a.ntypes <= kPackedTypes ? Mir::packed_type(mj) : a.types[j] - 1)
                              : 0;
        const int pidx = kMulti ? phi_index(ti, tj, nt) : 0;
        R dphi, drho_j, drho_i, rinv;
        if constexpr (kF32) {
          // mixed: pair_t_f32's interval and offset, derivatives from b,
          // 2c, 3d (the pair table holds 2c and 3d)
          const PairT p = pair_t_f32(floc, r2);
          rinv = p.rinv;
          if (kMulti && !kEnergy && a.pairtab) {
            const Q* e = static_cast<const Q*>(a.pairtab) +
                         (static_cast<size_t>(ti * nt + tj) * a.pair_nint + p.idx) * 3;
            const Q q0 = e[0], q1 = e[1], q2 = e[2];
            dphi = cubic_deriv_s(q0.x, q0.y, q0.z, p.t);
            drho_j = cubic_deriv_s(q0.w, q1.x, q1.y, p.t);
            drho_i = cubic_deriv_s(q1.z, q1.w, q2.x, p.t);
          } else {
            const Q cphi = coeff[sm[2 * nt + pidx].offset + p.idx];
            if (kEnergy)
              pe += 0.5 * static_cast<double>(
                              cphi.x + p.t * (cphi.y + p.t * (cphi.z + p.t * cphi.w)));
            dphi = cubic_deriv_f(cphi, p.t);
            drho_j = cubic_deriv_f(coeff[sm[nt + tj].offset + p.idx], p.t);
            drho_i = kMulti ? cubic_deriv_f(coeff[sm[nt + ti].offset + p.idx], p.t) : drho_j;
          }
        } else {
          const PairR<R> pr = pair_r<R>(r2);
          rinv = pr.rinv;
          if (kMulti && !kEnergy && a.pairtab) {
            // one interval (the three splines share the r grid), three
            // adjacent quads; the same expressions as spline_deriv
            R dx;
            const int idx = spline_locate<R>(sm[2 * nt + pidx], pr.r, &dx);
            const Q* e = static_cast<const Q*>(a.pairtab) +
                         (static_cast<size_t>(ti * nt + tj) * a.pair_nint + idx) * 3;
            const Q q0 = e[0], q1 = e[1], q2 = e[2];
            dphi = q0.x + dx * (static_cast<R>(2) * q0.y + dx * static_cast<R>(3) * q0.z);
            drho_j = q0.w + dx * (static_cast<R>(2) * q1.x + dx * static_cast<R>(3) * q1.y);
            drho_i = q1.z + dx * (static_cast<R>(2) * q1.w + dx * static_cast<R>(3) * q2.x);
          } else {
            if (kEnergy) {
              const SplineVal<R> ph = spline_both<R>(sm[2 * nt + pidx], coeff, pr.r);
              pe += 0.5 * static_cast<double>(ph.f);
              dphi = ph.df;
            } else {
              dphi = spline_deriv<R>(sm[2 * nt + pidx], coeff, pr.r);
            }
            drho_j = spline_deriv<R>(sm[nt + tj], coeff, pr.r);
            drho_i = kMulti ? spline_deriv<R>(sm[nt + ti], coeff, pr.r) : drho_j;
          }
        }
        const R fpj = Mir::template w_real<R>(mj);
        const double fpair = static_cast<double>(-(dphi + fpi * drho_j + fpj * drho_i) * rinv);
        if (kEnergy) vir += 0.5 * fpair * r2;
        fx = fma(fpair, dx, fx);
        fy = fma(fpair, dy, fy);
        fz = fma(fpair, dz, fz);
      }
    };
    if constexpr (kFew) {
      static_assert(!kMulti && !kEnergy, "one element, forces only");
      constexpr int kB = kFewBatch<R>;
      for_neighbours_few<T, kLanes, kB>(
          a, i, n, part, M2, [&](const T (&mj)[kB], const bool (&in_row)[kB]) {
            double dx[kB], dy[kB], dz[kB], r2[kB];
            bool ok[kB], any = false;
#pragma unroll
            for (int u = 0; u < kB; ++u) {
              r2[u] = Mir::delta(mi, mj[u], mpi, &dx[u], &dy[u], &dz[u]);
              ok[u] = in_row[u] && r2[u] < rc_sq;
              r2[u] = ok[u] ? r2[u] : 0.25 * rc_sq;
              any = any || ok[u];
            }
            if (!any) return;
            Q cphi[kB], crho[kB];
            R t[kB], trho[kB], rinv[kB];
#pragma unroll
            for (int u = 0; u < kB; ++u) {
              int kphi, krho;
              if constexpr (kF32) {
                const PairT p = pair_t_f32(floc, r2[u]);
                rinv[u] = p.rinv;
                t[u] = trho[u] = p.t;
                kphi = krho = p.idx;
              } else {
                const PairR<R> pr = pair_r<R>(r2[u]);
                rinv[u] = pr.rinv;
                kphi = spline_locate<R>(sm[2 * nt], pr.r, &t[u]);
                krho = spline_locate<R>(sm[nt], pr.r, &trho[u]);
              }
              cphi[u] = coeff[sm[2 * nt].offset + kphi];
              crho[u] = coeff[sm[nt].offset + krho];
            }
#pragma unroll
            for (int u = 0; u < kB; ++u) {
              auto deriv = [](const Q& c, R x) {
                if constexpr (kF32)
                  return cubic_deriv_f(c, x);
                else  // the same expression as spline_deriv
                  return c.y + x * (static_cast<R>(2) * c.z + x * static_cast<R>(3) * c.w);
              };
              const R drho = deriv(crho[u], trho[u]);
              const R fpj = Mir::template w_real<R>(mj[u]);
              const double fpair = static_cast<double>(
                  -(deriv(cphi[u], t[u]) + fpi * drho + fpj * drho) * rinv[u]);
              fx = ok[u] ? fma(fpair, dx[u], fx) : fx;
              fy = ok[u] ? fma(fpair, dy[u], fy) : fy;
              fz = ok[u] ? fma(fpair, dz[u], fz) : fz;
            }
          });
    } else if constexpr (kLanes == 1) {
      for_neighbours<T, kPairUnroll>(a, i, n, M2, pair);
    } else {
      for_neighbours_split<T, kLanes>(a, i, n, part, M2, pair);
    }
  }
  if constexpr (kLanes > 1) {  // every lane takes part in the shuffles
    fx = lane_sum<kLanes>(fx);
    fy = lane_sum<kLanes>(fy);
    fz = lane_sum<kLanes>(fz);
    if (kEnergy) {
      pe = lane_sum<kLanes>(pe);
      vir = lane_sum<kLanes>(vir);
    }
  }
  if (i < a.natoms && part == 0) {
    const double ke = epilogue<R, Mir, kEpi>(a, i, fx, fy, fz);
    red = kEnergy ? pe : ke;
  } else {
    vir = 0.0;
  }
  if (kEnergy || emits_ke(kEpi)) emit_partial(red, a.partials, blk);
  if (kEnergy) emit_partial(vir, a.partials_w, blk);
  pass_clock_end(pclk);
}

// ---------------------------------------------------------------------------
// Morse pass (morse.hpp:37-55; pair_math.hpp precision contract)
// ---------------------------------------------------------------------------

template <class R, class Mir, int kEpi, bool kEnergy, int kLanes, bool kFew = false>
__global__ void __launch_bounds__(kBlock) k_morse_force(StepArgs a, MorseCoef p) {
  // The pass gathers from M; with the fused kick-drift the next step's
  // records go to M2 and the host swaps the two buffers after the launch.
  // kLanes > 1: kLanes lanes per atom, the grid kLanes times larger.
  static_assert(kLanes >= 1 && 64 % kLanes == 0, "an atom's lanes share a wavefront");
  using T = typename Mir::T;
  unsigned long long* const pclk = a.pclock ? a.pclock + 4 : nullptr;
  pass_clock_begin(pclk);
  const int blk = xcd_block(gridDim.x);
  const int g = blk * kBlock + threadIdx.x;
  const int i = g / kLanes;
  const int part = g % kLanes;
  const T* __restrict__ M = static_cast<const T*>(a.M);
  double red = 0.0, fx = 0.0, fy = 0.0, fz = 0.0, pe = 0.0, vir = 0.0;
  if (i < a.natoms) {
    const T mi = M[i];
    const MirrorParams& mpi = mp_of<Mir>(a, i);
    const int n = a.cnt[i];
    auto pair = [&](int, const T& mj, bool in_row) {
      double dx, dy, dz;
      const double r2 = Mir::delta(mi, mj, mpi, &dx, &dy, &dz);
      if (in_row && r2 < p.rc_sq) {
        const PairR<R> pr = pair_r<R>(r2);
        R e;
        const double fpair = static_cast<double>(morse_fpair<R>(p, pr, &e));
        if (kEnergy) {
          pe += 0.5 * static_cast<double>(e);
          vir += 0.5 * fpair * r2;
        }
        fx = fma(fpair, dx, fx);
        fy = fma(fpair, dy, fy);
        fz = fma(fpair, dz, fz);
      }
    };
    if constexpr (kFew) {
      constexpr int kB = kFewBatch<R>;
      for_neighbours_few<T, kLanes, kB>(
          a, i, n, part, M, [&](const T (&mj)[kB], const bool (&in_row)[kB]) {
            double dx[kB], dy[kB], dz[kB], r2[kB];
            bool ok[kB], any = false;
#pragma unroll
            for (int u = 0; u < kB; ++u) {
              r2[u] = Mir::delta(mi, mj[u], mpi, &dx[u], &dy[u], &dz[u]);
              ok[u] = in_row[u] && r2[u] < p.rc_sq;
              r2[u] = ok[u] ? r2[u] : p.rc_sq;
              any = any || ok[u];
            }
            if (!any) return;
#pragma unroll
            for (int u = 0; u < kB; ++u) {
              R e;
              const double fpair =
                  static_cast<double>(morse_fpair<R>(p, pair_r<R>(r2[u]), &e));
              fx = ok[u] ? fma(fpair, dx[u], fx) : fx;
              fy = ok[u] ? fma(fpair, dy[u], fy) : fy;
              fz = ok[u] ? fma(fpair, dz[u], fz) : fz;
            }
          });
    } else if constexpr (kLanes == 1) {
      for_neighbours<T, kPairUnroll>(a, i, n, M, pair);
    } else {
      for_neighbours_split<T, kLanes>(a, i, n, part, M, pair);
    }
  }
  if constexpr (kLanes > 1) {  // every lane takes part in the shuffles
    fx = lane_sum<kLanes>(fx);
    fy = lane_sum<kLanes>(fy);
    fz = lane_sum<kLanes>(fz);
    if (kEnergy) {
      pe = lane_sum<kLanes>(pe);
      vir = lane_sum<kLanes>(vir);
    }
  }
  if (i < a.natoms && part == 0) {
    const double ke = epilogue<R, Mir, kEpi>(a, i, fx, fy, fz, a.M2);
    red = kEnergy ? pe : ke;
  } else {
    vir = 0.0;
  }
  if (kEnergy || emits_ke(kEpi)) emit_partial(red, a.partials, blk);
  if (kEnergy) emit_partial(vir, a.partials_w, blk);
  pass_clock_end(pclk);
}

// ---------------------------------------------------------------------------
// Rebuild: spatial sort and the ELL neighbour list. Every kernel first reads
// the rebuild flag and returns when it is clear, so the whole sequence can
// sit in a captured graph and only does work on steps that need it.
// ---------------------------------------------------------------------------

static __global__ void k_set_flag(int32_t* flags) {
  if (threadIdx.x == 0 && blockIdx.x == 0) flags[0] = 1;
}

static __global__ void __launch_bounds__(kBlock) k_zero_cells(const int32_t* flags, GridArgs g) {
  if (!flags[0]) return;
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r >= g.ncells) return;
  g.ccount[r] = 0;
  g.cursor[r] = 0;
}

// Binning grid of atom i's box; global cell id = off + (c2 n1 + c1) n0 + c0.
struct CellGrid {
  int n[3];
  double inv_cs[3];
  double lo[3];
  int off;
};

template <class Mir>
__device__ __forceinline__ CellGrid grid_of(const StepArgs& a, const GridArgs& g, int i) {
  CellGrid cg;
  if constexpr (Mir::kMB) {
    const BoxGeo& b = a.boxes[a.rep[i]];
    for (int d = 0; d < 3; ++d) {
      cg.n[d] = b.n[d];
      cg.inv_cs[d] = b.inv_cs[d];
      cg.lo[d] = b.mp.lo[d];
    }
    cg.off = b.cell_off;
  } else {
    for (int d = 0; d < 3; ++d) {
      cg.n[d] = g.n[d];
      cg.inv_cs[d] = g.inv_cs[d];
      cg.lo[d] = a.mp.lo[d];
    }
    cg.off = 0;
  }
  return cg;
}

__device__ __forceinline__ void cell_coords(const CellGrid& cg, double x, double y, double z,
                                            int c[3]) {
  const double p[3] = {x, y, z};
  for (int d = 0; d < 3; ++d) {
    int v = static_cast<int>((p[d] - cg.lo[d]) * cg.inv_cs[d]);
    v = v >= cg.n[d] ? cg.n[d] - 1 : v;
    c[d] = v < 0 ? 0 : v;
  }
}

// ---- per-item bodies, shared by the separate kernels (first build) and
// the fused rebuild kernel ----

template <class Mir>
__device__ __forceinline__ void bin_atom(const StepArgs& a, const GridArgs& g, int i) {
  int c[3];
  const CellGrid cg = grid_of<Mir>(a, g, i);
  cell_coords(cg, a.px[i], a.py[i], a.pz[i], c);
  const int rank = g.rank_of[cg.off + (c[2] * cg.n[1] + c[1]) * cg.n[0] + c[0]];
  g.key[i] = rank;
  (void)wave_add_one(g.ccount, rank);
}

// Exclusive scan of the cell counts by one workgroup of BLOCK threads
// (atomics-free): thread t owns a contiguous chunk of cells, sums it, the
// workgroup scans the chunk sums, and each thread writes its chunk's starts;
// out[ncells] = N.
template <int BLOCK>
__device__ __forceinline__ void scan_cells(const GridArgs& g, int32_t* out) {
  __shared__ int wsum[BLOCK / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int chunk = (g.ncells + BLOCK - 1) / BLOCK;
  const int c0 = min(static_cast<int>(threadIdx.x) * chunk, g.ncells);
  const int c1 = min(c0 + chunk, g.ncells);
  int v = 0;
  for (int c = c0; c < c1; ++c) v += g.ccount[c];
  int incl = v;
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off, 64);
    if (lane >= off) incl += o;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  int base = incl - v;
  for (int k = 0; k < w; ++k) base += wsum[k];
  for (int c = c0; c < c1; ++c) {
    out[c] = base;
    base += g.ccount[c];
  }
  if (threadIdx.x == BLOCK - 1) out[g.ncells] = base;
}

// (The order of a cell's atoms after the scatter is the atomics' order;
// the ordering pass then sorts each cell by upload index.)
__device__ __forceinline__ void scatter_atom(const GridArgs& g, int i, const int32_t* cstart) {
  const int r = g.key[i];
  g.sidx[cstart[r] + wave_add_one(g.cursor, r)] = i;
}

// Inclusive scan of v over the workgroup (BLOCK threads); *total gets the
// workgroup's sum. Uses `ws` (BLOCK / 64 ints of LDS); ends synchronised.
template <int BLOCK>
__device__ __forceinline__ int block_scan_incl(int v, int* total, int* ws) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int incl = v;
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off, 64);
    if (lane >= off) incl += o;
  }
  if (lane == 63) ws[w] = incl;
  __syncthreads();
  int before = 0, sum = 0;
  for (int k = 0; k < BLOCK / 64; ++k) {
    const int x = ws[k];
    before += k < w ? x : 0;
    sum += x;
  }
  __syncthreads();  // ws is reused by the next call
  *total = sum;
  return before + incl;
}

// The exclusive cell scan by the whole grid of the fused rebuild, in two
// phases with a grid barrier between them: workgroup w owns a contiguous
// chunk of cells; phase 1 sums its chunk into wsum[w]; phase 2 adds the sums
// of the chunks before it and scans its chunk. The same starts as
// scan_cells, which one workgroup computes alone.
template <int BLOCK>
__device__ __forceinline__ void scan_cells_grid(const GridArgs& g, int phase) {
  __shared__ int ws[BLOCK / 64];
  const int W = gridDim.x;
  const int chunk = (g.ncells + W - 1) / W;
  const int c0 = min(static_cast<int>(blockIdx.x) * chunk, g.ncells);
  const int c1 = min(c0 + chunk, g.ncells);
  int total = 0;
  if (phase == 1) {
    int v = 0;
    for (int c = c0 + threadIdx.x; c < c1; c += BLOCK) v += g.ccount[c];
    (void)block_scan_incl<BLOCK>(v, &total, ws);
    if (threadIdx.x == 0) g.wsum[blockIdx.x] = total;
    return;
  }
  int v = 0;
  for (int k = threadIdx.x; k < static_cast<int>(blockIdx.x); k += BLOCK) v += g.wsum[k];
  (void)block_scan_incl<BLOCK>(v, &total, ws);
  int run = total;  // cells before this chunk
  for (int c = c0; c < c1; c += BLOCK) {
    const int cc = c + threadIdx.x;
    const int n = cc < c1 ? g.ccount[cc] : 0;
    const int incl = block_scan_incl<BLOCK>(n, &total, ws);
    if (cc < c1) g.cstart[cc] = run + incl - n;
    run += total;
  }
  if (c1 == g.ncells && c0 < c1 && threadIdx.x == 0) g.cstart[g.ncells] = run;
}

// Deterministic order inside a cell, by upload index: one wavefront, 64 of the
// cell's atoms at a time; a lane counts the atoms with a smaller index than its
// own (indices are unique, so the counts are the sorted positions), and
// put(old index, new slot) is called for each atom. (Cells of more than 64 atoms
// used to be sorted by one lane: half or more of a rebuild from 74 atoms a cell.)
template <class Put>
__device__ __forceinline__ void order_cell_wave(const GridArgs& g, int r, Put&& put) {
  const int lane = static_cast<int>(threadIdx.x & 63);
  const int start = __builtin_amdgcn_readfirstlane(g.cstart[r]);
  const int n = __builtin_amdgcn_readfirstlane(g.cstart[r + 1]) - start;
  const int32_t* const seg = g.sidx + start;
  for (int b = 0; b < n; b += 64) {
    const int32_t v = b + lane < n ? seg[b + lane] : 0;
    const int32_t kv = b + lane < n ? g.orig[v] : 0x7fffffff;
    int pos = 0;
    for (int c = 0; c < n; c += 64) {
      const int32_t kc = c == b ? kv : c + lane < n ? g.orig[seg[c + lane]] : 0x7fffffff;
      const int e = min(64, n - c);
      for (int m = 0; m < e; ++m) pos += __builtin_amdgcn_readlane(kc, m) < kv ? 1 : 0;
    }
    if (b + lane < n) put(v, start + pos);
  }
}

// The same by a lane per atom of the scatter's order: for cells of few atoms,
// where a wavefront per cell leaves most lanes idle.
template <class Put>
__device__ __forceinline__ void order_slot(const GridArgs& g, int s, Put&& put) {
  const int v = g.sidx[s];
  const int kv = g.orig[v], r = g.key[v];
  const int start = g.cstart[r], end = g.cstart[r + 1];
  int pos = start;
  for (int c = start; c < end; ++c) pos += g.orig[g.sidx[c]] < kv ? 1 : 0;
  put(v, pos);
}

// Atom o (old slot) to slot s of the scratch arrays, and its gather record.
template <class R, class Mir>
__device__ __forceinline__ void permute_atom(const StepArgs& a, const GridArgs& g,
                                             const PermArgs& t, int o, int s) {
  const double x = a.px[o], y = a.py[o], z = a.pz[o];
  const int32_t ty = a.types[o];
  t.px[s] = x;
  t.py[s] = y;
  t.pz[s] = z;
  t.vx[s] = a.vx[o];
  t.vy[s] = a.vy[o];
  t.vz[s] = a.vz[o];
  rp<R>(t.fx)[s] = rp<R>(a.fx)[o];
  rp<R>(t.fy)[s] = rp<R>(a.fy)[o];
  rp<R>(t.fz)[s] = rp<R>(a.fz)[o];
  t.types[s] = ty;
  t.orig[s] = g.orig[o];
  static_cast<typename Mir::T*>(a.M)[s] = Mir::encode(mp_of<Mir>(a, s), x, y, z, ty - 1);
}

template <class R, class Mir>
__device__ __forceinline__ void copyback_atom(const StepArgs& a, const GridArgs& g,
                                              const PermArgs& t, int s) {
  const double x = t.px[s], y = t.py[s], z = t.pz[s];
  a.px[s] = x;
  a.py[s] = y;
  a.pz[s] = z;
  if constexpr (Mir::kFixed) {
    const MirrorParams& mp = mp_of<Mir>(a, s);
    reinterpret_cast<int32_t*>(a.bx)[s] = Mir::enc1(x, mp.lo[0], mp.q[0]);
    reinterpret_cast<int32_t*>(a.by)[s] = Mir::enc1(y, mp.lo[1], mp.q[1]);
    reinterpret_cast<int32_t*>(a.bz)[s] = Mir::enc1(z, mp.lo[2], mp.q[2]);
  } else {
    a.bx[s] = x;
    a.by[s] = y;
    a.bz[s] = z;
  }
  a.vx[s] = t.vx[s];
  a.vy[s] = t.vy[s];
  a.vz[s] = t.vz[s];
  rp<R>(a.fx)[s] = rp<R>(t.fx)[s];
  rp<R>(a.fy)[s] = rp<R>(t.fy)[s];
  rp<R>(a.fz)[s] = rp<R>(t.fz)[s];
  const_cast<int32_t*>(a.types)[s] = t.types[s];
  g.orig[s] = t.orig[s];
}

// Candidate prefilter of the list search with the 32-bit fixed-point
// records (MirrorFixed): r^2 in FP32 from the records' wrapping differences.
// The records round each coordinate to one unit (at most L / 2^32, or
// W / 2^30 on an open axis; cells are at most 1024 per axis, so a unit is
// below 1e-6 of r_list) and FP32 adds ~1e-6 relative, so a candidate whose
// FP32 r^2 lies outside [1 - kPreMargin, 1 + kPreMargin] times a bound is on
// the same side of it as its exact FP64 r^2. Inside that band (a few
// candidates per million atoms) the exact test decides.
constexpr double kPreMargin = 1e-5;

// When the three axes share one unit u (cubic boxes), r^2 is formed in
// units^2 and the bounds are divided by u^2 instead: three products fewer
// per candidate, the same relative error.
struct PreBounds {
  float lo_list, hi_list, lo_near, hi_near;
  float ux, uy, uz;
  bool iso;
};

__device__ __forceinline__ PreBounds pre_bounds(const MirrorParams& mp, double r_list_sq,
                                                double near_sq) {
  PreBounds b;
  b.iso = mp.unit[0] == mp.unit[1] && mp.unit[1] == mp.unit[2];
  const double s = b.iso ? 1.0 / (mp.unit[0] * mp.unit[0]) : 1.0;
  b.lo_list = static_cast<float>(r_list_sq * s * (1.0 - kPreMargin));
  b.hi_list = static_cast<float>(r_list_sq * s * (1.0 + kPreMargin));
  b.lo_near = static_cast<float>(near_sq * s * (1.0 - kPreMargin));
  b.hi_near = static_cast<float>(near_sq * s * (1.0 + kPreMargin));
  b.ux = static_cast<float>(mp.unit[0]);
  b.uy = static_cast<float>(mp.unit[1]);
  b.uz = static_cast<float>(mp.unit[2]);
  return b;
}

template <bool kIsoU>
__device__ __forceinline__ float pre_r2(const int4& mj, const int4& mi, const PreBounds& b) {
  float dx = static_cast<float>(MirrorFixed::wdiff(mj.x, mi.x));
  float dy = static_cast<float>(MirrorFixed::wdiff(mj.y, mi.y));
  float dz = static_cast<float>(MirrorFixed::wdiff(mj.z, mi.z));
  if constexpr (!kIsoU) {
    dx *= b.ux;
    dy *= b.uy;
    dz *= b.uz;
  }
  return dx * dx + dy * dy + dz * dz;
}

// The list search. ELL rows over the sorted atoms, whose positions are read
// from the sort's scratch arrays (the state's own are being written back
// beside the search). Inclusion exactly as the CPU list
// (neighbor_list.cpp:58-62): d = x_j - x_i in FP64, single minimum image,
// unfused r2 < r_list^2. kCount: only count.
//
// Each row is partitioned: neighbours inside the interaction cutoff at build
// time first, the skin shell (rc <= r < r_list) after them. Atoms move less
// than half the skin between builds, so in the force passes the in-cutoff
// test is true for the leading slots and false for the trailing ones in
// nearly every lane of a wave, and whole waves skip the pair work of the
// shell. Candidates are taken cell by cell in increasing rank, so both parts
// come out in increasing atom index. A row over the capacity keeps its first
// `cap` hits, and its true count is reported.
//
// nlist_atom_group: 32 lanes per atom, two atoms per wavefront, straight from
// memory: for sparse systems (GridArgs::list_lanes) and what nlist_cells leaves
// (below). Lane t < 27 of a group loads stencil entry t's cell range and image,
// shared by shuffles; each cell's candidates are then tested 32 at a time, and a
// hit's place in the row is its rank among the hits in candidate order (ballot,
// then a prefix count): near entries go to the front and shell entries to the
// back, from the row's end down; after a workgroup-scope fence (this wave's row
// stores complete before it reads them back) the shell block is moved behind the
// near block, in increasing index, and the row padded. Every lane of the wave
// runs the loop (the ballots and shuffles need them); `act` is false for a half
// with no atom, whose i is any valid atom.
template <bool kCount, class Mir>
__device__ __forceinline__ int nlist_atom_group(const StepArgs& a, const GridArgs& g,
                                                const PermArgs& p, int i,
                                                bool act, double r_list_sq, double near_sq,
                                                int32_t* nbr, int32_t* cnt) {
  const int lane = static_cast<int>(threadIdx.x & 63);
  const int l = lane & 31, sh = lane & 32;
  const uint32_t lt = (1u << l) - 1u;
  const int cap = a.cap;
  const double xi = p.px[i], yi = p.py[i], zi = p.pz[i];
  const MirrorParams& mp = mp_of<Mir>(a, i);
  const CellGrid cg = grid_of<Mir>(a, g, i);
  int c[3];
  cell_coords(cg, xi, yi, zi, c);
  const size_t row =
      27 * static_cast<size_t>(g.rank_of[cg.off + (c[2] * cg.n[1] + c[1]) * cg.n[0] + c[0]]);
  bool images;
  if constexpr (Mir::kMB)
    images = a.boxes[a.rep[i]].images != 0;
  else
    images = g.images != 0;
  int my_start = 0, my_end = 0, my_img = 0;
  if (act && l < 27) {
    const int r = g.around[row + l];
    my_start = g.cstart[r];
    my_end = g.cstart[r + 1];
    my_img = g.around_img[row + l];
  }
  int4 mi_rec = make_int4(0, 0, 0, 0);
  PreBounds pb{};
  if constexpr (Mir::kFixed) {
    mi_rec = static_cast<const int4*>(a.M)[i];
    pb = pre_bounds(mp, r_list_sq, near_sq);
  }
  int count = 0, nn = 0, nf = 0;
  for (int t = 0; t < 27; ++t) {
    const int start = __shfl(my_start, sh + t);
    const int end = __shfl(my_end, sh + t);
    const int img = __shfl(my_img, sh + t);
    const bool ix = images && (img & 3) != 0;
    const bool iy = images && ((img >> 2) & 3) != 0;
    const bool iz = images && ((img >> 4) & 3) != 0;
    const double sx = (img & 3) == 1 ? mp.L[0] : -mp.L[0];
    const double sy = ((img >> 2) & 3) == 1 ? mp.L[1] : -mp.L[1];
    const double sz = ((img >> 4) & 3) == 1 ? mp.L[2] : -mp.L[2];
    for (int j0 = start; __any(j0 < end); j0 += 32) {
      const int j = j0 + l;
      const bool valid = j < end;
      const int jj = valid ? j : i;
      auto exact_r2 = [&]() {
        double ddx, ddy, ddz;
        if constexpr (Mir::kFixed) {
          ddx = p.px[jj] - xi;
          ddy = p.py[jj] - yi;
          ddz = p.pz[jj] - zi;
        } else {  // an FP64 record holds the position itself
          const typename Mir::T m = static_cast<const typename Mir::T*>(a.M)[jj];
          ddx = m.x - xi;
          ddy = m.y - yi;
          ddz = m.z - zi;
        }
        if (images) {
          ddx = ix ? ddx + sx : ddx;
          ddy = iy ? ddy + sy : ddy;
          ddz = iz ? ddz + sz : ddz;
        } else {
          ddx = min_image(ddx, mp.L[0], mp.hL[0], mp.periodic[0]);
          ddy = min_image(ddy, mp.L[1], mp.hL[1], mp.periodic[1]);
          ddz = min_image(ddz, mp.L[2], mp.hL[2], mp.periodic[2]);
        }
        return r2_unfused(ddx, ddy, ddz);
      };
      bool in_list, in_near;
      if constexpr (Mir::kFixed) {
        // the record prefilter, the exact test in its band
        const float r2f = pb.iso ? pre_r2<true>(static_cast<const int4*>(a.M)[jj], mi_rec, pb)
                                 : pre_r2<false>(static_cast<const int4*>(a.M)[jj], mi_rec, pb);
        if ((r2f >= pb.lo_list && r2f <= pb.hi_list) ||
            (r2f >= pb.lo_near && r2f <= pb.hi_near)) {
          const double r2 = exact_r2();
          in_list = r2 < r_list_sq;
          in_near = r2 < near_sq;
        } else {
          in_list = r2f < pb.lo_list;
          in_near = r2f < pb.lo_near;
        }
      } else {
        const double r2 = exact_r2();
        in_list = r2 < r_list_sq;
        in_near = r2 < near_sq;
      }
      const bool hit = valid && j != i && in_list;
      const uint32_t hg = static_cast<uint32_t>(__ballot(hit) >> sh);
      if constexpr (kCount) {
        count += __popc(hg);
        continue;
      }
      const bool kept = hit && count + __popc(hg & lt) < cap;
      const bool near = kept && in_near;
      const uint32_t kg = static_cast<uint32_t>(__ballot(kept) >> sh);
      const uint32_t ng = static_cast<uint32_t>(__ballot(near) >> sh);
      if (kept) {
        if (near)
          nbr[ell(i, nn + __popc(ng & lt), cap)] = j;
        else
          nbr[ell(i, cap - 1 - (nf + __popc(kg & ~ng & lt)), cap)] = j;
      }
      count += __popc(hg);
      nn += __popc(ng);
      nf += __popc(kg & ~ng);
    }
  }
  if constexpr (kCount) return act ? count : 0;
  auto stored = [] {  // this wave's stores, before its other lanes read them
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  stored();
  const int gap = cap - nn - nf;  // [nn, cap - nf), the shell at [cap - nf, cap)
  const bool full = act && nf > gap;  // source and destination overlap
  if (__any(full)) {
    // turned round in place first, then down by the gap, 32 at a time
    if (full)
      for (int q = l; q < nf / 2; q += 32) {
        const size_t x = ell(i, cap - 1 - q, cap), y = ell(i, cap - nf + q, cap);
        const int32_t v = nbr[x];
        nbr[x] = nbr[y];
        nbr[y] = v;
      }
    stored();
    for (int q0 = 0; __any(full && q0 < nf); q0 += 32) {
      const bool move = full && gap > 0 && q0 + l < nf;
      const int32_t v = move ? nbr[ell(i, cap - nf + q0 + l, cap)] : 0;
      stored();
      if (move) nbr[ell(i, nn + q0 + l, cap)] = v;
    }
  }
  if (act) {
    if (!full)
      for (int q = l; q < nf; q += 32) nbr[ell(i, nn + q, cap)] = nbr[ell(i, cap - 1 - q, cap)];
    const int n = nn + nf;  // == min(count, cap)
    if (l == 0) {
      cnt[i] = n;
      a.cntn[i] = nn;
    }
    const int k = n + l;
    if (k < ((n + 7) & ~7)) nbr[ell(i, k, cap)] = i;
  }
  return act ? count : 0;
}

// nlist_atom: the same rows by one lane per atom, with a group of candidates'
// loads in flight at a time, for more atoms than there are groups of lanes.
template <bool kCount, class Mir>
__device__ __forceinline__ int nlist_atom(const StepArgs& a, const GridArgs& g, const PermArgs& p,
                                          int i, double r_list_sq, double near_sq, int32_t* nbr,
                                          int32_t* cnt) {
  using T = typename Mir::T;
  constexpr int kG = Mir::kFixed ? 8 : 4;
  const int cap = a.cap;
  const double xi = p.px[i], yi = p.py[i], zi = p.pz[i];
  const MirrorParams& mp = mp_of<Mir>(a, i);
  const CellGrid cg = grid_of<Mir>(a, g, i);
  int c[3];
  cell_coords(cg, xi, yi, zi, c);
  const size_t row =
      27 * static_cast<size_t>(g.rank_of[cg.off + (c[2] * cg.n[1] + c[1]) * cg.n[0] + c[0]]);
  const T* __restrict__ const M = static_cast<const T*>(a.M);
  int4 mi_rec = make_int4(0, 0, 0, 0);
  PreBounds pb{};
  if constexpr (Mir::kFixed) {
    mi_rec = M[i];
    pb = pre_bounds(mp, r_list_sq, near_sq);
  }
  int count = 0, nn = 0, nf = 0;
  int32_t* const to = kCount ? nullptr : nbr + ell(i, 0, cap);
  auto slot = [&](int k) -> int32_t& { return to[(k >> 2) * 256 + (k & 3)]; };
  // one copy of the search per image mode, so that a group's loads issue together
  auto search = [&](auto with_images, auto iso_units) {
    constexpr bool kImg = decltype(with_images)::value;
    constexpr bool kIsoU = decltype(iso_units)::value;
    for (int t = 0; t < 27; ++t) {
      const int r = g.around[row + t];
      const int start = g.cstart[r], end = g.cstart[r + 1];
      const int img = kImg ? g.around_img[row + t] : 0;
      auto shift = [&](int d) {
        const int s = (img >> (2 * d)) & 3;
        return s == 0 ? 0.0 : s == 1 ? mp.L[d] : -mp.L[d];
      };
      const double sx = shift(0), sy = shift(1), sz = shift(2);
      auto r2_of = [&](double x, double y, double z) {
        double dx = x - xi, dy = y - yi, dz = z - zi;
        if constexpr (kImg) {
          dx += sx;
          dy += sy;
          dz += sz;
        } else {
          dx = min_image(dx, mp.L[0], mp.hL[0], mp.periodic[0]);
          dy = min_image(dy, mp.L[1], mp.hL[1], mp.periodic[1]);
          dz = min_image(dz, mp.L[2], mp.hL[2], mp.periodic[2]);
        }
        return r2_unfused(dx, dy, dz);
      };
      for (int j0 = start; j0 < end; j0 += kG) {
        T m[kG];
#pragma unroll
        for (int q = 0; q < kG; ++q) m[q] = M[min(j0 + q, end - 1)];
        bool in[kG], near[kG];
        if constexpr (Mir::kFixed) {
          // (bitwise: no branch splits the group)
          bool band[kG], any = false;
#pragma unroll
          for (int q = 0; q < kG; ++q) {
            const float r2f = pre_r2<kIsoU>(m[q], mi_rec, pb);
            const bool valid = (j0 + q < end) & (j0 + q != i);
            in[q] = valid & (r2f < pb.lo_list);
            near[q] = valid & (r2f < pb.lo_near);
            band[q] = valid & (((r2f <= pb.hi_list) & !(r2f < pb.lo_list)) |
                               ((r2f <= pb.hi_near) & !(r2f < pb.lo_near)));
            any |= band[q];
          }
          if (any) {
#pragma unroll
            for (int q = 0; q < kG; ++q)
              if (band[q]) {
                const int j = j0 + q;
                const double r2 = r2_of(p.px[j], p.py[j], p.pz[j]);
                in[q] = r2 < r_list_sq;
                near[q] = r2 < near_sq;
              }
          }
        } else {
#pragma unroll
          for (int q = 0; q < kG; ++q) {
            const double r2 = r2_of(m[q].x, m[q].y, m[q].z);
            const bool valid = (j0 + q < end) & (j0 + q != i);
            in[q] = valid & (r2 < r_list_sq);
            near[q] = r2 < near_sq;
          }
        }
#pragma unroll
        for (int q = 0; q < kG; ++q)
          if (in[q]) {
            if (!kCount && nn + nf < cap) {
              if (near[q])
                slot(nn++) = j0 + q;
              else
                slot(cap - 1 - nf++) = j0 + q;
            }
            ++count;
          }
      }
    }
  };
  bool images;
  if constexpr (Mir::kMB)
    images = a.boxes[a.rep[i]].images != 0;
  else
    images = g.images != 0;
  if (images)
    pb.iso ? search(std::true_type{}, std::true_type{})
           : search(std::true_type{}, std::false_type{});
  else
    pb.iso ? search(std::false_type{}, std::true_type{})
           : search(std::false_type{}, std::false_type{});
  if constexpr (!kCount) {
    const int gap = cap - nn - nf;
    if (nf > gap) {  // turned round in place first, then down by the gap
      for (int q = 0; q < nf / 2; ++q) {
        const int32_t v = slot(cap - 1 - q);
        slot(cap - 1 - q) = slot(cap - nf + q);
        slot(cap - nf + q) = v;
      }
      if (gap > 0)
        for (int q = 0; q < nf; ++q) slot(nn + q) = slot(cap - nf + q);
    } else {
      for (int q = 0; q < nf; ++q) slot(nn + q) = slot(cap - 1 - q);
    }
    const int n = nn + nf;  // == min(count, cap)
    cnt[i] = n;
    a.cntn[i] = nn;
    for (int k = n; k < ((n + 7) & ~7); ++k) slot(k) = i;
  }
  return count;
}

// The rows of all atoms by kLanes lanes (1 or 32) each, by `waves` wavefronts of
// which this is `wave`. Returns the largest count this lane's rows had.
template <bool kCount, int kLanes, class Mir>
__device__ __forceinline__ int nlist_atoms(const StepArgs& a, const GridArgs& g, const PermArgs& p,
                                           double r_list_sq, double near_sq, int32_t* nbr,
                                           int32_t* cnt, int wave, int waves) {
  const int lane = static_cast<int>(threadIdx.x & 63);
  int most = 0;
  if constexpr (kLanes == 1) {
    for (int64_t i = 64 * static_cast<int64_t>(wave) + lane; i < a.natoms;
         i += 64 * static_cast<int64_t>(waves))
      most = max(most, nlist_atom<kCount, Mir>(a, g, p, static_cast<int>(i), r_list_sq, near_sq,
                                               nbr, cnt));
    return most;
  }
  for (int64_t b = 2 * static_cast<int64_t>(wave); b < a.natoms;
       b += 2 * static_cast<int64_t>(waves)) {
    const int i = static_cast<int>(b) + (lane >> 5);
    const bool act = i < a.natoms;
    most = max(most, nlist_atom_group<kCount, Mir>(a, g, p, act ? i : static_cast<int>(b), act,
                                                   r_list_sq, near_sq, nbr, cnt));
  }
  return most;
}

// The rows of all cells, dealt to teams of wavefronts: the whole 1024-thread
// workgroup, or halves or quarters of it where there are more cells than
// workgroups and their stencils fit a team's share of the LDS. A team stages its cell's candidates -- the atoms of the 27
// stencil cells, in rank order -- in LDS once: FP32 offsets from the cell's
// centre, from the wrapping difference of the fixed-point records or from the
// FP64 position with the stencil entry's image. Then, in three steps:
//
// 1. r^2 of all home atoms against all candidates on the matrix cores, 16 x 16
//    at a time, as |a|^2 - 2 a.b + |b|^2 with r_list^2 taken off the
//    accumulator's start: a sign bit is a hit, and a lane collects 16
//    candidates' signs, for either radius, into masks. A pair closer to a
//    radius than the FP32 error takes the exact test (loads of the positions,
//    which the whole workgroup waits for: a wider band costs time). That error,
//    with S = 2 |a| + r_list >= |a| + |b| near a radius: the offsets' rounding,
//    2^-22 r_list S; the squares', products' and sum's, 6.5 2^-24 S^2; and a
//    unit of the records on each axis, 3.5 r_list units (open axes are taken in
//    units of two, so that an atom far out keeps its side of the centre).
// 2. Half a wavefront turns a row's masks into the list of its candidates, near
//    ones first: a popcount prefix over the words, then each lane its own bits.
// 3. It writes the row, one quad of slots a lane.
//
// Boxes where the offsets' image could differ from the minimum image (under
// three cells of r_list on a periodic axis) take r^2 from the records'
// wrapping differences in step 1 (fixed point). nlist_atom_group takes such
// boxes with FP64 records, cells whose stencil or masks do not fit, and rows
// over the capacity.
//
// A round of cells (18-32 atoms, 500-860 candidates each) costs about 2.5 us of
// load latency for the tables and candidates, 3-6 us in the masks and 3-6 us in
// the rows, both of them VALU issue. List phase of a rebuild, us, against 32
// lanes an atom (up to 131,072 atoms) or one straight from memory: 256 EAM atoms
// 17.5 -> 10.8, 4,000 Morse 21 -> 16, 32,000 EAM 64 -> 41, 32,000 Morse in FP64
// 80 -> 32, 256,000 EAM in FP64 232 -> 195, 1,048,576 EAM 776 -> 764.
constexpr int kListBlock = 1024;
constexpr int kListCand = 4096;   // candidates staged by a workgroup
constexpr int kListMask = 8192;   // mask words (32 candidates) of a workgroup
constexpr int kListRow = 1024;    // entries of a row in LDS
constexpr float kSumError = 6.5e-7f;

struct ListLds {
  union {
    float rel[4 * (kListCand + 16)];  // per team: x, y, z, |.|^2 of tcand + 4 each
    uint16_t row[kListBlock / 32][kListRow];
  };
  int32_t idx[kListCand];
  uint32_t in[kListMask];
  uint32_t near[kListMask];
  int32_t start[2][4][27];  // two rounds' tables
  int32_t end[2][4][27];    // run t of team w: candidates [end[w][t - 1], end[w][t])
  uint8_t img[2][4][28];
  int32_t home[2][4][2];  // the cell's first atom and atom count
};

// Inclusive sum over the 32 lanes of a wavefront's half.
__device__ __forceinline__ int half_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, true);  // row_bcast:15
  return v;
}

// Returns the largest count this lane's rows had.
template <bool kCount, class Mir>
__device__ __forceinline__ int nlist_cells(const StepArgs& a, const GridArgs& g, const PermArgs& p,
                                           double r_list_sq, double near_sq, int32_t* nbr,
                                           int32_t* cnt, ListLds& L) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int kWaves = kListBlock / 64;
  const int lane = static_cast<int>(threadIdx.x & 63);
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int grid = static_cast<int>(gridDim.x);
  const int tsh = min(g.list_teams, g.ncells > 2 * grid ? 2 : g.ncells > grid ? 1 : 0);
  const int teams = 1 << tsh;
  const int tw = kWaves >> tsh;                           // wavefronts of a team
  const int team = w >> (4 - tsh), wt = w & (tw - 1);     // this one's team and place in it
  const int tcand = kListCand >> tsh;
  const int cs4 = tcand + 4;  // a component's stride: four in different LDS banks
  float* const rel = L.rel + team * 4 * cs4;
  int32_t* const idx = L.idx + team * tcand;
  uint32_t* const m_in = L.in + team * (kListMask >> tsh);
  uint32_t* const m_near = L.near + team * (kListMask >> tsh);
  const int cap = a.cap;
  const float rl2 = static_cast<float>(r_list_sq);
  const float gap = static_cast<float>(r_list_sq - near_sq);
  const float rl = sqrtf(rl2);
  const float pre = static_cast<float>(r_list_sq * kPreMargin);
  int most = 0;
  // groups of `teams` consecutive cells, dealt so that an XCD's are consecutive
  const int ngroups = (g.ncells + teams - 1) >> tsh;
  const int xcds = grid >= 8 ? 8 : 1;
  const int per = (ngroups + xcds - 1) / xcds;
  const int x = static_cast<int>(blockIdx.x) % xcds;
  const int step = (grid - x + xcds - 1) / xcds;  // workgroups that share these groups
  // the stencil's runs of this team's cell in group m0, by one wavefront
  auto table = [&](int m0, int buf) {
    const int c = ((x * per + m0) << tsh) + team;
    const bool in_grid = m0 < per && x * per + m0 < ngroups && c < g.ncells;
    int n = 0;
    if (in_grid && lane < 27) {
      const int r = g.around[27 * static_cast<size_t>(c) + lane];
      const int s = g.cstart[r];
      n = g.cstart[r + 1] - s;
      L.start[buf][team][lane] = s;
      L.img[buf][team][lane] = g.around_img[27 * static_cast<size_t>(c) + lane];
      if (r == c) {
        L.home[buf][team][0] = s;
        L.home[buf][team][1] = n;
      }
    }
    if (!in_grid && lane == 0) L.home[buf][team][1] = 0;
    n = half_scan(n);
    if (lane < 27) L.end[buf][team][lane] = n;
  };
  if (wt == 0) table(static_cast<int>(blockIdx.x) / xcds, 0);
  int buf = 0;
  for (int m0 = static_cast<int>(blockIdx.x) / xcds; m0 < per; m0 += step, buf ^= 1) {
    __syncthreads();  // the table stands, the LDS of the previous cells is done with
    const int nh = __builtin_amdgcn_readfirstlane(L.home[buf][team][1]);
    const int h0 = nh > 0 ? __builtin_amdgcn_readfirstlane(L.home[buf][team][0]) : 0;
    const int m = nh > 0 ? __builtin_amdgcn_readfirstlane(L.end[buf][team][26]) : 0;
    const int nch = (m + 63) >> 6;
    const MirrorParams& mp = mp_of<Mir>(a, h0);
    bool images = false, flat = false;  // flat: offsets carry the image
    double ctr[3] = {0.0, 0.0, 0.0};
    int ref[3] = {0, 0, 0}, half[3] = {0, 0, 0};  // the centre as a record
    float u[3] = {0.0f, 0.0f, 0.0f}, unit_err = 0.0f;
    auto shift = [&](int img, int d) {
      const int s = (img >> (2 * d)) & 3;
      return s == 0 ? 0.0 : s == 1 ? mp.L[d] : -mp.L[d];
    };
    if (nh > 0) {
      if constexpr (Mir::kMB)
        images = a.boxes[a.rep[h0]].images != 0;
      else
        images = g.images != 0;
      flat = images;
      const CellGrid cg = grid_of<Mir>(a, g, h0);
      const double at[3] = {p.px[h0], p.py[h0], p.pz[h0]};
      int cc[3];
      cell_coords(cg, at[0], at[1], at[2], cc);
      for (int d = 0; d < 3; ++d) {
        const double cs = 1.0 / cg.inv_cs[d];
        ctr[d] = cg.lo[d] + (cc[d] + 0.5) * cs;
        if constexpr (Mir::kFixed) {
          // half a cell and r_list stay within half the box
          flat = flat && (!mp.periodic[d] || cs * cs >= r_list_sq * 1.00001);
          u[d] = static_cast<float>(mp.unit[d]);
          // (an open axis: 0 to 2^30 units, a periodic one mod 2^32)
          ref[d] = MirrorFixed::enc1(ctr[d], mp.lo[d], mp.q[d]);
        } else {
          // FP64 itself resolves 1e-7 r_list there
          flat = flat && (fabs(ctr[d]) + mp.L[d]) * (fabs(ctr[d]) + mp.L[d]) < 1e16 * r_list_sq;
        }
      }
      if constexpr (Mir::kFixed) {
        for (int d = 0; d < 3; ++d) {
          // an open axis in units of two: an atom far out may be more than 2^31
          // units from the centre
          half[d] = flat && !mp.periodic[d] ? 1 : 0;
          ref[d] >>= half[d];
          u[d] = half[d] ? 2.0f * u[d] : u[d];
          unit_err = fmaxf(unit_err, 4.0f * rl * u[d]);
        }
      }
    }
    const bool staged =
        m <= tcand && nh * nch * 2 <= (kListMask >> tsh) && (Mir::kFixed || flat);
    // the run that candidate q lies in: the first that ends beyond it
    auto run_of = [&](int q) {
      int t = 0;
#pragma unroll
      for (int s = 16; s > 0; s >>= 1)
        if (t + s <= 26 && L.end[buf][team][t + s - 1] <= q) t += s;
      return t;
    };
    if (staged) {
      for (int q = wt * 64 + lane; q < m; q += tw * 64) {
        const int t = run_of(q);
        const int j = L.start[buf][team][t] + (q - (t > 0 ? L.end[buf][team][t - 1] : 0));
        const typename Mir::T v = static_cast<const typename Mir::T*>(a.M)[j];
        idx[q] = j;
        float o[3];
        if constexpr (Mir::kFixed) {
          if (flat) {
            o[0] = static_cast<float>(MirrorFixed::wdiff(v.x >> half[0], ref[0])) * u[0];
            o[1] = static_cast<float>(MirrorFixed::wdiff(v.y >> half[1], ref[1])) * u[1];
            o[2] = static_cast<float>(MirrorFixed::wdiff(v.z >> half[2], ref[2])) * u[2];
          } else {
            o[0] = __int_as_float(v.x);
            o[1] = __int_as_float(v.y);
            o[2] = __int_as_float(v.z);
          }
        } else {
          const int img = L.img[buf][team][t];
          o[0] = static_cast<float>(v.x + shift(img, 0) - ctr[0]);
          o[1] = static_cast<float>(v.y + shift(img, 1) - ctr[1]);
          o[2] = static_cast<float>(v.z + shift(img, 2) - ctr[2]);
        }
        float n2 = o[0] * o[0] + o[1] * o[1] + o[2] * o[2];
        if (!Mir::kFixed && !(n2 < 1e30f)) {  // far out or not finite: no hit, or asked for
          o[0] = o[1] = o[2] = 0.0f;
          n2 = __builtin_huge_valf();
        }
        rel[q] = o[0];
        rel[cs4 + q] = o[1];
        rel[2 * cs4 + q] = o[2];
        rel[3 * cs4 + q] = n2;
      }
    }
    __syncthreads();
    if (wt == tw - 1) table(m0 + step, buf ^ 1);
    if (staged && nh > 0) {
      // the first candidate of the home cell's own run: there an atom meets itself
      int lo = 0;
      bool own = false;
      if (lane < 27) {
        lo = lane > 0 ? L.end[buf][team][lane - 1] : 0;
        own = L.start[buf][team][lane] == h0 && L.end[buf][team][lane] > lo;
      }
      const unsigned long long home = __builtin_amdgcn_ballot_w64(own);
      const int self0 = __builtin_amdgcn_readlane(lo, home != 0 ? __builtin_ctzll(home) : 0);
      // lane (piece s of the chunk, home atom b + col): bit e of its piece is
      // candidate 64 ch + 16 s + e
      const int col = lane & 15, s = lane >> 4;
      for (int b = 0; b < nh; b += 16) {
        const int h = self0 + min(b + col, nh - 1);
        float width = pre, bv = 0.0f;
        f32x4 c_list{};
        if (!Mir::kFixed || flat) {
          const float a2 = rel[3 * cs4 + h];
          const float span = 2.0f * sqrtf(a2) + rl;
          width = kSumError * span * span + unit_err;
          bv = s < 3 ? -2.0f * rel[s * cs4 + h] : 1.0f;
          c_list = f32x4{1.0f, 1.0f, 1.0f, 1.0f} * (a2 - rl2);
        }
        for (int ch = wt; ch < nch; ch += tw) {
          const int q0 = 64 * ch + 16 * s;
          unsigned in = 0, near = 0;
          float v[16], f[16];  // r^2 - r_list^2, r^2 - r_near^2 of the piece
          if (!Mir::kFixed || flat) {
            // rows 4 s + e of product t: candidates 64 ch + 16 s + 4 t + e
            const float* const from = rel + s * cs4 + 64 * ch + 16 * (col >> 2) + (col & 3);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const f32x4 r = __builtin_amdgcn_mfma_f32_16x16x4f32(from[4 * t], bv, c_list, 0, 0, 0);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                v[4 * t + e] = r[e];
                f[4 * t + e] = r[e] + gap;
              }
            }
          } else {
            const int ax = __float_as_int(rel[h]), ay = __float_as_int(rel[cs4 + h]),
                      az = __float_as_int(rel[2 * cs4 + h]);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const float dx =
                  u[0] * static_cast<float>(MirrorFixed::wdiff(__float_as_int(rel[q0 + e]), ax));
              const float dy = u[1] * static_cast<float>(
                                          MirrorFixed::wdiff(__float_as_int(rel[cs4 + q0 + e]), ay));
              const float dz = u[2] * static_cast<float>(MirrorFixed::wdiff(
                                          __float_as_int(rel[2 * cs4 + q0 + e]), az));
              const float r2 = dx * dx + dy * dy + dz * dz;
              v[e] = r2 - rl2;
              f[e] = v[e] + gap;
            }
          }
          float closest = __builtin_huge_valf();
#pragma unroll
          for (int e = 15; e >= 0; --e) {
            in = __builtin_amdgcn_alignbit(in, __float_as_uint(v[e]), 31);
            near = __builtin_amdgcn_alignbit(near, __float_as_uint(f[e]), 31);
            closest = fminf(fminf(fabsf(v[e]), fabsf(f[e])), closest);
          }
          unsigned valid = 0xffffu;
          if (ch == nch - 1) {
            const int left = m - q0;
            valid = left >= 16 ? 0xffffu : left > 0 ? (1u << left) - 1u : 0u;
          }
          if (self0 + b < 64 * ch + 64 && self0 + b + 16 > 64 * ch) {
            const int self = h - q0;
            if (self >= 0 && self < 16) valid &= ~(1u << self);
          }
          if (!(closest > width) && valid != 0) {
            unsigned ask = 0;
#pragma unroll
            for (int e = 0; e < 16; ++e)
              if (!(fabsf(v[e]) > width && fabsf(f[e]) > width)) ask |= 1u << e;
            const int i = h0 + h - self0;
            for (ask &= valid; ask != 0; ask &= ask - 1) {
              const int e = __builtin_ctz(ask);
              const int j = idx[q0 + e];
              const int img = L.img[buf][team][run_of(q0 + e)];
              double dx, dy, dz;
              if constexpr (Mir::kFixed) {
                dx = p.px[j] - p.px[i];
                dy = p.py[j] - p.py[i];
                dz = p.pz[j] - p.pz[i];
              } else {  // an FP64 record holds the position itself
                const typename Mir::T rj = static_cast<const typename Mir::T*>(a.M)[j];
                const typename Mir::T ri = static_cast<const typename Mir::T*>(a.M)[i];
                dx = rj.x - ri.x;
                dy = rj.y - ri.y;
                dz = rj.z - ri.z;
              }
              if (images) {
                dx = (img & 3) ? dx + shift(img, 0) : dx;
                dy = ((img >> 2) & 3) ? dy + shift(img, 1) : dy;
                dz = ((img >> 4) & 3) ? dz + shift(img, 2) : dz;
              } else {
                dx = min_image(dx, mp.L[0], mp.hL[0], mp.periodic[0]);
                dy = min_image(dy, mp.L[1], mp.hL[1], mp.periodic[1]);
                dz = min_image(dz, mp.L[2], mp.hL[2], mp.periodic[2]);
              }
              const double r2 = r2_unfused(dx, dy, dz);
              in = (in & ~(1u << e)) | ((r2 < r_list_sq ? 1u : 0u) << e);
              near = (near & ~(1u << e)) | ((r2 < near_sq ? 1u : 0u) << e);
            }
          }
          if (b + col < nh) {
            const int o = ((b + col) * nch + ch) * 4 + s;
            reinterpret_cast<uint16_t*>(m_in)[o] = static_cast<uint16_t>(in & valid);
            reinterpret_cast<uint16_t*>(m_near)[o] = static_cast<uint16_t>(in & near & valid);
          }
        }
      }
    }
    __syncthreads();
    // rows, one to a half wavefront
    const int hl = lane & 31;
    uint16_t* const list = L.row[2 * w + (lane >> 5)];
    for (int b = 2 * wt; b < nh; b += 2 * tw) {
      const int h = b + (lane >> 5);
      const bool act = h < nh;
      const int i = h0 + (act ? h : b);
      int n = 0, nn = 0;
      bool slow = !staged;
      if (staged) {
        const uint32_t* const in = m_in + (act ? h : b) * nch * 2;
        const uint32_t* const near = m_near + (act ? h : b) * nch * 2;
        int sum = 0;  // in | near << 16: a row has at most kListCand
        for (int q = hl; q < 2 * nch; q += 32) sum += __popc(in[q]) | (__popc(near[q]) << 16);
        sum = __shfl(half_scan(sum), lane | 31);
        n = sum & 0xffff;
        nn = sum >> 16;
        if constexpr (kCount) {
          if (act) most = max(most, n);
          continue;
        }
        slow = __any(act && n > min(cap, kListRow));
      }
      if (slow) {
        const int got =
            nlist_atom_group<kCount, Mir>(a, g, p, i, act, r_list_sq, near_sq, nbr, cnt);
        if (act) most = max(most, got);
        continue;
      }
      if constexpr (!kCount) {
        const uint32_t* const in = m_in + (act ? h : b) * nch * 2;
        const uint32_t* const near = m_near + (act ? h : b) * nch * 2;
        int base = 0;
        for (int q0 = 0; q0 < 2 * nch; q0 += 32) {
          const int q = q0 + hl;
          const uint32_t bits = q < 2 * nch ? in[q] : 0u;
          const uint32_t nb = q < 2 * nch ? near[q] : 0u;
          const int own = __popc(bits) | (__popc(nb) << 16);
          const int incl = base + half_scan(own);
          const int before = incl - own;
          base = __shfl(incl, lane | 31);
          const int before_near = before >> 16;
          uint16_t* to = list + before_near;
          for (uint32_t left = nb; left != 0; left &= left - 1)
            *to++ = static_cast<uint16_t>(32 * q + __builtin_ctz(left));
          to = list + nn + (before & 0xffff) - before_near;
          for (uint32_t left = bits ^ nb; left != 0; left &= left - 1)
            *to++ = static_cast<uint16_t>(32 * q + __builtin_ctz(left));
        }
        // the wave's own LDS stores, read by its other lanes
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (act) {
          // padded to a multiple of 8 with the atom itself, so unrolled readers
          // can load whole groups of slots (cap is a multiple of 8)
          int32_t* const row = nbr + ell(i, 0, cap);
          for (int q = hl; q < 2 * ((n + 7) >> 3); q += 32) {
            int4 v;
            v.x = 4 * q < n ? idx[list[4 * q]] : i;
            v.y = 4 * q + 1 < n ? idx[list[4 * q + 1]] : i;
            v.z = 4 * q + 2 < n ? idx[list[4 * q + 2]] : i;
            v.w = 4 * q + 3 < n ? idx[list[4 * q + 3]] : i;
            *reinterpret_cast<int4*>(row + 256 * q) = v;
          }
          if (hl == 0) {
            cnt[i] = n;
            a.cntn[i] = nn;
          }
          most = max(most, n);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      }
    }
  }
  return most;
}

// Largest row count of the wave: recorded for sizing (kCount) or flagged as
// an overflow of the capacity.
template <bool kCount>
__device__ __forceinline__ void report_count(const StepArgs& a, int count, int32_t* maxcnt) {
  const int m = wave_max_i(count);
  if ((threadIdx.x & 63) == 0 && m > 0) {
    if (kCount) {
      atomicMax(maxcnt, m);
    } else if (m > a.cap) {
      atomicMax(&a.flags[1], m);
    }
  }
}

// ---- the separate kernels (first build; every one returns at once when
// the rebuild flag is clear) ----

template <class Mir>
__global__ void __launch_bounds__(kBlock) k_bin(StepArgs a, GridArgs g) {
  if (!a.flags[0]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.natoms) return;
  bin_atom<Mir>(a, g, i);
}

static __global__ void __launch_bounds__(1024) k_cell_scan(const int32_t* flags, GridArgs g) {
  if (!flags[0]) return;
  scan_cells<1024>(g, g.cstart);
}

static __global__ void __launch_bounds__(kBlock) k_scatter(StepArgs a, GridArgs g) {
  if (!a.flags[0]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.natoms) return;
  scatter_atom(g, i, g.cstart);
}

// One wavefront per cell, or one lane per atom with the searches by atoms.
template <class R, class Mir>
__global__ void __launch_bounds__(kBlock) k_order_permute(StepArgs a, GridArgs g, PermArgs t) {
  if (!a.flags[0]) return;
  if (g.list_lanes > 0) {
    const int s = blockIdx.x * kBlock + threadIdx.x;
    if (s < a.natoms) order_slot(g, s, [&](int o, int to) { permute_atom<R, Mir>(a, g, t, o, to); });
    return;
  }
  const int r = blockIdx.x * (kBlock / 64) + static_cast<int>(threadIdx.x >> 6);
  if (r >= g.ncells) return;
  order_cell_wave(g, r, [&](int o, int s) { permute_atom<R, Mir>(a, g, t, o, s); });
}

template <class R, class Mir>
__global__ void __launch_bounds__(kBlock) k_copyback(StepArgs a, GridArgs g, PermArgs t) {
  if (!a.flags[0]) return;
  const int s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= a.natoms) return;
  copyback_atom<R, Mir>(a, g, t, s);
}

template <bool kCount, class Mir>
__global__ void __launch_bounds__(kListBlock)
k_nlist_ell(StepArgs a, GridArgs g, PermArgs t, double r_list_sq, double near_sq, int32_t* nbr,
            int32_t* cnt, int32_t* maxcnt) {
  if (!kCount && !a.flags[0]) return;
  __shared__ ListLds L;
  const int count = nlist_cells<kCount, Mir>(a, g, t, r_list_sq, near_sq, nbr, cnt, L);
  report_count<kCount>(a, count, maxcnt);
}

template <bool kCount, int kLanes, class Mir>
__global__ void __launch_bounds__(kBlock)
k_nlist_atoms(StepArgs a, GridArgs g, PermArgs t, double r_list_sq, double near_sq, int32_t* nbr,
              int32_t* cnt, int32_t* maxcnt) {
  if (!kCount && !a.flags[0]) return;
  constexpr int kWaves = kBlock / 64;
  const int count = nlist_atoms<kCount, kLanes, Mir>(
      a, g, t, r_list_sq, near_sq, nbr, cnt,
      static_cast<int>(blockIdx.x) * kWaves + static_cast<int>(threadIdx.x >> 6),
      static_cast<int>(gridDim.x) * kWaves);
  report_count<kCount>(a, count, maxcnt);
}

// End of a rebuild: the last block to finish clears the flag (every block has
// read it by then), so the next step's kernels see a clean state.
static __global__ void __launch_bounds__(kBlock) k_rebuild_done(int32_t* flags, int32_t* done,
                                                         int nblocks, int64_t* rebuilds) {
  if (!flags[0]) return;
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    const int prev = atomicAdd(done, 1);
    if (prev == nblocks - 1) {
      *done = 0;
      flags[4] = 1;  // the rows changed: halos are rebuilt next
      flags[0] = 0;
      *rebuilds += 1;
    }
  }
}

// ---------------------------------------------------------------------------
// Halos of the LDS-staged passes. Block b of those passes covers atoms
// [1024 b, 1024 b + 1024); its halo is the set of atoms its rows name (the
// block's own atoms included), in increasing index. A pass copies the halo's
// records into LDS once and gathers neighbour records from there, so a
// block reads ~3.5 records per atom from L2 instead of one per row slot.
//
// Built after every rebuild by one workgroup per block at a time -- as the
// last phase of the fused rebuild, or by k_halo after a rebuild by separate
// kernels (flags[4]). The set is kept as 64-atom chunks: an LDS hash maps a
// chunk id (j >> 6) to a 64-bit mask of its atoms present. Atoms are in
// cell order, so a row names its neighbours in runs of a few chunks (a
// stencil cell's atoms are adjacent indices): a thread ORs one mask per run
// into the set instead of inserting every slot. The chunk ids are sorted
// (a few hundred at most), a scan of their popcounts gives each chunk's
// first list position, the list goes out, and a row slot j becomes
// base(j >> 6) + popcount(mask(j >> 6) below bit j & 63). A halo larger
// than stage_cap (or than kHaloMax), or spread over more than kChunkMax
// chunks, leaves the block on its 32-bit rows. k_halo's last workgroup to
// finish clears flags[4].
// ---------------------------------------------------------------------------
constexpr int kHaloMax = 6144;                 // distinct atoms a staged halo may hold
constexpr int kChunkBits = 10;
constexpr int kChunkSlots = 1 << kChunkBits;   // hash slots of the chunk set
constexpr int kChunkMax = 768;                 // distinct chunks a halo may touch
static_assert(kHaloMax <= 65536 && kChunkMax <= kChunkSlots, "halo sizing");

constexpr int kHaloBlock = 1024;  // atoms per staged block (= the passes' workgroup)
static_assert(kChunkSlots == kHaloBlock, "one chunk slot per thread in the compaction");

// One slot of the chunk set: chunk id (empty = -1), first list position of
// its atoms, mask of its atoms present. 16 bytes: a probe is one LDS read.
struct alignas(16) HaloChunk {
  int32_t key;
  int32_t base;
  uint64_t mask;
};

struct HaloLds {
  HaloChunk ent[kChunkSlots];
  int32_t srt[kChunkSlots];   // chunk ids, sorted
  int32_t slot[kChunkSlots];  // hash slot of srt[p]
  int32_t wsum[kHaloBlock / 64];
  int nc, fill, ovf;
};

// Multiplicative (Fibonacci) hash of a chunk id onto the set's slots.
__device__ __forceinline__ unsigned chunk_hash(int c) {
  return (static_cast<unsigned>(c) * 2654435761u) >> (32 - kChunkBits);
}

// OR mask m into chunk c of the set (linear probing; a slot's key goes
// from -1 to its chunk once, by CAS). Counts new chunks in *nc; returns
// false once more than kChunkMax are held (the caller stops inserting) or
// the probe finds no slot.
__device__ __forceinline__ bool chunk_or(HaloChunk* ent, int c, uint64_t m, int* nc) {
  unsigned h = chunk_hash(c);
  for (int p = 0; p < kChunkSlots; ++p) {
    int k = __hip_atomic_load(&ent[h].key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (k == -1) {
      k = atomicCAS(&ent[h].key, -1, c);
      if (k == -1) {
        if (atomicAdd(nc, 1) >= kChunkMax) return false;
        k = c;
      }
    }
    if (k == c) {
      atomicOr(reinterpret_cast<unsigned long long*>(&ent[h].mask),
               static_cast<unsigned long long>(m));
      return true;
    }
    h = (h + 1) & (kChunkSlots - 1);
  }
  return false;
}

// Slot of chunk c, which the set holds, read whole: {key, base, mask lo,
// mask hi}. The probe is bounded by the table size all the same.
__device__ __forceinline__ int4 chunk_find(const HaloChunk* ent, int c) {
  unsigned h = chunk_hash(c);
  int4 e = *reinterpret_cast<const int4*>(&ent[h]);
  for (int p = 1; e.x != c && p < kChunkSlots; ++p) {
    h = (h + 1) & (kChunkSlots - 1);
    e = *reinterpret_cast<const int4*>(&ent[h]);
  }
  return e;
}

// List position of atom j, whose chunk the set holds.
__device__ __forceinline__ uint32_t halo_pos(const HaloChunk* ent, int j) {
  const int4 e = chunk_find(ent, j >> 6);
  const uint64_t m = static_cast<uint32_t>(e.z) | (static_cast<uint64_t>(static_cast<uint32_t>(e.w)) << 32);
  const uint64_t below = (uint64_t{1} << (j & 63)) - 1u;
  return static_cast<uint32_t>(e.y + __popcll(m & below));
}

// One row slot j into the thread's current run (chunk cc, mask m); a slot
// in another chunk ORs the run into the set first (ok turns false when the
// set is full).
__device__ __forceinline__ void halo_merge(int j, int& cc, uint64_t& m, bool& ok, HaloLds& L) {
  if ((j >> 6) != cc) {
    ok = ok && chunk_or(L.ent, cc, m, &L.nc);
    cc = j >> 6;
    m = 0;
  }
  m |= uint64_t{1} << (j & 63);
}

// Halos of blocks blockIdx.x, blockIdx.x + gridDim.x, ... (< nblocks), by a
// workgroup of kHaloBlock threads; its LDS is `L`.
__device__ __forceinline__ void build_halos(const StepArgs& a, int nblocks, HaloLds& L) {
  constexpr int nt = kHaloBlock;
  const int tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6;
  const int cap = a.cap;
  int32_t* hj = const_cast<int32_t*>(a.hj);
  int32_t* hn = const_cast<int32_t*>(a.hn);
  int32_t* hmode = const_cast<int32_t*>(a.hmode);
  uint16_t* nbr16 = const_cast<uint16_t*>(a.nbr16);
  const int4* __restrict__ q4 = reinterpret_cast<const int4*>(a.nbr);
  for (int b = blockIdx.x; b < nblocks; b += gridDim.x) {
    L.ent[tid].key = -1;
    L.ent[tid].mask = 0;
    if (tid == 0) {
      L.nc = 0;
      L.fill = 0;
      L.ovf = 0;
    }
    __syncthreads();
    const int i = b * kHaloBlock + tid;
    if (i < a.natoms) {
      // runs of one chunk are merged in (cc, m) and ORed in when the chunk
      // changes; the row in quads, the next quad loaded while this one is
      // merged; slots past the count in the last quad are padding (i, whose
      // chunk starts the first run, since row padding names i itself)
      int cc = i >> 6;
      uint64_t m = uint64_t{1} << (i & 63);
      bool ok = true;
      // (the next quad is loaded by index, the last one reloading itself,
      // rather than selected between a load and a copy: a select of loaded
      // vectors kept them in scratch memory)
      const int nq = (a.cnt[i] + 3) >> 2;
      int4 cur = make_int4(i, i, i, i);
      if (nq > 0) cur = q4[ell(i, 0, cap) >> 2];
      for (int q = 0; q < nq && ok; ++q) {
        const int qn = q + 1 < nq ? q + 1 : q;
        const int4 nxt = q4[ell(i, 4 * qn, cap) >> 2];
        halo_merge(cur.x, cc, m, ok, L);
        halo_merge(cur.y, cc, m, ok, L);
        halo_merge(cur.z, cc, m, ok, L);
        halo_merge(cur.w, cc, m, ok, L);
        cur = nxt;
      }
      if (ok) ok = chunk_or(L.ent, cc, m, &L.nc);
      if (!ok) L.ovf = 1;
    }
    __syncthreads();
    if (L.ovf) {  // the same in every thread
      if (tid == 0) {
        hn[b] = kHaloMax + 1;
        hmode[b] = 1;
      }
      __syncthreads();  // LDS is reused by the next block
      continue;
    }
    // compaction: one slot per thread
    {
      const int k = L.ent[tid].key;
      if (k != -1) L.srt[atomicAdd(&L.fill, 1)] = k;
    }
    __syncthreads();
    const int C = L.fill;
    int P = 1;
    while (P < C) P <<= 1;
    if (tid >= C && tid < P) L.srt[tid] = 0x7fffffff;
    __syncthreads();
    // bitonic sort of srt[0, P), ascending
    for (int size = 2; size <= P; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        if (tid < (P >> 1)) {
          const int lo = 2 * tid - (tid & (stride - 1));
          const int hi = lo + stride;
          const bool up = (lo & size) == 0;
          const int x = L.srt[lo], y = L.srt[hi];
          if ((x > y) == up) {
            L.srt[lo] = y;
            L.srt[hi] = x;
          }
        }
        __syncthreads();
      }
    }
    // exclusive scan of the sorted chunks' popcounts: each chunk's base
    int h = 0, n = 0;
    if (tid < C) {
      h = static_cast<int>(chunk_hash(L.srt[tid]));
      while (L.ent[h].key != L.srt[tid]) h = (h + 1) & (kChunkSlots - 1);
      n = __popcll(L.ent[h].mask);
    }
    int incl = n;
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(incl, off, 64);
      if (lane >= off) incl += o;
    }
    if (lane == 63) L.wsum[w] = incl;
    __syncthreads();
    int base = incl - n, H = 0;
    for (int k = 0; k < nt / 64; ++k) {
      const int s = L.wsum[k];
      base += k < w ? s : 0;
      H += s;
    }
    if (H > a.stage_cap || H > kHaloMax) {  // the same in every thread
      if (tid == 0) {
        hn[b] = H;
        hmode[b] = 1;
      }
      __syncthreads();
      continue;
    }
    if (tid < C) {
      L.ent[h].base = base;
      L.slot[tid] = h;
    }
    __syncthreads();
    // the list: one wavefront per chunk, lane l writes atom 64 c + l if present
    for (int p = w; p < C; p += nt / 64) {
      const HaloChunk e = L.ent[L.slot[p]];
      if ((e.mask >> lane) & 1u) {
        const uint64_t below = (uint64_t{1} << lane) - 1u;
        hj[static_cast<size_t>(b) * kHaloMax + e.base + __popcll(e.mask & below)] =
            e.key * 64 + lane;
      }
    }
    if (i < a.natoms) {
      // the padded row in quads; a quad's four 16-bit positions are
      // adjacent in the 16-bit layout (eight slots per 16 bytes)
      const int mq = ((a.cnt[i] + 7) & ~7) >> 2;
      int4 cur = make_int4(i, i, i, i);
      if (mq > 0) cur = q4[ell(i, 0, cap) >> 2];
      for (int q = 0; q < mq; ++q) {
        const int qn = q + 1 < mq ? q + 1 : q;
        const int4 nxt = q4[ell(i, 4 * qn, cap) >> 2];
        const uint32_t p0 = halo_pos(L.ent, cur.x);
        const uint32_t p1 = halo_pos(L.ent, cur.y);
        const uint32_t p2 = halo_pos(L.ent, cur.z);
        const uint32_t p3 = halo_pos(L.ent, cur.w);
        *reinterpret_cast<uint2*>(nbr16 + ell16(i, 4 * q, cap)) =
            make_uint2(p0 | (p1 << 16), p2 | (p3 << 16));
        cur = nxt;
      }
    }
    if (tid == 0) {
      hn[b] = H;
      hmode[b] = 0;
    }
    __syncthreads();
  }
}

// Standalone halo build after a rebuild by separate kernels (flags[4]).
static __global__ void __launch_bounds__(kHaloBlock) k_halo(StepArgs a, int nblocks, int32_t* done) {
  if (!a.flags[4]) return;
  __shared__ HaloLds L;
  build_halos(a, nblocks, L);
  if (threadIdx.x == 0) {
    __threadfence();
    if (atomicAdd(done, 1) == static_cast<int>(gridDim.x) - 1) {
      *done = 0;
      a.flags[4] = 0;
    }
  }
}

// ---------------------------------------------------------------------------
// Fused rebuild: the whole sort + list sequence in one launch, its phases
// separated by a grid barrier, so a step that needs no rebuild costs one
// early-returning launch instead of seven. The phases: bin | scan + scatter |
// order + permute (records, scratch arrays) | copy back + list (| halos); a
// barrier costs 1.3-7 us, so work moves into a neighbouring phase where its
// inputs allow.
//
// The host keeps the grid to at most one workgroup a CU (the LDS of the list
// search holds one), so every workgroup of the launch runs at once and the
// barrier can complete. Its wait is bounded: a workgroup that has polled
// GridArgs::polls times sets flags[3] and returns (the host reports the error)
// instead of hanging. One that gave up arrives at no later barrier, so none is
// passed and no later phase starts. What it leaves -- cell counters in use,
// arrivals that `gen` does not cover -- is no state to start from: every launch
// until the host has cleared it (check_flags, upload) returns at its first
// barrier, whose arrivals would otherwise count as complete.
//
// Only thread 0 of each workgroup touches the barrier: one release fence, a
// relaxed arrival, relaxed polls, one acquire fence, all at agent scope, and
// the workgroup barriers on either side extend them to the other threads: one
// L2 write-back and one invalidate per workgroup and phase. (An acquiring poll
// would invalidate the XCD's L2 at every poll, under the workgroups still
// working.) Polls back off with a growing sleep.
// ---------------------------------------------------------------------------

// `passed`: barriers this workgroup has passed (GridBarrier::gen at the
// launch's start, counted on here). `gone`, thread 0's: gives up without
// arriving. `polls`: GridArgs::polls.
__device__ __forceinline__ bool grid_barrier(GridBarrier* b, unsigned int* passed,
                                             int32_t* flags, int polls, bool gone = false) {
  __shared__ int ok;
  __syncthreads();
  const unsigned int n = ++*passed;
  if (threadIdx.x == 0 && gone) {
    ok = 0;
  } else if (threadIdx.x == 0) {
    ok = 1;
    unsigned int target = n * gridDim.x;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    if (gridDim.x <= kBarrierFlat) {
      __hip_atomic_fetch_add(&b->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      const unsigned int x = blockIdx.x & 7u;
      const unsigned int nx = (gridDim.x - x + 7u) >> 3;  // workgroups in group x
      target = n * 8u;
      if (__hip_atomic_fetch_add(&b->sub[32u * x], 1u, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT) == n * nx - 1u) {
        // last of its group: passes on what the group's arrivals released
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");
        __hip_atomic_fetch_add(&b->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    for (int spins = 0;; ++spins) {
      if (spins == polls) {
        ok = 0;
        atomicExch(&flags[3], 1);
        break;
      }
      if (static_cast<int>(__hip_atomic_load(&b->count, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT) -
                           target) >= 0)
        break;
      if (spins < 64)
        __builtin_amdgcn_s_sleep(1);
      else if (spins < 256)
        __builtin_amdgcn_s_sleep(16);
      else
        __builtin_amdgcn_s_sleep(64);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  return ok != 0;
}

constexpr int kRebuildBlock = 1024;  // workgroup of the fused rebuild

template <class R, class Mir>
__global__ void __launch_bounds__(kRebuildBlock)
k_rebuild_fused(StepArgs a, GridArgs g, PermArgs t, double r_list_sq, double near_sq,
                int32_t* nbr, int32_t* cnt, GridBarrier* bar, int64_t* rebuilds, int forced) {
  // uniform: nothing writes the flag before the last phase
  if (!forced && !a.flags[0]) return;
  const int tid = blockIdx.x * kRebuildBlock + threadIdx.x;
  const int nthr = gridDim.x * kRebuildBlock;
  const int N = a.natoms;
  __shared__ union {  // one phase's at a time, a grid barrier between them
    int32_t cstart[kScanOwn + 1];
    ListLds list;
    HaloLds halo;
  } lds;
  unsigned int passed = bar->gen;  // written below once every workgroup has read it
  // (read by one thread: workgroups of this launch may be giving up already)
  const bool gone = threadIdx.x == 0 && __hip_atomic_load(&a.flags[3], __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT) != 0;
  // (the cell counters are clear: the phase that last reads them clears them)
  for (int i = tid; i < N; i += nthr) bin_atom<Mir>(a, g, i);
  if (!grid_barrier(bar, &passed, a.flags, g.polls, gone)) return;
  if (g.ncells <= kScanOwn) {
    // few cells: every workgroup scans them for itself, without a barrier
    int32_t* const cstart = lds.cstart;
    scan_cells<kRebuildBlock>(g, cstart);
    __syncthreads();
    if (blockIdx.x == 0)
      for (int r = threadIdx.x; r <= g.ncells; r += kRebuildBlock) g.cstart[r] = cstart[r];
    for (int i = tid; i < N; i += nthr) scatter_atom(g, i, cstart);
  } else {
    scan_cells_grid<kRebuildBlock>(g, 1);
    if (!grid_barrier(bar, &passed, a.flags, g.polls)) return;
    scan_cells_grid<kRebuildBlock>(g, 2);
    if (!grid_barrier(bar, &passed, a.flags, g.polls)) return;
    for (int i = tid; i < N; i += nthr) scatter_atom(g, i, g.cstart);
  }
  if (!grid_barrier(bar, &passed, a.flags, g.polls)) return;
  {
    // one cell per wavefront, cells dealt to the workgroups wave by wave
    const int nw = gridDim.x * (kRebuildBlock / 64);
    const int wv = (threadIdx.x >> 6) * gridDim.x + blockIdx.x;
    auto put = [&](int o, int s) { permute_atom<R, Mir>(a, g, t, o, s); };
    if (g.list_lanes > 0)
      for (int s = tid; s < N; s += nthr) order_slot(g, s, put);
    else
      for (int r = wv; r < g.ncells; r += nw) order_cell_wave(g, r, put);
    for (int r = tid; r < g.ncells; r += nthr) {
      g.ccount[r] = 0;
      g.cursor[r] = 0;
    }
  }
  if (!grid_barrier(bar, &passed, a.flags, g.polls)) return;
  // the state's arrays back from the scratch ones, beside the list search,
  // which reads the scratch arrays and the records
  for (int s = tid; s < N; s += nthr) copyback_atom<R, Mir>(a, g, t, s);
  const int wave = tid >> 6, waves = nthr >> 6;
  int count;
  if (g.list_lanes == 0)
    count = nlist_cells<false, Mir>(a, g, t, r_list_sq, near_sq, nbr, cnt, lds.list);
  else if (g.list_lanes == 1)
    count = nlist_atoms<false, 1, Mir>(a, g, t, r_list_sq, near_sq, nbr, cnt, wave, waves);
  else
    count = nlist_atoms<false, 32, Mir>(a, g, t, r_list_sq, near_sq, nbr, cnt, wave, waves);
  report_count<false>(a, count, nullptr);
  if constexpr (Mir::kFixed) {
    if (a.stage_cap > 0) {  // halos of the staged passes, from the new rows
      if (!grid_barrier(bar, &passed, a.flags, g.polls)) return;
      static_assert(kRebuildBlock == kHaloBlock, "halos are built by whole workgroups");
      build_halos(a, (N + kHaloBlock - 1) / kHaloBlock, lds.halo);
    }
  }
  // every thread read the flag at entry, before the first barrier
  if (tid == 0) {
    a.flags[0] = 0;
    *rebuilds += 1;
    bar->gen = passed;
  }
}

}  // namespace sched
}  // namespace tdmd_hip
