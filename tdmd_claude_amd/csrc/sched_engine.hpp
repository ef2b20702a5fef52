// sched_engine.hpp -- the scheduler's state and its Engine: the launches of
// one precision and mirror encoding. Each engine is compiled in a unit of its
// own (sched_engine_*.cpp), since its kernels take most of the build.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <numeric>
#include <string>
#include <thread>
#include <vector>

#include <hip/hip_ext.h>

#include "sched_kernels.inl"
#include "sched_lds.inl"

namespace tdmd_hip {

using namespace sched;

// Lanes per neighbour row in the force passes (Morse, and EAM through the
// global-table passes). One lane per atom gives 32,000 atoms 125 workgroups on
// 256 CUs, each lane walking ~80 slots in turn, and the time is flat up to a
// wavefront per SIMD (65,536 atoms); eight lanes fill the chip at 8,000 atoms
// and pay their shuffles and idle slots from about 40,000 on. Steps without a
// rebuild, us with 1 / 4 / 8 lanes, mixed:
//   EAM (1: LDS passes)        32,000: 57.6 / 30.7 / 28.2   62,500: 69.6 / 49.1 / 54.5
//                              70,304: 59.7 / 60.1 / 62.5
//   three elements, replicas   22,000: 59.8 / 32.4 / 28.6   80,000: 93.1 / 72.9 / 83.7
//                              130,000: 98.7 / 117.0 / 122.8
//   Morse                      23,328: 23.9 / 14.8 / 12.8   108,000: 39.5 / 38.4 / 40.2
//                              131,072: 39.8 / 42.0 / 44.5
// and in FP64:
//   EAM                        32,000: 131.6 / 47.0 / 46.8  97,556: 139.4 / 129.8 / 132.4
//                              131,072: 142.0 / 172.5 / 174.4
//   three elements, replicas   80,000: 156.0 / 120.1 / 123.0  130,000: 158.0 / 174.6 / 184.0
//   Morse                      62,500: 52.4 / 48.0 / 50.0   131,072: 67.5 / 66.1 / 72.6
//                              186,624: 93.6 / 93.5 / 99.5
constexpr int kSplitLanes = 8;  // the most
constexpr int kSplit8Max = 40960;
// Up to a wavefront a SIMD at eight lanes, the passes for few wavefronts
// (for_neighbours_few). Steps without a rebuild, us, for_neighbours_split /
// these: EAM 256 atoms 14.0 / 12.1, 4,000 17.0 / 14.3 (FP64 21.3 / 19.0),
// 8,788 18.8 / 17.8 (FP64 26.6 / 27.1); Morse 4,000 9.5 / 8.6 (FP64 11.8 /
// 10.7), 8,788 10.4 / 10.6; at 32,000 their loads past a row's end and
// registers cost 3%.
constexpr int kFewMax = 8192;
inline int lanes_by_size(int natoms, bool eam, int ntypes, bool fp64) {
  if (natoms <= kSplit8Max) return kSplitLanes;
  const int max4 = !eam         ? (fp64 ? 131072 : 114688)
                   : ntypes > 1 ? 106496
                                : (fp64 ? 98304 : 65536);
  return natoms <= max4 ? 4 : 1;
}
// Operation codes of a step sequence (also the graph-cache key alphabet).
enum Op : char {
  OP_BOOT = 'b',        // half kick + drift (window start, NVE)
  OP_KD_FULL = 'k',     // full kick + drift as its own launch (Morse pass timing)
  OP_NVT_PRE = 'p',     // chain half-step before the step
  OP_KD_NVT = 'q',      // scaled half kick + drift
  OP_KD_NVT2 = 'Q',     // the previous step's closing half kick, then as 'q'
  OP_REB_FORCED = 'R',  // set flag + rebuild
  OP_REB_COND = 'r',    // rebuild if the device flag is set
  OP_DENS = 'd',        // EAM density pass
  OP_F_FULL = 'F',      // force + next step's kick-drift (Morse: into the other record buffer)
  OP_F_ONLY = 'o',      // force, store F
  OP_F_HALF = 'h',      // force + closing half kick
  OP_F_KICK2 = '2',     // force + half kick + KE partials (NVT)
  OP_F_KE = 'e',        // force + KE partials of the half-kicked v, v not stored
                        // (NVT inside a window: the next 'Q' applies the kick)
  OP_NVT_POST = 'P',    // chain half-step after the step
  OP_NVT_POST_PRE = 'N',// chain half-step after the step + the next step's
  OP_NVT_FINAL = 'Z'    // apply pending chain scale, commit
};

inline int round_up(int x, int m) { return (x + m - 1) / m * m; }

// ---------------------------------------------------------------------------
// Engine: precision- and mirror-specific launches.
// ---------------------------------------------------------------------------
struct EngineBase {
  virtual ~EngineBase() = default;
  virtual int init() = 0;
  virtual int launch(char op, hipStream_t s) = 0;
  virtual int write_mirror(hipStream_t s) = 0;
  virtual int energy_pass(hipStream_t s, double* d_out) = 0;  // d_out[0..2]
  virtual int count_pass(hipStream_t s, int32_t* d_max) = 0;
  virtual int fill_pass(hipStream_t s) = 0;
  virtual int sort_pass(hipStream_t s) = 0;
  // Time the candidate kernel shapes on the current state and keep the
  // fastest; out = {pair_unroll, lds_budget bytes (0: not applicable)}.
  virtual int tune(int iters, int32_t* out) = 0;
  // {lanes per row, neighbour slots per pipelined group, LDS window budget}
  virtual void shape(int32_t* out) const = 0;
  // Bracket the next force-path launch (EAM density / force, Morse
  // kick-drift / force) with events stamped by the dispatch itself.
  hipEvent_t ev_start = nullptr, ev_stop = nullptr;
  void time_next(hipEvent_t a, hipEvent_t b) {
    ev_start = a;
    ev_stop = b;
  }
};

}  // namespace tdmd_hip

struct tdmd_sched {
  int kind = 0;  // 0 Morse, 1 EAM
  tdmd_box box{};
  int natoms = 0;
  int nblocks = 0;   // 256-thread grid (multiple of 8)
  int nb_force = 0;  // grid of the EAM/Morse passes = block partials they emit
  int lanes = 1;  // lanes per atom of the force passes (Morse, global-table EAM)
  bool stage_ok = false;  // halo buffers exist: the staged LDS passes can be chosen
  int nb_rebuild = 0;  // fused rebuild grid (all resident at once); 0: separate kernels
  tdmd_hip::sched::GridBarrier* d_bar = nullptr;
  tdmd_sched_config cfg{};
  tdmd_morse_params morse{};
  tdmd_eam_tables* tables = nullptr;
  hipStream_t stream = nullptr;
  double cutoff = 0, r_list = 0;
  tdmd_hip::sched::StepArgs a{};
  tdmd_hip::sched::GridArgs g{};
  tdmd_hip::sched::PermArgs t{};
  tdmd_hip::sched::NhcParams nhcp{};
  std::unique_ptr<tdmd_hip::EngineBase> eng;
  std::vector<void*> allocs;
  int32_t* d_maxcnt = nullptr;
  int64_t* d_rebuilds = nullptr;
  double* d_scalars = nullptr;
  mutable double* h_stage = nullptr;  // pinned, from the first download on
  mutable hipEvent_t ev_stage[4] = {};
  // the staging buffer's and the scratch block's: a download gathers into the
  // latter, which a rebuild by separate kernels uses from one to the next
  mutable std::mutex scratch_mu;
  std::vector<int32_t> h_types, h_ids;
  std::vector<double> h_masses;
  bool uploaded = false, initial_forces = false;
  // Morse: the gather records alternate between two buffers (the fused
  // kick-drift writes the next step's into the one not being gathered);
  // true when a.M / a.M2 are exchanged relative to their allocation
  bool rec_swapped = false;
  int current_step = 0, steps_since = 0;
  int64_t ticks = 0, launches = 0, host_rebuilds = 0, graph_launches = 0;
  // In-window pass timing: the passes' own device clock (StepArgs::pclock)
  bool pass_timing = false;
  unsigned long long* d_pclock = nullptr;  // 8 words: density, force
  int clock_khz = 0;                       // device wall clock rate
  std::map<std::string, hipGraphExec_t> graphs;
  std::map<std::string, hipGraph_t> graph_defs;
  std::map<std::string, int64_t> graph_kernels;
  std::map<std::string, bool> graph_swaps;  // the graph exchanges the record buffers
  // batches of independent boxes (replicas), atoms of replica r in slots
  // [rep_off[r], rep_off[r+1])
  bool multibox = false;
  std::vector<tdmd_hip::sched::BoxGeo> h_boxes;
  std::vector<int> rep_off;
};

namespace tdmd_hip {

template <class R, class Mir>
struct Engine final : EngineBase {
  tdmd_sched* S;
  explicit Engine(tdmd_sched* s) : S(s) {}

  using Q = typename Quad<R>::type;

  template <class K, class... Args>
  void go(K kernel, dim3 grid, dim3 block, size_t lds, hipStream_t s, Args... args) {
    if (ev_start) {
      hipExtLaunchKernelGGL(kernel, grid, block, static_cast<uint32_t>(lds), s, ev_start, ev_stop,
                            0u, args...);
      ev_start = ev_stop = nullptr;
    } else {
      kernel<<<grid, block, lds, s>>>(args...);
    }
  }

  const SplineMeta* meta() const { return static_cast<const SplineMeta*>(S->tables->d_meta); }
  const Q* coeff() const { return static_cast<const Q*>(S->tables->d_coeff); }
  double rc_sq() const { return S->tables->cutoff * S->tables->cutoff; }
  MorseCoef mp() const {
    return MorseCoef{S->morse.d, S->morse.alpha, S->morse.r0, S->morse.rc_sq};
  }

  // Single-element EAM runs the LDS-table kernels (sched_lds.inl); the
  // windows are sized once from the LDS budget (the device's per-workgroup
  // limit unless the configuration asks for less, e.g. to fit two
  // workgroups per CU).
  bool lds = false;
  // Halo staging (k_halo + the kStage passes) for 16-byte gather records.
  static constexpr bool kCanStage = sizeof(typename Mir::T) == 16;
  bool stage = false;
  bool lds_ok = false;  // single-element tables on one r grid: the LDS passes can run
  int nb_lds = 0;       // 1024-atom blocks of the LDS passes (multiple of 8)
  bool iso = false;  // fixed-point mirror with one unit on all axes (every box)
  int ncu = 0;
  size_t lds_cu = 160 * 1024;  // LDS of one CU
  int32_t* d_halo_done = nullptr;
  size_t stage_bytes() const { return stage ? static_cast<size_t>(kStageCap) * 16 : 0; }
  int unroll = 4;
  int lds_grid = 0;   // persistent workgroups of the LDS passes
  int lds_limit = 0;  // per-workgroup dynamic LDS the kernels are allowed
  int nint = 0;       // r-grid intervals
  int budget = 0;     // current window budget
  LdsWindow w_dens[2]{}, w_force[2]{};  // [kEnergy]
  size_t b_dens[2]{}, b_force[2]{};

  static LdsWindow window(int nint, size_t per, size_t budget, size_t* bytes) {
    LdsWindow w;
    w.nwin = static_cast<int>(std::min<size_t>(static_cast<size_t>(nint), budget / per));
    w.k_lo = nint - w.nwin;
    *bytes = window_bytes(w.nwin, per);
    return w;
  }
  template <class K>
  static int allow_lds(K* fn, size_t bytes) {
    TDMD_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                     static_cast<int>(bytes)));
    return TDMD_OK;
  }

  template <bool kWin, int kU, bool kSt, bool kIs>
  int allow_all() {
    int rc = 0;
    const size_t L = static_cast<size_t>(lds_limit);
    if ((rc = allow_lds(&k_eam_density_lds<R, Mir, false, kWin, kU, kSt, kIs>, L)) ||
        (rc = allow_lds(&k_eam_density_lds<R, Mir, true, kWin, kU, kSt, kIs>, L)) ||
        (rc = allow_lds(&k_eam_force_lds<R, Mir, kForceOnly, true, kWin, kU, kSt, kIs>, L)) ||
        (rc = allow_lds(&k_eam_force_lds<R, Mir, kForceOnly, false, kWin, kU, kSt, kIs>, L)) ||
        (rc = allow_lds(&k_eam_force_lds<R, Mir, kFullKickDrift, false, kWin, kU, kSt, kIs>,
                        L)) ||
        (rc = allow_lds(&k_eam_force_lds<R, Mir, kHalfKick, false, kWin, kU, kSt, kIs>, L)) ||
        (rc = allow_lds(&k_eam_force_lds<R, Mir, kKick2Ke, false, kWin, kU, kSt, kIs>, L)) ||
        (rc = allow_lds(&k_eam_force_lds<R, Mir, kKe, false, kWin, kU, kSt, kIs>, L)))
      return rc;
    return TDMD_OK;
  }
  template <bool kSt, bool kIs>
  int allow_shapes() {
    int rc = 0;
    if ((rc = allow_all<false, 4, kSt, kIs>()) || (rc = allow_all<true, 4, kSt, kIs>()) ||
        (rc = allow_all<false, 8, kSt, kIs>()) || (rc = allow_all<true, 8, kSt, kIs>()))
      return rc;
    return TDMD_OK;
  }

  // Windows for a budget (bytes, clamped to the allowed limit) and unroll.
  // With halo staging the windows get what the halo leaves.
  void configure(int u, int bytes) {
    budget = std::min(bytes > 0 ? bytes : lds_limit, lds_limit);
    const size_t wb = static_cast<size_t>(budget) - std::min(static_cast<size_t>(budget), stage_bytes());
    using V2 = typename Vec2<R>::type;
    for (int e = 0; e < 2; ++e) {
      w_dens[e] = window(nint, sizeof(Q), wb, &b_dens[e]);
      w_force[e] = window(nint, sizeof(Q) + sizeof(V2) + (e ? sizeof(R) : 0), wb, &b_force[e]);
    }
    unroll = u;
    // one workgroup per LDS slot of the device: as many as the CU's LDS
    // holds of the largest pass (at most two of 1024 threads), per CU
    const size_t per_wg = std::max(b_dens[0], b_force[0]) + stage_bytes() + 1024;
    const int per_cu = std::max(1, std::min(2, static_cast<int>(lds_cu / per_wg)));
    lds_grid = std::max(8, std::min(nb_lds, (std::max(ncu, 8) / 8) * 8 * per_cu));
  }

  // Interleaved derivative table of the several-element force pass (see
  // StepArgs::pairtab), from the tables' FP64 coefficients in the kernels'
  // precision: the same values the per-spline quads hold; in mixed
  // precision c and d are stored as 2c and 3d, scaled in float (the values
  // the per-spline path forms at use).
  int build_pair_table() {
    const tdmd_eam_tables* t = S->tables;
    const int nt = t->ntypes;
    SplineMeta m[kMaxSplines];
    const int ns = 2 * nt + nt * (nt + 1) / 2;
    TDMD_HIP_TRY(hipMemcpy(m, t->d_meta, ns * sizeof(SplineMeta), hipMemcpyDeviceToHost));
    for (int k = nt + 1; k < ns; ++k)  // rho and phi splines on one r grid
      if (m[k].n != m[nt].n || m[k].dr != m[nt].dr || m[k].rmin != m[nt].rmin) return TDMD_OK;
    const int nint = m[nt].n - 1;
    std::vector<Q> h(static_cast<size_t>(nt) * nt * nint * 3);
    constexpr bool kF32 = std::is_same_v<R, float>;
    auto co = [&](const std::vector<double>& v, int spline, int k) {
      return static_cast<R>(v[static_cast<size_t>(t->offsets[static_cast<size_t>(spline)] + k)]);
    };
    auto c2 = [&](int spline, int k) {
      const R c = co(t->c, spline, k);
      return kF32 ? static_cast<R>(2) * c : c;
    };
    auto d3 = [&](int spline, int k) {
      const R d = co(t->d, spline, k);
      return kF32 ? static_cast<R>(3) * d : d;
    };
    for (int ti = 0; ti < nt; ++ti)
      for (int tj = 0; tj < nt; ++tj) {
        const int sp = 2 * nt + phi_index(ti, tj, nt), sj = nt + tj, si = nt + ti;
        for (int k = 0; k < nint; ++k) {
          Q* e = &h[(static_cast<size_t>(ti * nt + tj) * nint + k) * 3];
          e[0].x = co(t->b, sp, k);
          e[0].y = c2(sp, k);
          e[0].z = d3(sp, k);
          e[0].w = co(t->b, sj, k);
          e[1].x = c2(sj, k);
          e[1].y = d3(sj, k);
          e[1].z = co(t->b, si, k);
          e[1].w = c2(si, k);
          e[2].x = d3(si, k);
          e[2].y = e[2].z = e[2].w = static_cast<R>(0);
        }
      }
    void* p = nullptr;
    if (int rc = tdmd_malloc(&p, h.size() * sizeof(Q))) return rc;
    S->allocs.push_back(p);
    TDMD_HIP_TRY(hipMemcpy(p, h.data(), h.size() * sizeof(Q), hipMemcpyHostToDevice));
    S->a.pairtab = p;
    S->a.pair_nint = nint;
    return TDMD_OK;
  }

  // Kernel path for `lanes` lanes per row: one lane with single-element
  // tables runs the LDS passes (halo-staged where the halo buffers exist);
  // otherwise the global-table passes with rows split over `lanes` lanes.
  // The fused rebuild builds halos only while the staged passes are chosen.
  void set_path(int lanes) {
    S->lanes = lanes;
    lds = lanes == 1 && lds_ok;
    stage = lds && S->stage_ok;
    S->a.stage_cap = stage ? kStageCap : 0;
    S->nb_force = lds ? nb_lds : S->nblocks * lanes;
  }

  // Workgroups of the fused rebuild: where the list is searched by cells, a cell
  // each up to 64, two each beyond (the rebuild of 864 atoms in 27 cells: 30.9 us
  // with 27, 34.6 with 14; of 10,976 in 216: 50.4 with 216, 45.7 with 108: a
  // barrier costs more the more arrive at it); one a CU, which the list search's LDS fills; and by the atoms one per
  // 32 where every launch rebuilds, one per 1024 under the displacement policy
  // and above 131,072. Rebuilds that run at the same time (schedulers on streams
  // or in processes of their own) have to be resident together, or they wait for
  // each other until they give up: on 256 CUs eight of 32,000 atoms under the
  // displacement policy, but under the fixed one a single scheduler of 8,192
  // atoms in 512 cells takes the chip. Such programs want split_rebuild.
  // (One per 512 atoms up to 64 under the displacement policy takes 17 us less a
  // rebuild of 32,000 Morse atoms in FP64, 63 workgroups against 32, and fits
  // four.)
  int list_grid(int ncu) const {
    const int n = S->natoms;
    const bool few = S->cfg.rebuild_policy == TDMD_REBUILD_DISPLACEMENT || n > 131072;
    const int by_atoms = few ? (n + 1023) / 1024 : (n + 31) / 32;
    if (S->g.list_lanes > 0) return std::max(1, std::min(ncu, by_atoms));
    const int cells = std::min(S->g.ncells, std::max(64, (S->g.ncells + 1) / 2));
    return std::max(1, std::min({ncu, by_atoms, cells}));
  }

  int init() override {
    // (partials: one per block of the larger grid)
    S->lanes = S->cfg.pair_lanes > 0
                   ? S->cfg.pair_lanes
                   : lanes_by_size(S->natoms, S->kind == 1, S->kind == 1 ? S->tables->ntypes : 0,
                                   std::is_same_v<R, double>);
    S->nb_force = S->nblocks * S->lanes;
    S->nb_rebuild = 0;
    if (!S->cfg.split_rebuild) {
      // every workgroup of the fused rebuild must be resident at once
      int dev = 0, ncu = 0, per_cu = 0;
      TDMD_HIP_TRY(hipGetDevice(&dev));
      TDMD_HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
      TDMD_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &per_cu, reinterpret_cast<const void*>(&k_rebuild_fused<R, Mir>), kRebuildBlock, 0));
      S->nb_rebuild = list_grid(ncu);
      if (per_cu < 1) S->nb_rebuild = 0;  // cannot guarantee residency: separate kernels
    }
    if (S->kind == 1 && S->tables->ntypes > 1) return build_pair_table();
    if (S->kind != 1 || S->tables->ntypes != 1) return TDMD_OK;
    // rho_0 and phi_00 must share the r grid (setfl: one Nr, dr).
    SplineMeta m[3];
    TDMD_HIP_TRY(hipMemcpy(m, S->tables->d_meta, sizeof(m), hipMemcpyDeviceToHost));
    if (m[1].n != m[2].n || m[1].dr != m[2].dr || m[1].rmin != m[2].rmin || m[1].n < 2)
      return TDMD_OK;
    int dev = 0, lmax = 0;
    TDMD_HIP_TRY(hipGetDevice(&dev));
    TDMD_HIP_TRY(hipDeviceGetAttribute(&lmax, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    // The dynamic window plus the kernels' static LDS (block reduction)
    // must fit the per-workgroup limit; keep 1 KiB for the static part.
    lds_limit = std::min(lmax, 160 * 1024) - 1024;
    if (S->cfg.lds_budget > 0 && S->cfg.lds_budget < 4096)
      return fail(TDMD_E_INVALID, "scheduler: lds_budget below 4096 bytes");
    nint = m[1].n - 1;
    int rc = 0;
    if ((rc = allow_shapes<false, false>())) return rc;
    TDMD_HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    int lcu = 0;
    if (hipDeviceGetAttribute(&lcu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) ==
            hipSuccess &&
        lcu > 0)
      lds_cu = static_cast<size_t>(lcu);
    lds_ok = true;
    nb_lds = round_up((S->natoms + kBigBlock - 1) / kBigBlock, 8);
    if constexpr (kCanStage) {
      iso = true;
      auto same_unit = [](const MirrorParams& p) {
        return p.unit[0] == p.unit[1] && p.unit[0] == p.unit[2];
      };
      if (S->multibox) {
        for (const BoxGeo& b : S->h_boxes) iso = iso && same_unit(b.mp);
      } else {
        iso = same_unit(S->a.mp);
      }
      if (iso && (rc = allow_shapes<false, true>())) return rc;
      if (!S->cfg.disable_halo && lds_limit >= static_cast<int>(kStageCap) * 16 + 16384) {
        if ((rc = (iso ? allow_shapes<true, true>() : allow_shapes<true, false>()))) return rc;
        const size_t nbf = static_cast<size_t>(nb_lds);
        void* p = nullptr;
        const size_t sizes[5] = {nbf * kHaloMax * 4, nbf * 4, nbf * 4, 4,
                                 static_cast<size_t>(round_up(S->natoms, 64)) * 4};
        void* ptrs[5];
        for (int k = 0; k < 5; ++k) {
          if ((rc = tdmd_malloc(&p, sizes[k]))) return rc;
          S->allocs.push_back(p);
          ptrs[k] = p;
        }
        S->a.hj = static_cast<const int32_t*>(ptrs[0]);
        S->a.hn = static_cast<const int32_t*>(ptrs[1]);
        S->a.hmode = static_cast<const int32_t*>(ptrs[2]);
        d_halo_done = static_cast<int32_t*>(ptrs[3]);
        S->a.cntc = static_cast<int32_t*>(ptrs[4]);
        TDMD_HIP_TRY(hipMemset(ptrs[2], 0xff, sizes[2]));  // no halo yet: not staged
        TDMD_HIP_TRY(hipMemset(d_halo_done, 0, 4));
        S->stage_ok = true;
      }
    }
    set_path(S->lanes);
    // default group: four slots in mixed precision, eight in FP64, the
    // faster shape of each on the 1M-atom EAM state (mixed force pass 108 us
    // with four against 111 with eight; FP64 305 us with eight against 317)
    configure(S->cfg.pair_unroll != 0 ? S->cfg.pair_unroll : (std::is_same_v<R, float> ? 4 : 8),
              S->cfg.lds_budget);
    return TDMD_OK;
  }

  // Halos of the staged passes, after a rebuild (returns at once otherwise).
  void halo(hipStream_t s) {
    if (!stage) return;
    const int grid = std::max(1, std::min(S->nb_force, 2 * std::max(ncu, 1)));
    k_halo<<<grid, kHaloBlock, 0, s>>>(S->a, (S->natoms + kHaloBlock - 1) / kHaloBlock,
                                       d_halo_done);
    ++S->launches;
  }

  void shape(int32_t* out) const override {
    out[0] = S->lanes;
    out[1] = lds ? unroll : kPairUnroll;
    out[2] = lds ? budget : 0;
  }

  // The force-path passes of one step with the force-only epilogue: they
  // rewrite M2 and F from the current positions and change nothing else.
  void probe_passes(hipStream_t s) {
    if (S->kind == 1) density<false>(s);
    force<kForceOnly, false>(s);
  }

  int tune(int iters, int32_t* out) override {
    // Candidates: lanes per row {1, 4, 8}; with one lane and single-element
    // tables the LDS passes, in two pipelined group sizes (and, without
    // halo staging, two spline-window budgets).
    struct Cand {
      int lanes, u, b;
    };
    std::vector<Cand> cands;
    if (lds_ok) {
      cands.push_back({1, 8, lds_limit});
      cands.push_back({1, 4, lds_limit});
      if (!S->stage_ok) {
        cands.push_back({1, 8, 80 * 1024 - 1024});
        cands.push_back({1, 4, 80 * 1024 - 1024});
      }
    } else {
      cands.push_back({1, 0, 0});
    }
    cands.push_back({4, 0, 0});
    cands.push_back({8, 0, 0});
    hipStream_t s = S->stream;
    hipEvent_t e0, e1;
    TDMD_HIP_TRY(hipEventCreate(&e0));
    TDMD_HIP_TRY(hipEventCreate(&e1));
    const Cand start{S->lanes, lds ? unroll : 0, lds ? budget : 0};
    std::vector<float> times;
    for (const Cand& c : cands) {
      if (int rc = apply_shape(c.lanes, c.u, c.b, s)) return rc;
      for (int k = 0; k < 2; ++k) probe_passes(s);
      TDMD_HIP_TRY(hipEventRecord(e0, s));
      for (int k = 0; k < iters; ++k) probe_passes(s);
      TDMD_HIP_TRY(hipEventRecord(e1, s));
      TDMD_HIP_TRY(hipEventSynchronize(e1));
      TDMD_LAUNCH_CHECK();
      float ms = 0.0f;
      TDMD_HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
      times.push_back(ms);
    }
    // the fastest shape; the starting shape when it is within 1 % of it
    size_t k_best = 0;
    for (size_t k = 1; k < cands.size(); ++k)
      if (times[k] < times[k_best]) k_best = k;
    Cand pick = cands[k_best];
    for (size_t k = 0; k < cands.size(); ++k) {
      const Cand& c = cands[k];
      const bool is_start =
          c.lanes == start.lanes && (c.lanes != 1 || !lds_ok || (c.u == start.u && c.b == start.b));
      if (is_start && times[k] <= 1.01f * times[k_best]) pick = c;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (int rc = apply_shape(pick.lanes, pick.u, pick.b, s)) return rc;
    // M2 and F as the chosen shape computes them, so the trajectory goes on
    // exactly as it would have with that shape (bitwise unchanged when the
    // choice is the starting shape)
    probe_passes(s);
    TDMD_LAUNCH_CHECK();
    out[0] = lds ? unroll : kPairUnroll;
    out[1] = lds ? budget : 0;
    return TDMD_OK;
  }

  // Switch the kernel shape (tuner): path, group size, window budget. A
  // switch to the staged passes rebuilds the halos of the current rows.
  int apply_shape(int lanes, int u, int b, hipStream_t s) {
    const bool was_staged = stage;
    set_path(lanes);
    if (lds) configure(u, b);
    if (stage && !was_staged) {
      TDMD_HIP_TRY(hipMemsetAsync(S->a.flags + 4, 0xff, 4, s));  // halos due
      halo(s);
      TDMD_LAUNCH_CHECK();
    }
    return TDMD_OK;
  }

  template <bool kEnergy, bool kWin, int kU, bool kSt, bool kIs>
  void density_go(hipStream_t s) {
    go(k_eam_density_lds<R, Mir, kEnergy, kWin, kU, kSt, kIs>, lds_grid, kBigBlock,
       b_dens[kEnergy] + (kSt ? stage_bytes() : 0), s, S->a, meta(), coeff(), rc_sq(),
       w_dens[kEnergy], S->nb_force);
  }
  template <bool kEnergy, bool kWin, int kU>
  void density_lds(hipStream_t s) {
    if constexpr (kCanStage) {
      if (stage) {
        iso ? density_go<kEnergy, kWin, kU, true, true>(s)
            : density_go<kEnergy, kWin, kU, true, false>(s);
        return;
      }
      if (iso) {
        density_go<kEnergy, kWin, kU, false, true>(s);
        return;
      }
    }
    density_go<kEnergy, kWin, kU, false, false>(s);
  }
  bool few() const { return S->lanes == 8 && S->natoms <= kFewMax; }

  template <bool kEnergy>
  void density(hipStream_t s) {
    if (!lds) {
      const int nb = S->nblocks;
      if (few() && !kEnergy)
        go(k_eam_density<R, Mir, false, 8, true>, nb * 8, kBlock, 0, s, S->a, meta(), coeff(),
           rc_sq());
      else if (S->lanes == 8)
        go(k_eam_density<R, Mir, kEnergy, 8>, nb * 8, kBlock, 0, s, S->a, meta(), coeff(),
           rc_sq());
      else if (S->lanes == 4)
        go(k_eam_density<R, Mir, kEnergy, 4>, nb * 4, kBlock, 0, s, S->a, meta(), coeff(),
           rc_sq());
      else
        go(k_eam_density<R, Mir, kEnergy, 1>, nb, kBlock, 0, s, S->a, meta(), coeff(),
           rc_sq());
      return;
    }
    const bool win = w_dens[kEnergy].k_lo > 0;
    if (unroll == 8)
      win ? density_lds<kEnergy, true, 8>(s) : density_lds<kEnergy, false, 8>(s);
    else
      win ? density_lds<kEnergy, true, 4>(s) : density_lds<kEnergy, false, 4>(s);
  }

  template <int kEpi, bool kEnergy, bool kWin, int kU, bool kSt, bool kIs>
  void force_go(hipStream_t s) {
    go(k_eam_force_lds<R, Mir, kEpi, kEnergy, kWin, kU, kSt, kIs>, lds_grid, kBigBlock,
       b_force[kEnergy] + (kSt ? stage_bytes() : 0), s, S->a, meta(), coeff(), rc_sq(),
       w_force[kEnergy], S->nb_force);
  }
  template <int kEpi, bool kEnergy, bool kWin, int kU>
  void force_lds(hipStream_t s) {
    if constexpr (kCanStage) {
      if (stage) {
        iso ? force_go<kEpi, kEnergy, kWin, kU, true, true>(s)
            : force_go<kEpi, kEnergy, kWin, kU, true, false>(s);
        return;
      }
      if (iso) {
        force_go<kEpi, kEnergy, kWin, kU, false, true>(s);
        return;
      }
    }
    force_go<kEpi, kEnergy, kWin, kU, false, false>(s);
  }

  template <int kEpi, bool kEnergy, bool kMulti>
  void eam_force_global(hipStream_t s) {
    const int nb = S->nblocks;
    if constexpr (!kMulti && !kEnergy) {
      if (few()) {
        go(k_eam_force<R, Mir, kEpi, false, false, 8, true>, nb * 8, kBlock, 0, s, S->a, meta(),
           coeff(), rc_sq());
        return;
      }
    }
    if (S->lanes == 8)
      go(k_eam_force<R, Mir, kEpi, kEnergy, kMulti, 8>, nb * 8, kBlock, 0, s, S->a, meta(),
         coeff(), rc_sq());
    else if (S->lanes == 4)
      go(k_eam_force<R, Mir, kEpi, kEnergy, kMulti, 4>, nb * 4, kBlock, 0, s, S->a, meta(),
         coeff(), rc_sq());
    else
      go(k_eam_force<R, Mir, kEpi, kEnergy, kMulti, 1>, nb, kBlock, 0, s, S->a, meta(),
         coeff(), rc_sq());
  }

  template <int kEpi, bool kEnergy>
  void force(hipStream_t s) {
    const int nb = S->nblocks;
    if (S->kind == 1) {
      const bool win = w_force[kEnergy].k_lo > 0;
      if (lds && unroll == 8)
        win ? force_lds<kEpi, kEnergy, true, 8>(s) : force_lds<kEpi, kEnergy, false, 8>(s);
      else if (lds)
        win ? force_lds<kEpi, kEnergy, true, 4>(s) : force_lds<kEpi, kEnergy, false, 4>(s);
      else if (S->tables->ntypes > 1)
        eam_force_global<kEpi, kEnergy, true>(s);
      else
        eam_force_global<kEpi, kEnergy, false>(s);
    } else {
      if (few() && !kEnergy)
        go(k_morse_force<R, Mir, kEpi, false, 8, true>, nb * 8, kBlock, 0, s, S->a, mp());
      else if (S->lanes == 8)
        go(k_morse_force<R, Mir, kEpi, kEnergy, 8>, nb * 8, kBlock, 0, s, S->a, mp());
      else if (S->lanes == 4)
        go(k_morse_force<R, Mir, kEpi, kEnergy, 4>, nb * 4, kBlock, 0, s, S->a, mp());
      else
        go(k_morse_force<R, Mir, kEpi, kEnergy, 1>, nb, kBlock, 0, s, S->a, mp());
      if constexpr (kEpi == kFullKickDrift) {
        // the epilogue wrote the next step's records into M2: it is now M
        std::swap(S->a.M, S->a.M2);
        S->rec_swapped = !S->rec_swapped;
      }
    }
  }

  // Conditional rebuild: one fused launch, or the separate kernels.
  // forced: rebuild whatever the flag says (the fused kernel takes it as an
  // argument; the separate kernels need the flag raised first)
  int rebuild(hipStream_t s, bool forced) {
    if (S->nb_rebuild > 0) {
      k_rebuild_fused<R, Mir><<<S->nb_rebuild, kRebuildBlock, 0, s>>>(
          S->a, S->g, S->t, S->r_list * S->r_list, S->cutoff * S->cutoff,
          const_cast<int32_t*>(S->a.nbr), const_cast<int32_t*>(S->a.cnt), S->d_bar,
          S->d_rebuilds, forced ? 1 : 0);
      ++S->launches;  // the fused kernel also builds the halos
      TDMD_LAUNCH_CHECK();
      return TDMD_OK;
    }
    const int rc = sort_pass(s);
    return rc ? rc : fill_pass(s);
  }

  int sort_pass(hipStream_t s) override {
    const int gb = grid_for(S->natoms), gc = grid_for(S->g.ncells);
    k_bin<Mir><<<gb, kBlock, 0, s>>>(S->a, S->g);
    k_cell_scan<<<1, 1024, 0, s>>>(S->a.flags, S->g);
    k_scatter<<<gb, kBlock, 0, s>>>(S->a, S->g);
    k_order_permute<R, Mir><<<S->g.list_lanes > 0 ? gb : grid_for(S->g.ncells, kBlock / 64),
                              kBlock, 0, s>>>(S->a, S->g, S->t);
    k_copyback<R, Mir><<<gb, kBlock, 0, s>>>(S->a, S->g, S->t);
    k_zero_cells<<<gc, kBlock, 0, s>>>(S->a.flags, S->g);
    S->launches += 6;
    TDMD_LAUNCH_CHECK();
    return TDMD_OK;
  }
  // Counts (into *d_max) or rows of the sorted atoms.
  template <bool kCount>
  void nlist(hipStream_t s, int32_t* d_max) {
    auto go = [&](auto kernel, int grid, int block) {
      kernel<<<grid, block, 0, s>>>(S->a, S->g, S->t, S->r_list * S->r_list,
                                    S->cutoff * S->cutoff,
                                    kCount ? nullptr : const_cast<int32_t*>(S->a.nbr),
                                    kCount ? nullptr : const_cast<int32_t*>(S->a.cnt), d_max);
    };
    if (S->g.list_lanes == 0)
      go(&k_nlist_ell<kCount, Mir>, std::min(256, (S->g.ncells + 1) / 2), kListBlock);
    else if (S->g.list_lanes == 1)
      go(&k_nlist_atoms<kCount, 1, Mir>, grid_for(S->natoms), kBlock);
    else
      go(&k_nlist_atoms<kCount, 32, Mir>, grid_for(32 * static_cast<int64_t>(S->natoms)), kBlock);
  }
  int fill_pass(hipStream_t s) override {
    const int gb = grid_for(S->natoms);
    nlist<false>(s, nullptr);
    k_rebuild_done<<<gb, kBlock, 0, s>>>(S->a.flags, S->g.done, gb, S->d_rebuilds);
    S->launches += 2;
    halo(s);
    TDMD_LAUNCH_CHECK();
    return TDMD_OK;
  }
  int count_pass(hipStream_t s, int32_t* d_max) override {
    nlist<true>(s, d_max);
    TDMD_LAUNCH_CHECK();
    return TDMD_OK;
  }
  int write_mirror(hipStream_t s) override {
    k_write_mirror<Mir><<<grid_for(S->natoms), kBlock, 0, s>>>(S->a);
    TDMD_LAUNCH_CHECK();
    return TDMD_OK;
  }
  int energy_pass(hipStream_t s, double* d_out) override {
    const int nb = S->nb_force;
    if (S->kind == 1) {
      density<true>(s);
      launch_sum_partials(S->a.partials, nb, d_out + 0, 0, s);
    } else {
      tdmd_fill_u32(d_out, 0u, 2, s);
    }
    force<kForceOnly, true>(s);
    launch_sum_partials(S->a.partials, nb, d_out + 1, 0, s);
    launch_sum_partials(S->a.partials_w, nb, d_out + 3, 0, s);
    k_ke_partials<R><<<grid_for(S->natoms), kBlock, 0, s>>>(S->a);
    launch_sum_partials(S->a.partials, grid_for(S->natoms), d_out + 2, 0, s);
    TDMD_LAUNCH_CHECK();
    return TDMD_OK;
  }

  int launch(char op, hipStream_t s) override {
    const int nb = S->nblocks;
    const int gb = grid_for(S->natoms);
    switch (op) {
      case OP_BOOT:
        k_kick_drift<R, Mir, false, false><<<nb, kBlock, 0, s>>>(S->a);
        break;
      case OP_KD_FULL:
        go(k_kick_drift<R, Mir, false, true>, nb, kBlock, 0, s, S->a);
        break;
      case OP_KD_NVT:
        k_kick_drift<R, Mir, true, false><<<nb, kBlock, 0, s>>>(S->a);
        break;
      case OP_KD_NVT2:
        k_kick_drift<R, Mir, true, false, true><<<nb, kBlock, 0, s>>>(S->a);
        break;
      case OP_NVT_PRE:
        k_nhc_pre<<<1, 64, 0, s>>>(S->a.nhc, S->nhcp);
        break;
      case OP_NVT_POST:
        k_nhc_post<false><<<1, 256, 0, s>>>(S->a.nhc, S->a.partials, S->nb_force, S->nhcp);
        break;
      case OP_NVT_POST_PRE:
        k_nhc_post<true><<<1, 256, 0, s>>>(S->a.nhc, S->a.partials, S->nb_force, S->nhcp);
        break;
      case OP_NVT_FINAL:
        k_scale_v<<<gb, kBlock, 0, s>>>(S->a);
        k_nhc_commit<<<1, 64, 0, s>>>(S->a.nhc);
        ++S->launches;
        break;
      case OP_REB_FORCED: {
        if (S->nb_rebuild == 0) {
          k_set_flag<<<1, 64, 0, s>>>(S->a.flags);
          ++S->launches;
        }
        return rebuild(s, true);
      }
      case OP_REB_COND:
        return rebuild(s, false);
      case OP_DENS:
        density<false>(s);
        break;
      case OP_F_FULL:
        force<kFullKickDrift, false>(s);
        break;
      case OP_F_ONLY:
        force<kForceOnly, false>(s);
        break;
      case OP_F_HALF:
        force<kHalfKick, false>(s);
        break;
      case OP_F_KICK2:
        force<kKick2Ke, false>(s);
        break;
      case OP_F_KE:
        force<kKe, false>(s);
        break;
      default:
        return fail(TDMD_E_STATE, std::string("scheduler: unknown op ") + op);
    }
    ++S->launches;
    TDMD_LAUNCH_CHECK();
    return TDMD_OK;
  }
};

// One per unit.
EngineBase* make_engine_fixed(tdmd_sched* s);        // mixed, 32-bit fixed-point records
EngineBase* make_engine_mixed_f64(tdmd_sched* s);    // mixed, FP64 records
EngineBase* make_engine_fp64(tdmd_sched* s);
EngineBase* make_engine_batch_fixed(tdmd_sched* s);  // the same for batches of boxes
EngineBase* make_engine_batch_mixed_f64(tdmd_sched* s);
EngineBase* make_engine_batch_fp64(tdmd_sched* s);

}  // namespace tdmd_hip
