// scheduler.cpp -- FastPipelineScheduler on gfx950
// (src/scheduler/fast_pipeline_scheduler.cuh:36-192,
//  src/scheduler/fast_pipeline_scheduler.cu:15-232).
//
// Same contract as the reference: construct with a box, an atom count and a
// potential; upload; run_until(step) (velocity Verlet with the cross-step
// fused kick, one stream, one synchronisation per call); download in upload
// order. Re-designed underneath:
//   * atoms are kept in a Morton-ordered cell sort, re-derived at each
//     neighbour rebuild on the device (no host round trip, no
//     cudaDeviceSynchronize -- compare device_cell_list.cu:103-111,148);
//   * neighbour lists are wave-interleaved (ELL) for coalesced reads;
//   * EAM runs as two passes per step: density+embedding, then force with
//     the next step's kick and drift fused into its epilogue;
//   * the rebuild trigger is decided on the device (fixed interval as the
//     reference, or max displacement > skin/2), so whole step sequences are
//     captured once as hipGraphs and replayed;
//   * NVT (Nose-Hoover chain, device_nose_hoover.cu:187-289) runs on the
//     device with the KE reduced from the kick epilogue's block partials.
#include "sched_engine.hpp"

namespace tdmd_hip {

int read_setfl(const std::string& path, SetflData* out);

namespace {

using namespace sched;

uint32_t spread3(uint32_t v) {
  uint32_t r = 0;
  for (int b = 0; b < 10; ++b) r |= ((v >> b) & 1u) << (3 * b);
  return r;
}

// Destroys every captured graph (the caller has synchronised the stream).
void drop_graphs(tdmd_sched* S) {
  for (auto& kv : S->graphs) (void)hipGraphExecDestroy(kv.second);
  for (auto& kv : S->graph_defs) (void)hipGraphDestroy(kv.second);
  S->graphs.clear();
  S->graph_defs.clear();
  S->graph_kernels.clear();
  S->graph_swaps.clear();
}

template <class T>
int dalloc(tdmd_sched* S, T** p, size_t n) {
  void* q = nullptr;
  const int rc = tdmd_malloc(&q, std::max<size_t>(n, 1) * sizeof(T));
  if (rc) return rc;
  S->allocs.push_back(q);
  *p = static_cast<T*>(q);
  return TDMD_OK;
}

// How a download reaches the host, by its bytes. Up to kStageSmall, one transfer
// into a pinned buffer and a copy out of it (4,000 atoms: 54 us; 150 as three
// transfers into pageable memory). Up to kStageLarge, straight into the caller's
// arrays: 32,000 atoms take 140 us either way, and pinning 2.3 MB once takes
// 440. Beyond, through kStageLarge of pinned memory by kCopyThreads threads: one
// copies at 14 GB/s where the transfer runs at 56 (1,048,576 atoms: 5.2 ms with
// one, 2.8 with four, 18 straight into fresh pages).
constexpr size_t kStageSmall = size_t{512} << 10;
constexpr size_t kStageLarge = size_t{8} << 20;
constexpr int kCopyThreads = 4;

// The state in upload order, as (x, y, z) triples: positions, velocities,
// forces, N triples each. Scattered triples of whole sectors, bound by HBM:
// 1,048,576 atoms take 62 us. (A whole download with ten transfers of single
// components, scattered by the host: 139 us for 256 atoms, 252 for 4,000, 278
// for 32,000, 3.7 ms for 256,000 in FP64, 20.6 for 1,048,576; now 38, 53, 149,
// 1.0 and 2.8.)
template <class R>
__global__ void __launch_bounds__(256)
k_upload_order(StepArgs a, const int32_t* orig, double* out) {
  const int s = blockIdx.x * 256 + threadIdx.x;
  const size_t n = static_cast<size_t>(a.natoms);
  if (s >= a.natoms) return;
  const size_t o = 3 * static_cast<size_t>(orig[s]);
  out[o] = a.px[s];
  out[o + 1] = a.py[s];
  out[o + 2] = a.pz[s];
  out[3 * n + o] = a.vx[s];
  out[3 * n + o + 1] = a.vy[s];
  out[3 * n + o + 2] = a.vz[s];
  out[6 * n + o] = static_cast<double>(static_cast<const R*>(a.fx)[s]);
  out[6 * n + o + 1] = static_cast<double>(static_cast<const R*>(a.fy)[s]);
  out[6 * n + o + 2] = static_cast<double>(static_cast<const R*>(a.fz)[s]);
}

// The stream's device as the calling thread's, for a scope: a download may be
// called from a thread that has another device current.
class StreamDevice {
 public:
  explicit StreamDevice(hipStream_t s) {
    int dev = 0;
    if (hipGetDevice(&before_) == hipSuccess && hipStreamGetDevice(s, &dev) == hipSuccess &&
        dev != before_)
      changed_ = hipSetDevice(dev) == hipSuccess;
  }
  ~StreamDevice() {
    if (changed_) (void)hipSetDevice(before_);
  }
  StreamDevice(const StreamDevice&) = delete;
  StreamDevice& operator=(const StreamDevice&) = delete;

 private:
  int before_ = 0;
  bool changed_ = false;
};

// Doubles [from, to) of the scratch block to the host by way of the staging
// buffer; the block holds dst[0..2], 3 N doubles each (null: not wanted).
int staged_download(const tdmd_sched* S, double* const dst[3], size_t from, size_t to) {
  const size_t N = static_cast<size_t>(S->natoms);
  const double* const out = S->t.px;
  const int parts = (to - from) * 8 <= kStageSmall ? 1 : kCopyThreads;
  if (!S->h_stage) {  // enough for any download of this scheduler
    const size_t bytes = 72 * N <= kStageSmall ? 72 * N : kStageLarge;
    TDMD_HIP_TRY(hipHostMalloc(reinterpret_cast<void**>(&S->h_stage), bytes, 0));
  }
  for (int t = 0; t < parts; ++t)
    if (!S->ev_stage[t])
      TDMD_HIP_TRY(hipEventCreateWithFlags(&S->ev_stage[t], hipEventDisableTiming));
  // every `parts`-th chunk through part t of the buffer
  const size_t chunk = (parts == 1 ? kStageSmall : kStageLarge / kCopyThreads) / 8;
  auto copy = [&](int t) -> int {
    double* const stage = S->h_stage + t * chunk;
    for (size_t b = from + t * chunk; b < to; b += parts * chunk) {
      const size_t e = std::min(to, b + chunk);
      TDMD_HIP_TRY(hipMemcpyAsync(stage, out + b, (e - b) * 8, hipMemcpyDeviceToHost, S->stream));
      TDMD_HIP_TRY(hipEventRecord(S->ev_stage[t], S->stream));
      TDMD_HIP_TRY(hipEventSynchronize(S->ev_stage[t]));
      for (size_t k = 0; k < 3; ++k) {
        const size_t lo = std::max(b, 3 * N * k), hi = std::min(e, 3 * N * (k + 1));
        if (dst[k] && lo < hi)
          std::memcpy(dst[k] + (lo - 3 * N * k), stage + (lo - b), (hi - lo) * 8);
      }
    }
    return TDMD_OK;
  };
  int dev = 0;
  TDMD_HIP_TRY(hipGetDevice(&dev));
  int rc[kCopyThreads] = {};
  std::thread th[kCopyThreads];
  for (int t = 1; t < parts; ++t) {
    auto work = [&copy, &rc, dev, t] {
      rc[t] = hipSetDevice(dev) == hipSuccess ? copy(t) : TDMD_E_HIP;
    };
    try {
      th[t] = std::thread(work);
    } catch (...) {  // no thread, or no memory for one, to be had
      rc[t] = copy(t);
    }
  }
  rc[0] = copy(0);
  for (auto& t : th)
    if (t.joinable()) t.join();
  for (int r : rc)
    if (r) return r == rc[0] ? r : fail(r, "sched_download: copy to the host failed");
  return TDMD_OK;
}

// How the lists are searched (GridArgs::list_lanes): by cells where cells hold
// enough atoms on average, else by atoms, as many lanes each as the rebuild's grid
// gives them. A cell costs a team of the workgroup about the same whatever it
// holds, so the search by cells is slow where they are nearly empty: vacuum around
// a droplet, a gas. Rebuilds in us, by cells / 32 lanes / 1 lane, mixed, by random
// atoms a cell:
//                              8                 4                 2
//   fixed        4,096    44 / 53 / 173     44 / 48 / 99      53 / 49 / 97
//                64,000  116 / 210 / 180   151 / 208 / 129   223 / 206 / 124
//               125,000  172 / 361 / 183   234 / 363 / 134   389 / 362 / 130
//               262,144  294 / 672 / 195   445 / 678 / 150   765 / 672 / 152
//                        (20: 273 / 681 / 306, 12: 282 / 677 / 244)
//   displacement  4,096  231 / 606 / 164   386 / 605 / 90    615 / 590 / 89
//                        (20: 208 / 794 / 303)
//   split        32,768   67 / 103 / 115    89 / 107 / 90    142 / 118 / 99
//   4,096 atoms of a solid in the middle of a box six times as wide, fixed:
//   124 / 63 / 257; 262,144 in a box twice as wide: 907 / 683 / 328.
// FP64 records in boxes of under three cells of r_list on a periodic axis are
// searched from memory in any case, and by atoms faster (fixed, FP64: 500 atoms
// 63 / 45 / 208, films of 57,600 atoms 311 / 235 / 391, 160,000 1012 / 815 / 377,
// 500 boxes of 108 atoms 606 / 339 / 176).
int list_lanes(const tdmd_sched* S) {
  const int n = S->natoms;
  const bool split = S->cfg.split_rebuild != 0;
  const bool few = S->cfg.rebuild_policy == TDMD_REBUILD_DISPLACEMENT && !split;
  const int by_atoms = !few && n <= (split ? 16384 : 65536) ? 32 : 1;
  const int per_cell = by_atoms == 32        ? 2
                       : few || n > 131072 ? 15
                       : n > 32768         ? 7
                                           : 4;
  if (n < static_cast<int64_t>(per_cell) * S->g.ncells) return by_atoms;
  if (S->cfg.precision == TDMD_MIXED && !S->cfg.mirror_fp64) return 0;
  int64_t narrow = S->g.images ? 0 : n;
  if (S->multibox) {
    narrow = 0;
    for (size_t b = 0; b < S->h_boxes.size(); ++b)
      if (!S->h_boxes[b].images) narrow += S->rep_off[b + 1] - S->rep_off[b];
  }
  return 4 * narrow > n ? by_atoms : 0;
}

int sched_alloc(tdmd_sched* S) {
  const int N = S->natoms;
  const size_t fsz = S->cfg.precision == TDMD_MIXED ? sizeof(float) : sizeof(double);
  StepArgs& a = S->a;
  int rc = 0;
  double** d9[9] = {&a.px, &a.py, &a.pz, &a.vx, &a.vy, &a.vz, &a.bx, &a.by, &a.bz};
  for (auto* p : d9)
    if ((rc = dalloc(S, p, N))) return rc;
  void** f3[3] = {&a.fx, &a.fy, &a.fz};
  for (auto* p : f3) {
    char* q;
    if ((rc = dalloc(S, &q, N * fsz))) return rc;
    *p = q;
  }
  int32_t* types;
  if ((rc = dalloc(S, &types, N))) return rc;
  a.types = types;
  double* masses;
  if ((rc = dalloc(S, &masses, 64))) return rc;
  a.masses = masses;
  const bool fixed = S->cfg.precision == TDMD_MIXED && !S->cfg.mirror_fp64;
  const size_t msz = fixed ? 16 : 32;
  // gathers address records by a 32-bit byte offset
  if (static_cast<uint64_t>(N) * msz >= (uint64_t{1} << 32))
    return fail(TDMD_E_INVALID, "scheduler: at most " + std::to_string((uint64_t{1} << 32) / msz - 1) +
                                    " atoms in one scheduler at this precision");
  char *M, *M2;
  if ((rc = dalloc(S, &M, N * msz))) return rc;
  if ((rc = dalloc(S, &M2, N * msz))) return rc;
  a.M = M;
  a.M2 = M2;
  if ((rc = dalloc(S, &a.flags, 8))) return rc;
  // room for the per-block partials of the widest pass (Morse rows split
  // over kSplitLanes lanes)
  if ((rc = dalloc(S, &a.partials, static_cast<size_t>(S->nblocks) * kSplitLanes + 64))) return rc;
  if ((rc = dalloc(S, &a.partials_w, static_cast<size_t>(S->nblocks) * kSplitLanes + 64))) return rc;
  if ((rc = dalloc(S, &a.nhc, 64))) return rc;
  int32_t* cnt;
  if ((rc = dalloc(S, &cnt, round_up(N, 64)))) return rc;
  a.cnt = cnt;
  if ((rc = dalloc(S, &a.cntn, round_up(N, 64)))) return rc;
  // permutation scratch, one block: a download gathers into it
  PermArgs& t = S->t;
  const size_t stride = round_up(N, 16);
  double* block;
  if ((rc = dalloc(S, &block, 9 * stride))) return rc;
  double** t6[6] = {&t.px, &t.py, &t.pz, &t.vx, &t.vy, &t.vz};
  for (int k = 0; k < 6; ++k) *t6[k] = block + k * stride;
  void** tf[3] = {&t.fx, &t.fy, &t.fz};
  for (int k = 0; k < 3; ++k) *tf[k] = block + (6 + k) * stride;
  if ((rc = dalloc(S, &t.types, N))) return rc;
  if ((rc = dalloc(S, &t.orig, N))) return rc;
  GridArgs& g = S->g;
  int32_t* rank_of;
  if ((rc = dalloc(S, &rank_of, g.ncells))) return rc;
  g.rank_of = rank_of;
  if ((rc = dalloc(S, &g.ccount, g.ncells))) return rc;
  if ((rc = dalloc(S, &g.cstart, static_cast<size_t>(g.ncells) + 1))) return rc;
  if ((rc = dalloc(S, &g.cursor, g.ncells))) return rc;
  if ((rc = dalloc(S, &g.key, N))) return rc;
  if ((rc = dalloc(S, &g.sidx, N))) return rc;
  if ((rc = dalloc(S, &g.orig, N))) return rc;
  if ((rc = dalloc(S, &g.done, 4))) return rc;
  if ((rc = dalloc(S, &g.wsum, sched::kMaxScanGroups))) return rc;
  if ((rc = dalloc(S, &S->d_maxcnt, 4))) return rc;
  if ((rc = dalloc(S, &S->d_rebuilds, 1))) return rc;
  if ((rc = dalloc(S, &S->d_scalars, 16))) return rc;
  if ((rc = dalloc(S, &S->d_bar, 1))) return rc;
  TDMD_HIP_TRY(hipMemset(S->d_bar, 0, sizeof(GridBarrier)));
  // Morton rank of every cell of each box's grid; a box's cells take the
  // global ranks [cell_off, cell_off + ncells_box), so the sort keeps every
  // box in its own slot range.
  std::vector<int32_t> h_rank(static_cast<size_t>(g.ncells));
  const int nbox = S->multibox ? static_cast<int>(S->h_boxes.size()) : 1;
  for (int b = 0; b < nbox; ++b) {
    const int* n = S->multibox ? S->h_boxes[static_cast<size_t>(b)].n : g.n;
    const int off = S->multibox ? S->h_boxes[static_cast<size_t>(b)].cell_off : 0;
    const int nc = n[0] * n[1] * n[2];
    std::vector<std::pair<uint32_t, int>> order(static_cast<size_t>(nc));
    for (int z = 0, c = 0; z < n[2]; ++z)
      for (int y = 0; y < n[1]; ++y)
        for (int x = 0; x < n[0]; ++x, ++c)
          order[static_cast<size_t>(c)] = {spread3(x) | (spread3(y) << 1) | (spread3(z) << 2), c};
    std::sort(order.begin(), order.end());
    for (int r = 0; r < nc; ++r)
      h_rank[static_cast<size_t>(off + order[static_cast<size_t>(r)].second)] = off + r;
  }
  TDMD_HIP_TRY(hipMemcpy(rank_of, h_rank.data(), h_rank.size() * 4, hipMemcpyHostToDevice));
  // The list search's stencil: for each cell (row = its rank), the ranks of
  // the 27 cells around it with periodic wrap, in increasing rank, the order
  // in which the search visits them (atoms are sorted by cell rank, so rows
  // come out in increasing atom index), and each entry's periodic image:
  // +L where the stencil wrapped past the upper face, -L past the lower.
  // When every periodic axis has at least 3 cells no smaller than r_list,
  // a pair within r_list lies in exactly one stencil entry, whose image is
  // its minimum image; the search then skips the per-candidate test.
  std::vector<int32_t> h_around(27 * static_cast<size_t>(g.ncells));
  std::vector<uint8_t> h_img(27 * static_cast<size_t>(g.ncells));
  bool images = true;
  for (int b = 0; b < nbox; ++b) {
    const int* n = S->multibox ? S->h_boxes[static_cast<size_t>(b)].n : g.n;
    const int off = S->multibox ? S->h_boxes[static_cast<size_t>(b)].cell_off : 0;
    const MirrorParams& mp = S->multibox ? S->h_boxes[static_cast<size_t>(b)].mp : S->a.mp;
    bool box_images = true;
    for (int d = 0; d < 3; ++d)
      box_images = box_images && (!mp.periodic[d] || (n[d] >= 3 && mp.L[d] / n[d] >= S->r_list));
    if (S->multibox) S->h_boxes[static_cast<size_t>(b)].images = box_images ? 1 : 0;
    images = images && box_images;
    for (int z = 0; z < n[2]; ++z)
      for (int y = 0; y < n[1]; ++y)
        for (int x = 0; x < n[0]; ++x) {
          std::pair<int32_t, uint8_t> e[27];
          for (int t = 0; t < 27; ++t) {
            const int c[3] = {x + t % 3 - 1, y + (t / 3) % 3 - 1, z + t / 9 - 1};
            int w[3];
            unsigned code = 0;
            for (int d = 0; d < 3; ++d) {
              w[d] = (c[d] + n[d]) % n[d];
              if (mp.periodic[d] && c[d] >= n[d]) code |= 1u << (2 * d);  // +L
              if (mp.periodic[d] && c[d] < 0) code |= 2u << (2 * d);      // -L
            }
            e[t] = {h_rank[static_cast<size_t>(off + (w[2] * n[1] + w[1]) * n[0] + w[0])],
                    static_cast<uint8_t>(code)};
          }
          std::sort(e, e + 27);
          const int own = h_rank[static_cast<size_t>(off + (z * n[1] + y) * n[0] + x)];
          for (int t = 0; t < 27; ++t) {
            h_around[27 * static_cast<size_t>(own) + t] = e[t].first;
            h_img[27 * static_cast<size_t>(own) + t] = e[t].second;
          }
        }
  }
  int32_t* around;
  if ((rc = dalloc(S, &around, h_around.size()))) return rc;
  TDMD_HIP_TRY(hipMemcpy(around, h_around.data(), h_around.size() * 4, hipMemcpyHostToDevice));
  g.around = around;
  uint8_t* img;
  if ((rc = dalloc(S, &img, h_img.size()))) return rc;
  TDMD_HIP_TRY(hipMemcpy(img, h_img.data(), h_img.size(), hipMemcpyHostToDevice));
  g.around_img = img;
  g.list_teams = 2;  // until the first count
  g.polls = sched::kBarrierPolls;
  g.images = images ? 1 : 0;  // batches: decided per box (BoxGeo::images)
  g.list_lanes = list_lanes(S);
  if (S->multibox) {
    BoxGeo* boxes;
    int32_t* rep;
    if ((rc = dalloc(S, &boxes, S->h_boxes.size()))) return rc;
    if ((rc = dalloc(S, &rep, N))) return rc;
    std::vector<int32_t> h_rep(static_cast<size_t>(N));
    for (size_t b = 0; b < S->h_boxes.size(); ++b)
      for (int i = S->rep_off[b]; i < S->rep_off[b + 1]; ++i) h_rep[static_cast<size_t>(i)] = static_cast<int32_t>(b);
    TDMD_HIP_TRY(hipMemcpy(boxes, S->h_boxes.data(), S->h_boxes.size() * sizeof(BoxGeo),
                           hipMemcpyHostToDevice));
    TDMD_HIP_TRY(hipMemcpy(rep, h_rep.data(), h_rep.size() * 4, hipMemcpyHostToDevice));
    a.boxes = boxes;
    a.rep = rep;
  }
  TDMD_HIP_TRY(hipMemset(g.ccount, 0, static_cast<size_t>(g.ncells) * 4));
  TDMD_HIP_TRY(hipMemset(g.cursor, 0, static_cast<size_t>(g.ncells) * 4));
  TDMD_HIP_TRY(hipMemset(g.done, 0, 16));
  TDMD_HIP_TRY(hipMemset(a.flags, 0, 32));
  TDMD_HIP_TRY(hipMemset(S->d_rebuilds, 0, 8));
  TDMD_HIP_TRY(hipMemset(a.nhc, 0, 64 * 8));
  const double one = 1.0;  // no pending chain scale
  TDMD_HIP_TRY(hipMemcpy(a.nhc + 24, &one, 8, hipMemcpyHostToDevice));
  TDMD_HIP_TRY(hipDeviceSynchronize());
  return TDMD_OK;
}

// Mirror parameters and binning grid of one box.
int setup_box(const tdmd_box& box, double r_list, double cell_min, MirrorParams* mp, int n[3],
              double inv_cs[3]) {
  for (int d = 0; d < 3; ++d) {
    mp->lo[d] = box.lo[d];
    mp->L[d] = box.hi[d] - box.lo[d];
    mp->hL[d] = 0.5 * mp->L[d];
    mp->periodic[d] = box.periodic[d] ? 1 : 0;
    if (!(mp->L[d] > 0)) return fail(TDMD_E_INVALID, "scheduler: box must have positive size");
  }
  // 32-bit fixed point (MirrorFixed): a periodic axis spans exactly 2^32
  // units; an open axis gets unit W 2^-30, W = max(L, r_list), so any listed
  // pair difference stays far below 2^31 units.
  for (int d = 0; d < 3; ++d) {
    const double W = mp->periodic[d] ? mp->L[d] : std::max(mp->L[d], r_list);
    const int e = mp->periodic[d] ? 32 : 30;
    mp->q[d] = std::ldexp(1.0, e) / W;
    mp->unit[d] = std::ldexp(W, -e);
  }
  // Binning grid: cells no smaller than cell_min >= r_list (with a relative
  // margin so rounding in the bin computation can never push a neighbour
  // out of the 27-cell stencil), at least 3 per axis (cell_list.cpp:22-27).
  for (int d = 0; d < 3; ++d) {
    n[d] = std::max(3, static_cast<int>(std::floor(mp->L[d] / (cell_min * (1.0 + 1e-9)))));
    inv_cs[d] = static_cast<double>(n[d]) / mp->L[d];
    if (n[d] > 1024) return fail(TDMD_E_INVALID, "scheduler: more than 1024 cells per axis");
  }
  return TDMD_OK;
}

// boxes.size() == 1 and !multibox: one system. multibox: a batch of
// independent boxes with counts[r] atoms each, concatenated in box order.
int sched_setup(tdmd_sched* S, const std::vector<tdmd_box>& boxes, const std::vector<int>& counts,
                const tdmd_sched_config& cfg, bool multibox) {
  int64_t total = 0;
  for (int c : counts) {
    if (c <= 0) return fail(TDMD_E_INVALID, "scheduler: natoms must be positive");
    total += c;
  }
  if (boxes.empty() || boxes.size() != counts.size() || total > (1LL << 30))
    return fail(TDMD_E_INVALID, "scheduler: bad box / atom counts");
  const int natoms = static_cast<int>(total);
  if (!(cfg.dt > 0) || !(cfg.r_skin >= 0) || cfg.rebuild_every < 1)
    return fail(TDMD_E_INVALID, "scheduler: bad dt / r_skin / rebuild_every");
  if (cfg.precision != TDMD_FP64 && cfg.precision != TDMD_MIXED)
    return fail(TDMD_E_INVALID, "scheduler: bad precision");
  if (cfg.t_target > 0 && (cfg.nhc_length < 1 || cfg.nhc_length > 8 || !(cfg.t_period > 0)))
    return fail(TDMD_E_INVALID, "scheduler: NHC chain length must be 1..8, t_period > 0");
  if (multibox && cfg.t_target > 0)
    return fail(TDMD_E_INVALID, "scheduler: a batch of boxes runs NVE (one thermostat per box "
                                "is not provided)");
  if (cfg.pair_unroll != 0 && cfg.pair_unroll != 4 && cfg.pair_unroll != 8)
    return fail(TDMD_E_INVALID, "scheduler: pair_unroll must be 0 (default), 4 or 8");
  if (cfg.lds_budget < 0) return fail(TDMD_E_INVALID, "scheduler: lds_budget must be >= 0");
  if (cfg.pair_lanes != 0 && cfg.pair_lanes != 1 && cfg.pair_lanes != 4 && cfg.pair_lanes != 8)
    return fail(TDMD_E_INVALID, "scheduler: pair_lanes must be 0 (by size), 1, 4 or 8");
  if (cfg.cell_pct != 0 && (cfg.cell_pct < 100 || cfg.cell_pct > 400))
    return fail(TDMD_E_INVALID, "scheduler: cell_pct must be 0 or 100..400");
  S->box = boxes[0];
  S->natoms = natoms;
  S->cfg = cfg;
  S->multibox = multibox;
  S->nblocks = round_up(grid_for(natoms), 8);
  S->r_list = S->cutoff + cfg.r_skin;
  GridArgs& g = S->g;
  const double cell_min = S->r_list * (cfg.cell_pct > 0 ? cfg.cell_pct : 100) / 100.0;
  int rc = setup_box(boxes[0], S->r_list, cell_min, &S->a.mp, g.n, g.inv_cs);
  if (rc) return rc;
  g.ncells = g.n[0] * g.n[1] * g.n[2];
  if (multibox) {
    S->h_boxes.resize(boxes.size());
    S->rep_off.assign(1, 0);
    int cells = 0;
    for (size_t b = 0; b < boxes.size(); ++b) {
      BoxGeo& bg = S->h_boxes[b];
      std::memset(&bg, 0, sizeof(bg));
      if ((rc = setup_box(boxes[b], S->r_list, cell_min, &bg.mp, bg.n, bg.inv_cs))) return rc;
      bg.cell_off = cells;
      cells += bg.n[0] * bg.n[1] * bg.n[2];
      S->rep_off.push_back(S->rep_off.back() + counts[b]);
    }
    g.ncells = cells;
  }
  S->a.natoms = natoms;
  S->a.ntypes = S->tables ? S->tables->ntypes : 1;
  if (S->a.ntypes < 1 || S->a.ntypes > kMaxTypes ||
      2 * S->a.ntypes + S->a.ntypes * (S->a.ntypes + 1) / 2 > kMaxSplines)
    return fail(TDMD_E_INVALID, "scheduler: 1..8 element types");
  S->a.nblocks = S->nblocks;
  S->a.dt = cfg.dt;
  S->a.skin_half_sq = 0.25 * cfg.r_skin * cfg.r_skin;
  S->nhcp.M = cfg.t_target > 0 ? cfg.nhc_length : 0;
  S->nhcp.n_dof = 3 * natoms - 3;  // pipeline_scheduler.cu:38
  S->nhcp.t_target = cfg.t_target;
  S->nhcp.t_period = cfg.t_period;
  S->nhcp.dt = cfg.dt;
  TDMD_HIP_TRY(hipStreamCreateWithFlags(&S->stream, hipStreamNonBlocking));
  rc = sched_alloc(S);
  if (rc) return rc;
  const bool fixed = cfg.precision == TDMD_MIXED && !cfg.mirror_fp64;
  if (multibox) {
    if (cfg.precision == TDMD_FP64)
      S->eng.reset(make_engine_batch_fp64(S));
    else if (fixed)
      S->eng.reset(make_engine_batch_fixed(S));
    else
      S->eng.reset(make_engine_batch_mixed_f64(S));
  } else if (cfg.precision == TDMD_FP64) {
    S->eng.reset(make_engine_fp64(S));
  } else if (fixed) {
    S->eng.reset(make_engine_fixed(S));
  } else {
    S->eng.reset(make_engine_mixed_f64(S));
  }
  return S->eng->init();
}

int sched_setup(tdmd_sched* S, const tdmd_box& box, int natoms, const tdmd_sched_config& cfg) {
  return sched_setup(S, std::vector<tdmd_box>{box}, std::vector<int>{natoms}, cfg, false);
}

void sched_free(tdmd_sched* S) {
  if (S->stream) (void)hipStreamSynchronize(S->stream);
  drop_graphs(S);
  for (void* p : S->allocs) (void)hipFree(p);
  if (S->a.nbr) (void)hipFree(const_cast<int32_t*>(S->a.nbr));
  if (S->a.nbr16) (void)hipFree(const_cast<uint16_t*>(S->a.nbr16));
  if (S->a.nbrc16) (void)hipFree(S->a.nbrc16);
  if (S->tables) eam_tables_destroy(S->tables);
  if (S->h_stage) (void)hipHostFree(S->h_stage);
  for (hipEvent_t e : S->ev_stage)
    if (e) (void)hipEventDestroy(e);
  if (S->stream) (void)hipStreamDestroy(S->stream);
}

// What a rebuild expects at its start, whatever the last one left: flags and
// cell counters clear, no arrivals at the barrier.
int clear_rebuild(tdmd_sched* S) {
  TDMD_HIP_TRY(hipMemset(S->d_bar, 0, sizeof(GridBarrier)));
  TDMD_HIP_TRY(hipMemset(S->g.ccount, 0, static_cast<size_t>(S->g.ncells) * 4));
  TDMD_HIP_TRY(hipMemset(S->g.cursor, 0, static_cast<size_t>(S->g.ncells) * 4));
  TDMD_HIP_TRY(hipMemset(S->a.flags, 0, 32));
  return TDMD_OK;
}

int check_flags(tdmd_sched* S) {
  int32_t f[4];
  TDMD_HIP_TRY(hipMemcpy(f, S->a.flags, 16, hipMemcpyDeviceToHost));
  if (f[3]) {
    // The rebuild stopped between phases: the atoms may be half permuted (and,
    // integrated on, non-finite: this flag comes first). The kernels have ended
    // (the stream was synchronised), so the counters are cleared here; the state
    // is unusable until the next upload.
    S->uploaded = false;
    S->initial_forces = false;
    if (const int rc = clear_rebuild(S)) return rc;
    return fail(TDMD_E_HIP, "scheduler: fused rebuild grid barrier timed out (workgroups not "
                            "co-resident); upload again, or use split_rebuild");
  }
  if (f[2])
    return fail(TDMD_E_NONFINITE,
                "scheduler: non-finite position, or an atom outside the representable range "
                "of an open axis (lo - 2W .. lo + 2W, W = max(box length, r_list))");
  if (f[1] > S->a.cap)
    return fail(TDMD_E_OVERFLOW, "scheduler: neighbour capacity " + std::to_string(S->a.cap) +
                                     " exceeded (max count " + std::to_string(f[1]) + ")");
  return TDMD_OK;
}

// log2 of the teams that a list search's workgroup may form for stencils of m
// atoms: a team has its share of the candidates (4,096) and of the mask words
// (8,192; m / 27 rows of m / 32 words), and what does not fit is searched from
// memory.
int list_teams(double m) {
  for (int t = 2; t > 0; --t)
    if (m <= 4096 >> t && m * m / (27 * 32) <= 8192 >> t) return t;
  return 0;
}

// First neighbour build: sort, count exactly, size the list, fill.
int first_build(tdmd_sched* S) {
  std::lock_guard<std::mutex> lock(S->scratch_mu);
  hipStream_t s = S->stream;
  k_set_flag<<<1, 64, 0, s>>>(S->a.flags);
  TDMD_LAUNCH_CHECK();
  int rc = S->eng->sort_pass(s);
  if (rc) return rc;
  TDMD_HIP_TRY(hipMemsetAsync(S->d_maxcnt, 0, 4, s));
  if ((rc = S->eng->count_pass(s, S->d_maxcnt))) return rc;
  int32_t maxc = 0;
  TDMD_HIP_TRY(hipMemcpyAsync(&maxc, S->d_maxcnt, 4, hipMemcpyDeviceToHost, s));
  TDMD_HIP_TRY(hipStreamSynchronize(s));
  int cap = S->cfg.max_neighbors > 0 ? S->cfg.max_neighbors
                                     : round_up(static_cast<int>(std::ceil(maxc * 1.25)) + 8, 4);
  cap = round_up(std::max(cap, kRowPad), kRowPad);  // rows are padded to kRowPad slots
  if (S->a.nbr == nullptr || cap > S->a.cap) {
    if (S->a.nbr) TDMD_HIP_TRY(hipFree(const_cast<int32_t*>(S->a.nbr)));
    if (S->a.nbr16) TDMD_HIP_TRY(hipFree(const_cast<uint16_t*>(S->a.nbr16)));
    if (S->a.nbrc16) TDMD_HIP_TRY(hipFree(S->a.nbrc16));
    S->a.nbr = nullptr;
    S->a.nbr16 = nullptr;
    S->a.nbrc16 = nullptr;
    const size_t slots = static_cast<size_t>(round_up(S->natoms, 64)) * cap;
    void* p = nullptr;
    if ((rc = tdmd_malloc(&p, slots * 4))) return rc;
    S->a.nbr = static_cast<int32_t*>(p);
    if (S->stage_ok) {  // 16-bit rows of the staged passes, full and cut
      if ((rc = tdmd_malloc(&p, slots * 2))) return rc;
      S->a.nbr16 = static_cast<uint16_t*>(p);
      if ((rc = tdmd_malloc(&p, slots * 2))) return rc;
      S->a.nbrc16 = static_cast<uint16_t*>(p);
    }
    S->a.cap = cap;
    drop_graphs(S);
  }
  // a stencil's candidates, from the longest row: the 27 cells against its sphere
  double cells = 27.0 * 3.0 / (4.0 * M_PI);
  for (int d = 0; d < 3; ++d) {
    double inv = S->multibox ? S->h_boxes[0].inv_cs[d] : S->g.inv_cs[d];
    if (S->multibox)
      for (const BoxGeo& b : S->h_boxes) inv = std::min(inv, b.inv_cs[d]);
    cells /= inv * S->r_list;
  }
  const int teams = list_teams(cells * (maxc + 1));
  if (teams != S->g.list_teams) {
    drop_graphs(S);  // captured graphs hold it
    S->g.list_teams = teams;
  }
  rc = S->eng->fill_pass(s);
  if (rc) return rc;
  ++S->host_rebuilds;
  return TDMD_OK;
}

int launch_ops(tdmd_sched* S, const std::string& ops, hipStream_t s) {
  for (char op : ops) {
    const int rc = S->eng->launch(op, s);
    if (rc) return rc;
  }
  return TDMD_OK;
}

// Enqueue a sequence of ops, as one cached graph when enabled.
int run_ops(tdmd_sched* S, const std::string& ops) {
  if (ops.empty()) return TDMD_OK;
  std::lock_guard<std::mutex> lock(S->scratch_mu);
  hipStream_t s = S->stream;
  if (!S->cfg.use_graph) return launch_ops(S, ops, s);
  // a graph holds the record buffers of the state it was captured in (and
  // the pass clock, when pass timing is on)
  const std::string key = ops + (S->rec_swapped ? "/1" : "/0") + (S->pass_timing ? "t" : "");
  auto it = S->graphs.find(key);
  if (it == S->graphs.end()) {
    const int64_t saved = S->launches;
    const bool swapped0 = S->rec_swapped;
    TDMD_HIP_TRY(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    {
      const int rc = launch_ops(S, ops, s);
      if (rc) {
        hipGraph_t dummy;
        (void)hipStreamEndCapture(s, &dummy);
        return rc;
      }
    }
    hipGraph_t gdef;
    TDMD_HIP_TRY(hipStreamEndCapture(s, &gdef));
    hipGraphExec_t exec;
    TDMD_HIP_TRY(hipGraphInstantiate(&exec, gdef, nullptr, nullptr, 0));
    S->graph_defs[key] = gdef;
    S->graph_kernels[key] = S->launches - saved;
    S->graph_swaps[key] = S->rec_swapped != swapped0;
    // capture enqueued nothing: back to the state before it, then replay
    if (S->graph_swaps[key]) {
      std::swap(S->a.M, S->a.M2);
      S->rec_swapped = swapped0;
    }
    it = S->graphs.emplace(key, exec).first;
    S->launches = saved;
  }
  S->launches += S->graph_kernels[key];  // kernels the graph replays
  if (S->graph_swaps[key]) {  // the replay leaves the records in the other buffer
    std::swap(S->a.M, S->a.M2);
    S->rec_swapped = !S->rec_swapped;
  }
  TDMD_HIP_TRY(hipGraphLaunch(it->second, s));
  ++S->graph_launches;
  return TDMD_OK;
}

int compute_initial_forces(tdmd_sched* S) {
  // fast_pipeline_scheduler.cu:168-193: build the list, compute F(t=0).
  int rc = first_build(S);
  if (rc) return rc;
  S->steps_since = 0;
  hipStream_t s = S->stream;
  if (S->kind == 1) {
    if ((rc = S->eng->launch(OP_DENS, s))) return rc;
  }
  if ((rc = S->eng->launch(OP_F_ONLY, s))) return rc;
  if (S->nhcp.M > 0) {
    // Stored KE of the uploaded velocities (the chain state was reset by
    // upload, with no pending scale).
    k_ke_partials<double><<<grid_for(S->natoms), kBlock, 0, s>>>(S->a);
    k_nhc_set_ke<<<1, 256, 0, s>>>(S->a.nhc, S->a.partials, grid_for(S->natoms), 0);
    TDMD_LAUNCH_CHECK();
  }
  S->initial_forces = true;
  return TDMD_OK;
}

constexpr int kChunk = 16;  // steps per captured graph

int run_window(tdmd_sched* S, int n) {
  // Step ops; the rebuild test happens after the kick-drift of each step
  // (fast_pipeline_scheduler.cu:101-166 + maybe_rebuild_nlist :225-232).
  const bool nvt = S->nhcp.M > 0;
  const bool eam = S->kind == 1;
  const bool disp = S->cfg.rebuild_policy == TDMD_REBUILD_DISPLACEMENT;
  std::vector<std::string> steps;
  steps.reserve(static_cast<size_t>(n));
  for (int k = 1; k <= n; ++k) {
    std::string st;
    if (nvt) {
      // later steps: the chain's pre half-step is fused into 'N', and the
      // previous step's closing half kick into this kick-drift
      if (k == 1) st += static_cast<char>(OP_NVT_PRE);
      st += static_cast<char>(k == 1 ? OP_KD_NVT : OP_KD_NVT2);
    } else if (k == 1) {
      st += static_cast<char>(OP_BOOT);
    }  // NVE: later steps' kick-drift is the previous force pass's epilogue
    if (disp) {
      st += static_cast<char>(OP_REB_COND);
    } else if (S->steps_since >= S->cfg.rebuild_every) {
      st += static_cast<char>(OP_REB_FORCED);
      S->steps_since = 0;
      ++S->host_rebuilds;
    }
    if (eam) st += static_cast<char>(OP_DENS);
    if (nvt) {
      // the window's last force pass stores the kicked velocities (the
      // window end scales them; the next window starts from them)
      st += static_cast<char>(k < n ? OP_F_KE : OP_F_KICK2);
      st += static_cast<char>(k < n ? OP_NVT_POST_PRE : OP_NVT_POST);
    } else if (k == n) {
      st += static_cast<char>(OP_F_HALF);
    } else {
      st += static_cast<char>(OP_F_FULL);
    }
    if (nvt && k == n) st += static_cast<char>(OP_NVT_FINAL);
    steps.push_back(st);
    ++S->steps_since;
    ++S->current_step;
    ++S->ticks;
  }
  for (size_t k = 0; k < steps.size(); k += kChunk) {
    std::string ops;
    for (size_t q = k; q < std::min(steps.size(), k + kChunk); ++q) ops += steps[q];
    const int rc = run_ops(S, ops);
    if (rc) return rc;
  }
  return TDMD_OK;
}

}  // namespace
}  // namespace tdmd_hip

using namespace tdmd_hip;

extern "C" {

void tdmd_sched_config_default(tdmd_sched_config* cfg) {
  std::memset(cfg, 0, sizeof(*cfg));
  cfg->dt = 0.001;  // FastPipelineConfig defaults, fast_pipeline_scheduler.cuh:42-46
  cfg->r_skin = 1.0;
  cfg->rebuild_every = 10;
  cfg->precision = TDMD_MIXED;
  cfg->rebuild_policy = TDMD_REBUILD_FIXED;
  cfg->t_target = 0.0;
  cfg->t_period = 0.1;
  cfg->nhc_length = 3;
  cfg->use_graph = 1;
  cfg->mirror_fp64 = 0;
}

int tdmd_sched_create_morse(tdmd_sched** out, const tdmd_box* box, int32_t natoms,
                            const tdmd_morse_params* params, const tdmd_sched_config* cfg) {
  if (!out || !box || !params || !cfg) return fail(TDMD_E_INVALID, "sched_create_morse: null");
  if (!(params->rc > 0)) return fail(TDMD_E_INVALID, "sched_create_morse: rc must be positive");
  auto* S = new tdmd_sched();
  S->kind = 0;
  S->morse = *params;
  S->cutoff = params->rc;  // fast_pipeline_scheduler.cu:23 (cutoff_ = params.rc)
  const int rc = sched_setup(S, *box, natoms, *cfg);
  if (rc) {
    sched_free(S);
    delete S;
    return rc;
  }
  *out = S;
  return TDMD_OK;
}

int tdmd_sched_create_eam(tdmd_sched** out, const tdmd_box* box, int32_t natoms, int32_t ntypes,
                          int32_t nrho, double drho, int32_t nr, double dr, double cutoff,
                          const double* F, const double* rho, const double* rphi,
                          const tdmd_sched_config* cfg) {
  if (!out || !box || !cfg || !F || !rho || !rphi)
    return fail(TDMD_E_INVALID, "sched_create_eam: null");
  if (ntypes < 1 || ntypes > sched::kMaxTypes)
    return fail(TDMD_E_INVALID, "sched_create_eam: 1..8 element types");
  auto* S = new tdmd_sched();
  S->kind = 1;
  int rc = tdmd_eam_tables_create(&S->tables, cfg->precision, ntypes, nrho, drho, nr, dr, cutoff,
                                  F, rho, rphi);
  if (rc) {
    delete S;
    return rc;
  }
  S->cutoff = cutoff;  // fast_pipeline_scheduler.cu:35 (cutoff_ = eam.cutoff())
  rc = sched_setup(S, *box, natoms, *cfg);
  if (rc) {
    sched_free(S);
    delete S;
    return rc;
  }
  *out = S;
  return TDMD_OK;
}

int tdmd_sched_create_eam_tables(tdmd_sched** out, const tdmd_box* box, int32_t natoms,
                                 const tdmd_eam_tables* tables, const tdmd_sched_config* cfg) {
  if (!out || !box || !cfg || !tables)
    return fail(TDMD_E_INVALID, "sched_create_eam_tables: null");
  if (tables->ntypes < 1 || tables->ntypes > sched::kMaxTypes)
    return fail(TDMD_E_INVALID, "sched_create_eam_tables: 1..8 element types");
  auto* S = new tdmd_sched();
  S->kind = 1;
  int rc = eam_tables_clone(tables, cfg->precision, &S->tables);
  if (rc) {
    delete S;
    return rc;
  }
  S->cutoff = tables->cutoff;
  rc = sched_setup(S, *box, natoms, *cfg);
  if (rc) {
    sched_free(S);
    delete S;
    return rc;
  }
  *out = S;
  return TDMD_OK;
}

int tdmd_sched_create_eam_batch(tdmd_sched** out, int32_t nrep, const tdmd_box* boxes,
                                const int32_t* natoms, int32_t ntypes, int32_t nrho, double drho,
                                int32_t nr, double dr, double cutoff, const double* F,
                                const double* rho, const double* rphi,
                                const tdmd_sched_config* cfg) {
  if (!out || !boxes || !natoms || !cfg || !F || !rho || !rphi || nrep < 1)
    return fail(TDMD_E_INVALID, "sched_create_eam_batch: bad arguments");
  if (ntypes < 1 || ntypes > sched::kMaxTypes)
    return fail(TDMD_E_INVALID, "sched_create_eam_batch: 1..8 element types");
  auto* S = new tdmd_sched();
  S->kind = 1;
  int rc = tdmd_eam_tables_create(&S->tables, cfg->precision, ntypes, nrho, drho, nr, dr, cutoff,
                                  F, rho, rphi);
  if (rc) {
    delete S;
    return rc;
  }
  S->cutoff = cutoff;
  rc = sched_setup(S, std::vector<tdmd_box>(boxes, boxes + nrep),
                   std::vector<int>(natoms, natoms + nrep), *cfg, true);
  if (rc) {
    sched_free(S);
    delete S;
    return rc;
  }
  *out = S;
  return TDMD_OK;
}

int tdmd_sched_create_morse_batch(tdmd_sched** out, int32_t nrep, const tdmd_box* boxes,
                                  const int32_t* natoms, const tdmd_morse_params* params,
                                  const tdmd_sched_config* cfg) {
  if (!out || !boxes || !natoms || !params || !cfg || nrep < 1)
    return fail(TDMD_E_INVALID, "sched_create_morse_batch: bad arguments");
  if (!(params->rc > 0)) return fail(TDMD_E_INVALID, "sched_create_morse_batch: rc must be > 0");
  auto* S = new tdmd_sched();
  S->kind = 0;
  S->morse = *params;
  S->cutoff = params->rc;
  const int rc = sched_setup(S, std::vector<tdmd_box>(boxes, boxes + nrep),
                             std::vector<int>(natoms, natoms + nrep), *cfg, true);
  if (rc) {
    sched_free(S);
    delete S;
    return rc;
  }
  *out = S;
  return TDMD_OK;
}

int tdmd_sched_autotune(tdmd_sched* S, int32_t iters, int32_t out[2]) {
  if (!S || !out || iters < 1) return fail(TDMD_E_INVALID, "sched_autotune: bad arguments");
  if (!S->uploaded) return fail(TDMD_E_STATE, "sched_autotune: upload first");
  if (!S->initial_forces) {
    const int rc = compute_initial_forces(S);
    if (rc) return rc;
  }
  const int rc = S->eng->tune(iters, out);
  if (rc) return rc;
  // captured graphs hold the previous kernel choice
  TDMD_HIP_TRY(hipStreamSynchronize(S->stream));
  drop_graphs(S);
  S->cfg.pair_unroll = out[0];
  S->cfg.lds_budget = out[1];
  S->cfg.pair_lanes = S->lanes;
  return check_flags(S);
}

int tdmd_sched_kernel_shape(const tdmd_sched* S, int32_t out[3]) {
  if (!S || !out || !S->eng) return fail(TDMD_E_INVALID, "sched_kernel_shape: null");
  S->eng->shape(out);
  return TDMD_OK;
}

int tdmd_sched_rebuild_barrier(tdmd_sched* S, int32_t polls, int32_t* workgroups) {
  if (!S) return fail(TDMD_E_INVALID, "sched_rebuild_barrier: null");
  if (workgroups) *workgroups = S->nb_rebuild;
  if (polls >= 0 && polls != S->g.polls) {
    // captured graphs hold the limit
    TDMD_HIP_TRY(hipStreamSynchronize(S->stream));
    drop_graphs(S);
    S->g.polls = polls;
  }
  return TDMD_OK;
}

int tdmd_sched_destroy(tdmd_sched* s) {
  if (!s) return TDMD_OK;
  sched_free(s);
  delete s;
  return TDMD_OK;
}

int tdmd_sched_upload(tdmd_sched* S, const double* pos, const double* vel, const double* forces,
                      const int32_t* types, const int32_t* ids, const double* masses,
                      int32_t n_masses) {
  if (!S || !pos || !vel || !types || !masses || n_masses < 2 || n_masses > 64)
    return fail(TDMD_E_INVALID, "sched_upload: bad arguments (masses indexed by 1-based type)");
  const int N = S->natoms;
  const int ntypes_max = S->kind == 1 ? S->tables->ntypes : n_masses - 1;
  for (int i = 0; i < N; ++i)
    if (types[i] < 1 || types[i] > ntypes_max || types[i] >= n_masses)
      return fail(TDMD_E_INVALID, "sched_upload: atom type out of range at index " +
                                      std::to_string(i));
  for (int k = 1; k < n_masses; ++k)
    if (!(masses[k] > 0)) return fail(TDMD_E_INVALID, "sched_upload: masses must be positive");
  S->h_types.assign(types, types + N);
  S->h_ids.assign(N, 0);
  if (ids) S->h_ids.assign(ids, ids + N);
  S->h_masses.assign(masses, masses + n_masses);
  const bool mixed = S->cfg.precision == TDMD_MIXED;
  std::vector<double> buf(static_cast<size_t>(N));
  std::vector<float> fbuf(static_cast<size_t>(N));
  double* pd[3] = {S->a.px, S->a.py, S->a.pz};
  double* vd[3] = {S->a.vx, S->a.vy, S->a.vz};
  void* fd[3] = {S->a.fx, S->a.fy, S->a.fz};
  for (int d = 0; d < 3; ++d) {
    for (int i = 0; i < N; ++i) buf[static_cast<size_t>(i)] = pos[3 * i + d];
    TDMD_HIP_TRY(hipMemcpy(pd[d], buf.data(), N * 8, hipMemcpyHostToDevice));
    for (int i = 0; i < N; ++i) buf[static_cast<size_t>(i)] = vel[3 * i + d];
    TDMD_HIP_TRY(hipMemcpy(vd[d], buf.data(), N * 8, hipMemcpyHostToDevice));
    for (int i = 0; i < N; ++i) buf[static_cast<size_t>(i)] = forces ? forces[3 * i + d] : 0.0;
    if (mixed) {
      for (int i = 0; i < N; ++i) fbuf[static_cast<size_t>(i)] = static_cast<float>(buf[static_cast<size_t>(i)]);
      TDMD_HIP_TRY(hipMemcpy(fd[d], fbuf.data(), N * 4, hipMemcpyHostToDevice));
    } else {
      TDMD_HIP_TRY(hipMemcpy(fd[d], buf.data(), N * 8, hipMemcpyHostToDevice));
    }
  }
  TDMD_HIP_TRY(hipMemcpy(const_cast<int32_t*>(S->a.types), types, N * 4, hipMemcpyHostToDevice));
  // captured graphs hold the kernel arguments, this flag among them
  const int one_type = std::all_of(types, types + N, [](int32_t t) { return t == 1; }) ? 1 : 0;
  if (one_type != S->a.one_type) {
    TDMD_HIP_TRY(hipStreamSynchronize(S->stream));
    drop_graphs(S);
    S->a.one_type = one_type;
  }
  std::vector<double> m64(64, 1.0);
  std::copy(masses, masses + n_masses, m64.begin());
  TDMD_HIP_TRY(hipMemcpy(const_cast<double*>(S->a.masses), m64.data(), 64 * 8, hipMemcpyHostToDevice));
  std::vector<int32_t> iota(static_cast<size_t>(N));
  std::iota(iota.begin(), iota.end(), 0);
  TDMD_HIP_TRY(hipMemcpy(S->g.orig, iota.data(), N * 4, hipMemcpyHostToDevice));
  if (const int rc = clear_rebuild(S)) return rc;
  std::vector<double> nhc0(64, 0.0);  // fresh chain, no pending scale
  nhc0[24] = 1.0;
  TDMD_HIP_TRY(hipMemcpy(S->a.nhc, nhc0.data(), 64 * 8, hipMemcpyHostToDevice));
  TDMD_HIP_TRY(hipDeviceSynchronize());
  const int rc = S->eng->write_mirror(S->stream);
  if (rc) return rc;
  TDMD_HIP_TRY(hipStreamSynchronize(S->stream));
  // fast_pipeline_scheduler.cu:70-72
  S->uploaded = true;
  S->initial_forces = false;
  S->current_step = 0;
  S->steps_since = 0;
  return TDMD_OK;
}

int tdmd_sched_run_until(tdmd_sched* S, int32_t target_step) {
  if (!S) return fail(TDMD_E_INVALID, "sched_run_until: null");
  if (!S->uploaded) return fail(TDMD_E_STATE, "sched_run_until: upload() first");
  int rc;
  if (!S->initial_forces && (rc = compute_initial_forces(S))) return rc;
  if (S->current_step < target_step) {
    rc = run_window(S, target_step - S->current_step);
    if (rc) return rc;
  }
  TDMD_HIP_TRY(hipStreamSynchronize(S->stream));
  return check_flags(S);
}

int tdmd_sched_download(const tdmd_sched* S, double* pos, double* vel, double* forces,
                        int32_t* types, int32_t* ids, int32_t natoms) {
  if (!S || natoms != S->natoms) return fail(TDMD_E_INVALID, "sched_download: natoms mismatch");
  if (!S->uploaded) return fail(TDMD_E_STATE, "sched_download: nothing uploaded");
  const size_t N = static_cast<size_t>(S->natoms);
  double* const dst[3] = {pos, vel, forces};
  int first = 0, last = 3;
  while (first < 3 && !dst[first]) ++first;
  while (last > first && !dst[last - 1]) --last;
  if (first < last) {
    // one download at a time, and none between the kernels of a rebuild that
    // another thread is enqueuing
    std::lock_guard<std::mutex> lock(S->scratch_mu);
    const StreamDevice device(S->stream);
    double* const out = S->t.px;
    const int nb = (S->natoms + 255) / 256;
    if (S->cfg.precision == TDMD_MIXED)
      k_upload_order<float><<<nb, 256, 0, S->stream>>>(S->a, S->g.orig, out);
    else
      k_upload_order<double><<<nb, 256, 0, S->stream>>>(S->a, S->g.orig, out);
    TDMD_HIP_TRY(hipGetLastError());
    const size_t from = 3 * N * static_cast<size_t>(first), to = 3 * N * static_cast<size_t>(last);
    const size_t bytes = (to - from) * 8;
    if (bytes > kStageSmall && bytes <= kStageLarge) {
      for (size_t k = 0; k < 3; ++k)
        if (dst[k])
          TDMD_HIP_TRY(hipMemcpyAsync(dst[k], out + 3 * N * k, 3 * N * 8, hipMemcpyDeviceToHost,
                                      S->stream));
      TDMD_HIP_TRY(hipStreamSynchronize(S->stream));
    } else if (const int rc = staged_download(S, dst, from, to)) {
      return rc;
    }
  }
  if (types) std::copy(S->h_types.begin(), S->h_types.end(), types);
  if (ids) std::copy(S->h_ids.begin(), S->h_ids.end(), ids);
  return TDMD_OK;
}

int tdmd_sched_stats(const tdmd_sched* S, int64_t out[4]) {
  if (!S || !out) return fail(TDMD_E_INVALID, "sched_stats: null");
  int64_t dev_rebuilds = 0;
  TDMD_HIP_TRY(hipMemcpy(&dev_rebuilds, S->d_rebuilds, 8, hipMemcpyDeviceToHost));
  out[0] = S->ticks;
  out[1] = S->launches;
  out[2] = dev_rebuilds;
  out[3] = S->graph_launches;
  return TDMD_OK;
}

int tdmd_sched_current_step(const tdmd_sched* S, int32_t* step) {
  if (!S || !step) return fail(TDMD_E_INVALID, "sched_current_step: null");
  *step = S->current_step;
  return TDMD_OK;
}

int tdmd_sched_interaction_cutoff(const tdmd_sched* S, double* rc) {
  if (!S || !rc) return fail(TDMD_E_INVALID, "sched_interaction_cutoff: null");
  *rc = S->cutoff;
  return TDMD_OK;
}

int tdmd_sched_time_passes(tdmd_sched* S, int32_t steps, float* ms_out) {
  // A window of `steps` steps with HIP events around each pass of the
  // steady-state step: EAM NVE -> [density, force + kick-drift], EAM NVT ->
  // [density, force + KE partials] (the chain half-steps and the scaled
  // kick-drift run between them, untimed), Morse -> [kick-drift,
  // force]. No rebuild test inside the window.
  if (!S || !ms_out || steps < 2) return fail(TDMD_E_INVALID, "sched_time_passes: bad args");
  if (!S->uploaded) return fail(TDMD_E_STATE, "sched_time_passes: upload() first");
  const bool nvt = S->nhcp.M > 0;
  const bool eam = S->kind == 1;
  if (nvt && !eam) return fail(TDMD_E_STATE, "sched_time_passes: NVT timing is for EAM");
  int rc;
  if (!S->initial_forces && (rc = compute_initial_forces(S))) return rc;
  hipStream_t s = S->stream;
  const char a_op = eam ? OP_DENS : OP_KD_FULL;
  const char b_op = nvt ? OP_F_KE : eam ? OP_F_FULL : OP_F_ONLY;
  // Events are stamped by the kernel dispatches themselves
  // (hipExtLaunchKernel), so each interval is one kernel's execution.
  std::vector<hipEvent_t> ev(static_cast<size_t>(4 * steps));
  for (auto& e : ev) TDMD_HIP_TRY(hipEventCreate(&e));
  if (nvt) {
    if ((rc = S->eng->launch(OP_NVT_PRE, s))) return rc;
  } else {
    if ((rc = S->eng->launch(OP_BOOT, s))) return rc;
    if (!eam && (rc = S->eng->launch(OP_F_ONLY, s))) return rc;
  }
  for (int k = 0; k < steps - 1; ++k) {
    if (nvt && (rc = S->eng->launch(k == 0 ? OP_KD_NVT : OP_KD_NVT2, s))) return rc;
    S->eng->time_next(ev[4 * k], ev[4 * k + 1]);
    if ((rc = S->eng->launch(a_op, s))) return rc;
    S->eng->time_next(ev[4 * k + 2], ev[4 * k + 3]);
    if ((rc = S->eng->launch(b_op, s))) return rc;
    S->eng->time_next(nullptr, nullptr);
    if (nvt && (rc = S->eng->launch(OP_NVT_POST_PRE, s))) return rc;
  }
  if (nvt) {
    for (char op : {OP_KD_NVT2, OP_DENS, OP_F_KICK2, OP_NVT_POST, OP_NVT_FINAL})
      if ((rc = S->eng->launch(op, s))) return rc;
  } else {
    if (eam && (rc = S->eng->launch(OP_DENS, s))) return rc;
    if (!eam && (rc = S->eng->launch(OP_KD_FULL, s))) return rc;
    if ((rc = S->eng->launch(OP_F_HALF, s))) return rc;
  }
  TDMD_HIP_TRY(hipStreamSynchronize(s));
  double ta = 0, tb = 0;
  for (int k = 0; k < steps - 1; ++k) {
    float x, y;
    TDMD_HIP_TRY(hipEventElapsedTime(&x, ev[4 * k], ev[4 * k + 1]));
    TDMD_HIP_TRY(hipEventElapsedTime(&y, ev[4 * k + 2], ev[4 * k + 3]));
    ta += x;
    tb += y;
  }
  for (auto& e : ev) (void)hipEventDestroy(e);
  ms_out[0] = static_cast<float>(ta / (steps - 1));
  ms_out[1] = static_cast<float>(tb / (steps - 1));
  S->current_step += steps;
  S->steps_since += steps;
  S->ticks += steps;
  return check_flags(S);
}

int tdmd_sched_pass_timing(tdmd_sched* S, int32_t on) {
  if (!S) return fail(TDMD_E_INVALID, "sched_pass_timing: null");
  if (on && !S->d_pclock) {
    int dev = 0;
    TDMD_HIP_TRY(hipGetDevice(&dev));
    TDMD_HIP_TRY(hipDeviceGetAttribute(&S->clock_khz, hipDeviceAttributeWallClockRate, dev));
    if (S->clock_khz <= 0) return fail(TDMD_E_HIP, "sched_pass_timing: no device wall clock");
    int rc = dalloc(S, &S->d_pclock, 8);
    if (rc) return rc;
  }
  TDMD_HIP_TRY(hipStreamSynchronize(S->stream));
  if (on) {
    const unsigned long long init[8] = {~0ull, 0, 0, 0, ~0ull, 0, 0, 0};
    TDMD_HIP_TRY(hipMemcpy(S->d_pclock, init, sizeof(init), hipMemcpyHostToDevice));
  }
  S->pass_timing = on != 0;
  S->a.pclock = on ? S->d_pclock : nullptr;
  return TDMD_OK;
}

int tdmd_sched_pass_times(tdmd_sched* S, float* ms_out) {
  if (!S || !ms_out) return fail(TDMD_E_INVALID, "sched_pass_times: null");
  if (!S->pass_timing) return fail(TDMD_E_STATE, "sched_pass_times: pass timing is off");
  TDMD_HIP_TRY(hipStreamSynchronize(S->stream));
  unsigned long long w[8];
  TDMD_HIP_TRY(hipMemcpy(w, S->d_pclock, sizeof(w), hipMemcpyDeviceToHost));
  if (w[7] == 0) return fail(TDMD_E_STATE, "sched_pass_times: no force pass ran since timing on");
  for (int p = 0; p < 2; ++p)
    ms_out[p] = w[4 * p + 3] ? static_cast<float>(static_cast<double>(w[4 * p + 2]) /
                                                  static_cast<double>(w[4 * p + 3]) / S->clock_khz)
                             : 0.0f;
  return TDMD_OK;
}

int tdmd_sched_halo_info(tdmd_sched* S, int64_t out[4]) {
  if (!S || !out) return fail(TDMD_E_INVALID, "sched_halo_info: null");
  for (int k = 0; k < 4; ++k) out[k] = 0;
  if (S->a.stage_cap == 0) return TDMD_OK;
  const int nb = (S->natoms + 1023) / 1024;
  std::vector<int32_t> hn(static_cast<size_t>(nb)), mode(static_cast<size_t>(nb));
  TDMD_HIP_TRY(hipStreamSynchronize(S->stream));
  TDMD_HIP_TRY(hipMemcpy(hn.data(), S->a.hn, hn.size() * 4, hipMemcpyDeviceToHost));
  TDMD_HIP_TRY(hipMemcpy(mode.data(), S->a.hmode, mode.size() * 4, hipMemcpyDeviceToHost));
  out[0] = nb;
  for (int b = 0; b < nb; ++b) {
    out[1] += mode[static_cast<size_t>(b)] == 0;
    out[2] = std::max<int64_t>(out[2], hn[static_cast<size_t>(b)]);
    out[3] += hn[static_cast<size_t>(b)];
  }
  return TDMD_OK;
}

int tdmd_sched_stream(const tdmd_sched* S, void** stream) {
  if (!S || !stream) return fail(TDMD_E_INVALID, "sched_stream: null");
  *stream = S->stream;
  return TDMD_OK;
}

int tdmd_sched_observables(tdmd_sched* S, tdmd_observables* o) {
  if (!S || !o) return fail(TDMD_E_INVALID, "sched_observables: null");
  if (!S->uploaded) return fail(TDMD_E_STATE, "sched_observables: upload() first");
  double th[6];
  int rc = tdmd_sched_thermo(S, th);
  if (rc) return rc;
  double sc[4];
  TDMD_HIP_TRY(hipMemcpy(sc, S->d_scalars, 32, hipMemcpyDeviceToHost));
  double vol = 0.0;
  if (S->multibox) {
    for (const auto& b : S->h_boxes) vol += b.mp.L[0] * b.mp.L[1] * b.mp.L[2];
  } else {
    vol = S->a.mp.L[0] * S->a.mp.L[1] * S->a.mp.L[2];
  }
  o->step = S->current_step;
  o->natoms = S->natoms;
  o->pe = th[0];
  o->ke = th[1];
  o->te = th[0] + th[1];
  o->temp = th[3];
  o->nhc_energy = th[2];
  o->conserved = o->te + th[2];
  o->virial = sc[3];
  o->volume = vol;
  // P = (2 KE + W) / (3 V), eV/A^3 -> bar (1 eV/A^3 = 1.602176634e6 bar)
  o->pressure = (2.0 * th[1] + sc[3]) / (3.0 * vol) * 1.602176634e6;
  o->max_neighbors = static_cast<int32_t>(th[4]);
  o->mean_neighbors = th[5];
  std::vector<int32_t> nn(static_cast<size_t>(S->natoms));
  TDMD_HIP_TRY(hipMemcpy(nn.data(), S->a.cntn, nn.size() * 4, hipMemcpyDeviceToHost));
  int64_t sn = 0;
  for (int32_t v : nn) sn += v;
  o->mean_near_neighbors = static_cast<double>(sn) / S->natoms;
  return TDMD_OK;
}

int tdmd_sched_thermo(tdmd_sched* S, double out[6]) {
  if (!S || !out) return fail(TDMD_E_INVALID, "sched_thermo: null");
  if (!S->uploaded) return fail(TDMD_E_STATE, "sched_thermo: upload() first");
  int rc;
  if (!S->initial_forces && (rc = compute_initial_forces(S))) return rc;
  if ((rc = S->eng->energy_pass(S->stream, S->d_scalars))) return rc;
  double sc[3];
  TDMD_HIP_TRY(hipMemcpyAsync(sc, S->d_scalars, 24, hipMemcpyDeviceToHost, S->stream));
  std::vector<int32_t> cnt(static_cast<size_t>(S->natoms));
  TDMD_HIP_TRY(hipMemcpyAsync(cnt.data(), S->a.cnt, S->natoms * 4, hipMemcpyDeviceToHost, S->stream));
  double nhc[32];
  TDMD_HIP_TRY(hipMemcpyAsync(nhc, S->a.nhc, 32 * 8, hipMemcpyDeviceToHost, S->stream));
  TDMD_HIP_TRY(hipStreamSynchronize(S->stream));
  out[0] = sc[0] + sc[1];
  out[1] = sc[2];
  double enhc = 0.0;
  const int M = S->nhcp.M;
  const double kt = kBoltzmann * S->cfg.t_target;
  for (int k = 0; k < M; ++k)
    enhc += 0.5 * nhc[16 + k] * nhc[8 + k] * nhc[8 + k] +
            (k == 0 ? static_cast<double>(S->nhcp.n_dof) * kt : kt) * nhc[k];
  out[2] = enhc;
  out[3] = 2.0 * sc[2] / (3.0 * static_cast<double>(S->natoms) * kBoltzmann);
  int64_t sum = 0;
  int mx = 0;
  for (int v : cnt) {
    sum += v;
    mx = std::max(mx, v);
  }
  out[4] = mx;
  out[5] = static_cast<double>(sum) / S->natoms;
  return check_flags(S);
}

}  // extern "C"
