// forces_csr.cpp -- Morse and EAM forces over a full CSR list: the
// compute_morse_gpu / DeviceEam::compute boundary
// (src/potentials/device_morse.cu:32-170, src/potentials/device_eam.cu:72-421).
//
// kRowLanes neighbouring lanes per atom: they read a row's consecutive slots
// side by side and combine their sums by a butterfly, a fixed order. (One lane
// per atom reads 64 rows ~400 bytes apart, a cache line for every slot, and
// walks ~100 dependent slots in turn: 16,384 atoms filled 64 of 256 CUs.)
// The next slot's index is loaded while a slot is evaluated. Pair geometry
// (difference, minimum image, r^2, cutoff, r) in FP64, pair functions in R
// (pair_math.hpp). Per-atom sums (force, density, energy) are FP64. Forces
// are stored, not accumulated (device_morse.cu:110-117); energies are added
// to *d_energy: one FP64 atomic per 256 atoms when no workspace is given,
// otherwise partials, one per 256 atoms, summed in a fixed order.
#include "csr_rows.hpp"

namespace tdmd_hip {

namespace {

// 0-based table index of a 1-based type. Types outside 1..ntypes (which the
// reference would use to index out of its tables) are clamped to the range.
__device__ __forceinline__ int clamp_type(int t, int ntypes) {
  t -= 1;
  return t < 0 ? 0 : (t >= ntypes ? ntypes - 1 : t);
}

__device__ __forceinline__ void emit_energy(double e, double* __restrict__ partials,
                                            double* __restrict__ d_energy) {
  const double t = block_sum<kEnergyBlock>(e);
  if (threadIdx.x == 0) {
    if (partials)
      partials[piece_of(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x))] = t;
    else
      atomicAdd(d_energy, t);
  }
}

// Forces of one atom, by the first of its lanes; kAccum adds to what
// `forces` holds (the zone pass, device_morse_zone.cu:29-117).
template <class R, bool kAccum>
__device__ __forceinline__ void put_force(R* __restrict__ forces, int i, double fx, double fy,
                                          double fz) {
  if (threadIdx.x % kRowLanes != 0) return;
  R* f = forces + 3 * static_cast<int64_t>(i);
  if (kAccum) {
    f[0] += static_cast<R>(fx);
    f[1] += static_cast<R>(fy);
    f[2] += static_cast<R>(fz);
  } else {
    f[0] = static_cast<R>(fx);
    f[1] = static_cast<R>(fy);
    f[2] = static_cast<R>(fz);
  }
}

// Atoms [first, first + count).
template <class R, bool kEnergy, bool kAccum>
__global__ void __launch_bounds__(kEnergy ? kEnergyBlock : kBlock)
morse_csr_kernel(const double* __restrict__ pos, R* __restrict__ forces,
                 const int32_t* __restrict__ nbrs, const int32_t* __restrict__ offsets,
                 const int32_t* __restrict__ counts, int first, int count, PairBox box,
                 MorseCoef p, double* __restrict__ partials, double* __restrict__ d_energy) {
  double pe = 0.0;
  for_atoms<kEnergy>(count, [&](int t) {
    const int i = first + t;
    const double* pi = pos + 3 * static_cast<int64_t>(i);
    const double xi = pi[0], yi = pi[1], zi = pi[2];
    double fx = 0.0, fy = 0.0, fz = 0.0;
    auto load = [&](int j) { return neighbour_at(pos, j); };
    for_row<kMorseSlots>(nbrs, offsets[i], counts[i], xi, yi, zi, box, load,
                         [&](int, const Neighbour&, double dx, double dy, double dz, double r2) {
      if (r2 < p.rc_sq) {
        const PairR<R> pr = pair_r<R>(r2);
        R e;
        const double fpair = static_cast<double>(morse_fpair<R>(p, pr, &e));
        if (kEnergy) pe += 0.5 * static_cast<double>(e);
        fx = fma(fpair, dx, fx);
        fy = fma(fpair, dy, fy);
        fz = fma(fpair, dz, fz);
      }
    });
    put_force<R, kAccum>(forces, i, row_sum(fx), row_sum(fy), row_sum(fz));
  });
  if (kEnergy) emit_energy(pe, partials, d_energy);
}

// Passes 1 and 2: rho_i = sum_j rho_{t_j}(r_ij), FP64 sum
// (device_eam.cu:72-133), and fp_i = F'_{t_i}(rho_i) (:137-162).
template <class R, bool kOne>
__global__ void __launch_bounds__(kBlock)
eam_density_csr_kernel(const double* __restrict__ pos, const int32_t* __restrict__ types,
                       const int32_t* __restrict__ nbrs, const int32_t* __restrict__ offsets,
                       const int32_t* __restrict__ counts, int natoms, EamLayout t, PairBox box,
                       const typename Quad<R>::type* __restrict__ coeff,
                       double* __restrict__ rho, R* __restrict__ fp) {
  for_atoms<false>(natoms, [&](int i) {
    const double* pi = pos + 3 * static_cast<int64_t>(i);
    const double xi = pi[0], yi = pi[1], zi = pi[2];
    double rho_i = 0.0;
    auto load = [&](int j) { return neighbour_at(pos, j); };
    for_row<kEamSlots>(nbrs, offsets[i], counts[i], xi, yi, zi, box, load,
                       [&](int j, const Neighbour&, double, double, double, double r2) {
      if (r2 < t.rc_sq) {
        R x;
        const int k = spline_locate<R>(t.r, pair_r<R>(r2).r, &x);
        const int tj = kOne ? 0 : clamp_type(types[j], t.ntypes);
        rho_i += static_cast<double>(quad_value<R>(coeff[t.rho_at(tj) + k], x));
      }
    });
    rho_i = row_sum(rho_i);
    if (threadIdx.x % kRowLanes == 0) {
      R x;
      const int k = spline_locate<R>(t.F, rho_i, &x);
      rho[i] = rho_i;
      fp[i] = quad_deriv<R>(coeff[t.f_at(kOne ? 0 : clamp_type(types[i], t.ntypes)) + k], x);
    }
  });
}

// Pass 3: F_i = sum_j -(phi' + fp_i rho'_{t_j} + fp_j rho'_{t_i})/r * d
// (device_eam.cu:176-278); energy 0.5 phi per pair of the full list and
// F(rho_i). One interval per pair: the three r splines share the grid.
template <class R, bool kEnergy, bool kOne>
__global__ void __launch_bounds__(kEnergy ? kEnergyBlock : kBlock)
eam_force_csr_kernel(const double* __restrict__ pos, R* __restrict__ forces,
                     const int32_t* __restrict__ types, const int32_t* __restrict__ nbrs,
                     const int32_t* __restrict__ offsets, const int32_t* __restrict__ counts,
                     int natoms, EamLayout t, PairBox box,
                     const typename Quad<R>::type* __restrict__ coeff,
                     const double* __restrict__ rho, const R* __restrict__ fp,
                     double* __restrict__ partials, double* __restrict__ d_energy) {
  double pe = 0.0;
  for_atoms<kEnergy>(natoms, [&](int i) {
    const double* pi = pos + 3 * static_cast<int64_t>(i);
    const double xi = pi[0], yi = pi[1], zi = pi[2];
    const int ti = kOne ? 0 : clamp_type(types[i], t.ntypes);
    const R fpi = fp[i];
    double fx = 0.0, fy = 0.0, fz = 0.0;
    struct WithFp : Neighbour {
      R fp;
    };
    auto load = [&](int j) { return WithFp{neighbour_at(pos, j), fp[j]}; };
    for_row<kEamSlots>(nbrs, offsets[i], counts[i], xi, yi, zi, box, load,
                       [&](int j, const WithFp& v, double dx, double dy, double dz, double r2) {
      if (r2 < t.rc_sq) {
        const PairR<R> pr = pair_r<R>(r2);
        const int tj = kOne ? 0 : clamp_type(types[j], t.ntypes);
        R x;
        const int k = spline_locate<R>(t.r, pr.r, &x);
        const auto cphi = coeff[t.phi_at(kOne ? 0 : phi_index(ti, tj, t.ntypes)) + k];
        const R dphi = quad_deriv<R>(cphi, x);
        if (kEnergy) pe += 0.5 * static_cast<double>(quad_value<R>(cphi, x));
        const R drho_j = quad_deriv<R>(coeff[t.rho_at(tj) + k], x);
        const R drho_i = kOne ? drho_j : quad_deriv<R>(coeff[t.rho_at(ti) + k], x);
        const double fpair =
            static_cast<double>(-(dphi + fpi * drho_j + v.fp * drho_i) * pr.rinv);
        fx = fma(fpair, dx, fx);
        fy = fma(fpair, dy, fy);
        fz = fma(fpair, dz, fz);
      }
    });
    put_force<R, false>(forces, i, row_sum(fx), row_sum(fy), row_sum(fz));
    if (kEnergy && threadIdx.x % kRowLanes == 0) {
      R x;
      const int k = spline_locate<R>(t.F, rho[i], &x);
      pe += static_cast<double>(quad_value<R>(coeff[t.f_at(ti) + k], x));
    }
  });
  if (kEnergy) emit_energy(pe, partials, d_energy);
}

template <class R, bool kAccum>
int morse_launch(const double* pos, void* forces, const int32_t* nbrs, const int32_t* offsets,
                 const int32_t* counts, int first, int count, const DevBox& box,
                 const tdmd_morse_params& p, double* d_energy, void* work, hipStream_t stream) {
  double* partials = static_cast<double*>(work);
  const MorseCoef c{p.d, p.alpha, p.r0, p.rc_sq};
  const PairBox pb = make_pair_box(box);
  const int grid = row_grid(count, d_energy != nullptr);
  if (d_energy) {
    morse_csr_kernel<R, true, kAccum><<<grid, kEnergyBlock, 0, stream>>>(
        pos, static_cast<R*>(forces), nbrs, offsets, counts, first, count, pb, c, partials,
        d_energy);
    TDMD_LAUNCH_CHECK();
    if (partials) return launch_sum_partials(partials, grid, d_energy, 1, stream);
  } else {
    morse_csr_kernel<R, false, kAccum><<<grid, kBlock, 0, stream>>>(
        pos, static_cast<R*>(forces), nbrs, offsets, counts, first, count, pb, c, nullptr,
        nullptr);
    TDMD_LAUNCH_CHECK();
  }
  return TDMD_OK;
}

template <class R, bool kOne>
int eam_passes(const tdmd_eam_tables* t, const double* pos, R* forces, const int32_t* types,
               const int32_t* nbrs, const int32_t* offsets, const int32_t* counts, int natoms,
               const PairBox& box, double* rho, R* fp, double* d_energy, double* partials,
               hipStream_t stream) {
  const auto* coeff = static_cast<const typename Quad<R>::type*>(t->d_coeff);
  const EamLayout e = eam_layout(t);
  const int grid = row_grid(natoms, false);
  eam_density_csr_kernel<R, kOne><<<grid, kBlock, 0, stream>>>(
      pos, types, nbrs, offsets, counts, natoms, e, box, coeff, rho, fp);
  TDMD_LAUNCH_CHECK();
  if (d_energy) {
    const int ge = row_grid(natoms, true);
    eam_force_csr_kernel<R, true, kOne><<<ge, kEnergyBlock, 0, stream>>>(
        pos, forces, types, nbrs, offsets, counts, natoms, e, box, coeff, rho, fp, partials,
        d_energy);
    TDMD_LAUNCH_CHECK();
    if (partials) return launch_sum_partials(partials, ge, d_energy, 1, stream);
  } else {
    eam_force_csr_kernel<R, false, kOne><<<grid, kBlock, 0, stream>>>(
        pos, forces, types, nbrs, offsets, counts, natoms, e, box, coeff, rho, fp, nullptr,
        nullptr);
    TDMD_LAUNCH_CHECK();
  }
  return TDMD_OK;
}

template <class R>
int eam_launch(const tdmd_eam_tables* t, const double* pos, void* forces, const int32_t* types,
               const int32_t* nbrs, const int32_t* offsets, const int32_t* counts, int natoms,
               const DevBox& box, double* rho, void* fp, double* d_energy, void* work,
               hipStream_t stream) {
  const PairBox pb = make_pair_box(box);
  auto* f = static_cast<R*>(forces);
  auto* d = static_cast<R*>(fp);
  auto* w = static_cast<double*>(work);
  return t->ntypes == 1 ? eam_passes<R, true>(t, pos, f, types, nbrs, offsets, counts, natoms, pb,
                                              rho, d, d_energy, w, stream)
                        : eam_passes<R, false>(t, pos, f, types, nbrs, offsets, counts, natoms,
                                               pb, rho, d, d_energy, w, stream);
}

// ---------------------------------------------------------------------------
// Allocation-free EAM compute: the per-atom densities, F'(rho) and the
// energy partials live in one file-scope device array instead of caller
// buffers. Its device address is looked up once per device
// (hipGetSymbolAddress) and kept; kernels get that address, never the
// array's host-side name. Every call on a device shares the array: calls
// that overlap on one device (several streams, several host threads) race.
// The kernels store every element they later read (rho, F'(rho), one
// partial per block), so nothing needs clearing between calls.
// ---------------------------------------------------------------------------
constexpr int kNoAllocMaxAtoms = 1 << 20;
constexpr size_t kScratchRho = 0;                                             // double[N]
constexpr size_t kScratchFp = static_cast<size_t>(kNoAllocMaxAtoms) * 8;      // real[N]
constexpr size_t kScratchPartials = static_cast<size_t>(kNoAllocMaxAtoms) * 16;  // double[grid]
constexpr size_t kScratchBytes =
    kScratchPartials + static_cast<size_t>((kNoAllocMaxAtoms + kBlock - 1) / kBlock + 64) * 8;

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
void* g_scratch[kMaxDevices] = {};

int scratch_for_current_device(unsigned char** out) {
  int dev = 0;
  TDMD_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(TDMD_E_INVALID, "eam_compute_noalloc: device index");
  if (!g_scratch[dev]) {
    void* p = nullptr;
    TDMD_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return fail(TDMD_E_HIP, "eam_compute_noalloc: no device address for the scratch array");
    g_scratch[dev] = p;
  }
  *out = static_cast<unsigned char*>(g_scratch[dev]);
  return TDMD_OK;
}

}  // namespace

}  // namespace tdmd_hip

using namespace tdmd_hip;

extern "C" {

int tdmd_morse_force(int32_t precision, const double* d_pos, void* d_forces,
                     const int32_t* d_neighbors, const int32_t* d_offsets,
                     const int32_t* d_counts, int32_t natoms, const tdmd_box* box,
                     const tdmd_morse_params* params, double* d_energy, void* d_work,
                     void* stream) {
  if (!box || !params || natoms < 0) return fail(TDMD_E_INVALID, "morse_force: bad arguments");
  if (natoms == 0) return TDMD_OK;  // device_morse.cu:141
  if (!d_pos || !d_forces || !d_offsets || !d_counts)
    return fail(TDMD_E_INVALID, "morse_force: null pointer");
  const DevBox db = make_devbox(*box);
  if (precision == TDMD_MIXED)
    return morse_launch<float, false>(d_pos, d_forces, d_neighbors, d_offsets, d_counts, 0,
                                      natoms, db, *params, d_energy, d_work, as_stream(stream));
  if (precision == TDMD_FP64)
    return morse_launch<double, false>(d_pos, d_forces, d_neighbors, d_offsets, d_counts, 0,
                                       natoms, db, *params, d_energy, d_work,
                                       as_stream(stream));
  return fail(TDMD_E_INVALID, "morse_force: bad precision");
}

int tdmd_morse_force_zone(int32_t precision, const double* d_pos, void* d_forces,
                          const int32_t* d_neighbors, const int32_t* d_offsets,
                          const int32_t* d_counts, int32_t first_atom, int32_t atom_count,
                          const tdmd_box* box, const tdmd_morse_params* params,
                          double* d_energy, void* d_work, void* stream) {
  if (!box || !params || first_atom < 0 || atom_count < 0)
    return fail(TDMD_E_INVALID, "morse_force_zone: bad arguments");
  if (atom_count == 0) return TDMD_OK;  // device_morse_zone.cu:126
  if (!d_pos || !d_forces || !d_offsets || !d_counts)
    return fail(TDMD_E_INVALID, "morse_force_zone: null pointer");
  const DevBox db = make_devbox(*box);
  if (precision == TDMD_MIXED)
    return morse_launch<float, true>(d_pos, d_forces, d_neighbors, d_offsets, d_counts,
                                     first_atom, atom_count, db, *params, d_energy, d_work,
                                     as_stream(stream));
  if (precision == TDMD_FP64)
    return morse_launch<double, true>(d_pos, d_forces, d_neighbors, d_offsets, d_counts,
                                      first_atom, atom_count, db, *params, d_energy, d_work,
                                      as_stream(stream));
  return fail(TDMD_E_INVALID, "morse_force_zone: bad precision");
}

int tdmd_eam_compute(const tdmd_eam_tables* t, const double* d_pos, void* d_forces,
                     const int32_t* d_types, const int32_t* d_neighbors,
                     const int32_t* d_offsets, const int32_t* d_counts, int32_t natoms,
                     const tdmd_box* box, double* d_rho, void* d_fp, double* d_energy,
                     void* d_work, void* stream) {
  if (!t || !box || natoms < 0) return fail(TDMD_E_INVALID, "eam_compute: bad arguments");
  if (natoms == 0) return TDMD_OK;  // device_eam.cu:345
  if (!d_pos || !d_forces || !d_types || !d_offsets || !d_counts || !d_rho || !d_fp)
    return fail(TDMD_E_INVALID, "eam_compute: null pointer");
  if (t->ntypes > 8) return fail(TDMD_E_INVALID, "eam_compute: at most 8 element types");
  const DevBox db = make_devbox(*box);
  if (t->precision == TDMD_MIXED)
    return eam_launch<float>(t, d_pos, d_forces, d_types, d_neighbors, d_offsets, d_counts,
                             natoms, db, d_rho, d_fp, d_energy, d_work, as_stream(stream));
  return eam_launch<double>(t, d_pos, d_forces, d_types, d_neighbors, d_offsets, d_counts,
                            natoms, db, d_rho, d_fp, d_energy, d_work, as_stream(stream));
}

int tdmd_eam_compute_noalloc(const tdmd_eam_tables* t, const double* d_pos, void* d_forces,
                             const int32_t* d_types, const int32_t* d_neighbors,
                             const int32_t* d_offsets, const int32_t* d_counts, int32_t natoms,
                             const tdmd_box* box, double* d_energy, void* stream) {
  if (!t || !box || natoms < 0) return fail(TDMD_E_INVALID, "eam_compute_noalloc: bad arguments");
  if (natoms > kNoAllocMaxAtoms)
    return fail(TDMD_E_INVALID, "eam_compute_noalloc: " + std::to_string(natoms) +
                                    " atoms exceed the scratch array's " +
                                    std::to_string(kNoAllocMaxAtoms));
  if (natoms == 0) return TDMD_OK;
  if (!d_pos || !d_forces || !d_types || !d_offsets || !d_counts)
    return fail(TDMD_E_INVALID, "eam_compute_noalloc: null pointer");
  if (t->ntypes > 8) return fail(TDMD_E_INVALID, "eam_compute_noalloc: at most 8 element types");
  unsigned char* base = nullptr;
  const int rc = scratch_for_current_device(&base);
  if (rc) return rc;
  double* rho = reinterpret_cast<double*>(base + kScratchRho);
  void* fp = base + kScratchFp;
  void* work = base + kScratchPartials;
  const DevBox db = make_devbox(*box);
  if (t->precision == TDMD_MIXED)
    return eam_launch<float>(t, d_pos, d_forces, d_types, d_neighbors, d_offsets, d_counts,
                             natoms, db, rho, fp, d_energy, work, as_stream(stream));
  return eam_launch<double>(t, d_pos, d_forces, d_types, d_neighbors, d_offsets, d_counts,
                            natoms, db, rho, fp, d_energy, work, as_stream(stream));
}

}  // extern "C"
