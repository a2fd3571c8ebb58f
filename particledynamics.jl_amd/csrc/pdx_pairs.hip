// Pair forces, per-particle half energies / half virials and FP64 totals over slot-major
// ELL rows: LJ, WCA, harmonic soft repulsion, each optionally with real-space Ewald Coulomb
// through an r^2 polynomial of the long-range correction.
//
// Thread layout: G lanes per particle (G in 1..64, a power of two) stride the particle's
// row (slots lane, lane+G, ...) and combine with xor-shuffles inside the wave64; the row
// slots of G=1 are read fully coalesced, larger G trade that for more parallelism on small
// systems (_pair_cooperative_kernel!, src/engine/PairTraversal.jl:66-125). Neighbor
// coordinates and charges come from one float4 gather (x, y, z, q).
#include "pdx_pair_kernels.hpp"

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

using namespace pdx;
using namespace pdx::pairk;

namespace {

// cell-ordered copy of the current coordinates and charges (every step, after the list check)
__global__ __launch_bounds__(TPB) void k_refresh_sorted(int N, const int32_t *__restrict__ ids,
                                                         const float4 *__restrict__ packed, float4 *sortedq,
                                                         const int64_t *state) {
  if (!(state[PDX_DN_VALID] != 0 && state[PDX_DN_ERROR] == 0)) return;
  const int t = blockIdx.x * TPB + threadIdx.x;
  if (t < N) sortedq[t] = packed[ids[t] - 1];
}

// ---------------------------------------------------------------- host: Ewald correction fit
// corr(s) = erf(alpha r)/r and fcorr(s) = -(1/r) d corr/dr at s = r^2 (long_range_correction,
// src/electrostatics/Splits.jl:142-161, restated in FP64): the alternating Taylor series in
// z = alpha^2 s below z = 1, the closed forms above (no cancellation there).
void ewald_correction(double alpha, double s, double &corr, double &fcorr) {
  const double pre = 2.0 * alpha / std::sqrt(M_PI);
  const double z = alpha * alpha * s;
  if (z < 1.0) {
    // corr = pre sum_n t_n/(2n+1) with t_n = (-z)^n/n!; fcorr = -2 d corr/ds
    //      = 2 pre alpha^2 sum_{n>=1} t_{n-1}/(2n+1)
    double ce = 1.0, cf = 0.0, term = 1.0;
    for (int n = 1; n < 60; ++n) {
      cf += term / (2 * n + 1);
      term = -term * z / n;
      ce += term / (2 * n + 1);
      if (std::fabs(term) < 1e-22) break;
    }
    corr = pre * ce;
    fcorr = 2.0 * pre * alpha * alpha * cf;
    return;
  }
  const double r = std::sqrt(s);
  const double ef = std::erf(alpha * r);
  corr = ef / r;
  fcorr = ef / (s * r) - pre * std::exp(-z) / s;
}

// Chebyshev interpolation on [-1, 1] at n first-kind nodes; truncate where the tail of
// |c_j| drops below tol * max|f|; return monomial coefficients in x.
std::vector<double> chebyshev_monomial(const std::vector<double> &fvals, double tol) {
  const int n = (int)fvals.size();
  std::vector<double> c(n, 0.0);
  double fmax = 0.0;
  for (double v : fvals) fmax = std::max(fmax, std::fabs(v));
  for (int j = 0; j < n; ++j) {
    double s = 0.0;
    for (int k = 0; k < n; ++k) s += fvals[k] * std::cos(M_PI * j * (k + 0.5) / n);
    c[j] = (j == 0 ? 1.0 : 2.0) * s / n;
  }
  int deg = n - 1;
  double tail = 0.0;
  for (int j = n - 1; j >= 1; --j) {
    tail += std::fabs(c[j]);
    if (tail > tol * std::max(fmax, 1e-300)) { deg = j; break; }
    deg = j - 1;
  }
  const int m = deg + 1;
  // T_k as monomials, accumulated: T_{k+1} = 2x T_k - T_{k-1}
  std::vector<double> mono(m, 0.0), t0(m, 0.0), t1(m, 0.0), t2(m, 0.0);
  t0[0] = 1.0;
  mono[0] += c[0];
  if (m > 1) {
    t1[1] = 1.0;
    mono[1] += c[1];
  }
  for (int k = 2; k < m; ++k) {
    std::fill(t2.begin(), t2.end(), 0.0);
    for (int q = 0; q + 1 < m; ++q) t2[q + 1] += 2.0 * t1[q];
    for (int q = 0; q < m; ++q) t2[q] -= t0[q];
    for (int q = 0; q < m; ++q) mono[q] += c[k] * t2[q];
    t0 = t1;
    t1 = t2;
  }
  return mono;
}

}  // namespace

// host helpers shared with the mesh translation unit
namespace pdx {
void host_ewald_correction(double alpha, double s, double &corr, double &fcorr) {
  ewald_correction(alpha, s, corr, fcorr);
}
}  // namespace pdx

extern "C" int pdx_pair_create(const pdx_pair_spec *spec, pdx_pair_t *out) {
  if (!spec || !out) return fail(PDX_ERR_ARGUMENT, "null argument");
  *out = nullptr;
  const pdx_pair_spec &sp = *spec;
  if (sp.model < PDX_PAIR_NONE || sp.model > PDX_PAIR_MATRIX_WCA) return fail(PDX_ERR_ARGUMENT, "unknown pair model");
  const bool typed = typed_model(sp.model);
  if (sp.model != PDX_PAIR_NONE && sp.model != PDX_PAIR_MATRIX_LJ && sp.model != PDX_PAIR_MATRIX_WCA) {
    if (!(std::isfinite(sp.epsilon) && (typed || (std::isfinite(sp.sigma) && sp.sigma > 0))))
      return fail(PDX_ERR_ARGUMENT, "pair epsilon and sigma must be finite, sigma positive");
    if ((sp.model == PDX_PAIR_LJ || sp.model == PDX_PAIR_MIXED_LJ || sp.model == PDX_PAIR_MIXED_WCA) &&
        !(std::isfinite(sp.cutoff) && sp.cutoff > 0))
      return fail(PDX_ERR_ARGUMENT, "LJ cutoff (the rcut factor of the mixed-sigma models) must be finite and positive");
  }
  if (typed && sp.lanes < 0) return fail(PDX_ERR_ARGUMENT, "typed pair models use the lanes layout (lanes >= 0)");
  if (sp.coulomb) {
    if (!(sp.coulomb_C > 0 && std::isfinite(sp.coulomb_C)))
      return fail(PDX_ERR_ARGUMENT, "coulomb_prefactor must be finite and positive");
    if (!(sp.coulomb_cutoff > 0 && std::isfinite(sp.coulomb_cutoff)))
      return fail(PDX_ERR_ARGUMENT, "real_cutoff must be finite and positive");
    if (sp.coulomb != 1 && sp.coulomb != 2) return fail(PDX_ERR_ARGUMENT, "coulomb must be 0, 1 (Gaussian) or 2 (prolate)");
    if (sp.coulomb == 1 && !(sp.alpha > 0 && std::isfinite(sp.alpha)))
      return fail(PDX_ERR_ARGUMENT, "Ewald alpha must be finite and positive.");
    if (sp.coulomb == 2 && !(sp.split_shape > 0 && std::isfinite(sp.split_shape)))
      return fail(PDX_ERR_ARGUMENT, "ESP split shape must be finite and positive.");
  }
  if (sp.lanes > 0 && (sp.lanes > 64 || (sp.lanes & (sp.lanes - 1))))
    return fail(PDX_ERR_ARGUMENT, "lanes per particle must be a power of two in 1..64");
  if (sp.lanes < 0 && !(sp.lanes == -2 || sp.lanes == -4 || sp.lanes == -8 || sp.lanes == -16))
    return fail(PDX_ERR_ARGUMENT, "split layouts use 2, 4, 8 or 16 waves (lanes = -2, -4, -8, -16)");
  auto *p = new pdx_pair_s();
  p->spec = sp;
  const float eps = (float)sp.epsilon, sig = (float)sp.sigma;
  p->eps = eps;
  p->sig2 = sig * sig;
  if (sp.model == PDX_PAIR_LJ) {
    const float rc = (float)sp.cutoff;
    p->rc2 = rc * rc;
    if (sp.shift && rc > 0) {  // lj_cutoff_energy (PairModels.jl:20-25), in the list precision
      const float s2 = p->sig2 / (rc * rc), s6 = s2 * s2 * s2;
      p->eshift = 4.0f * eps * (s6 * s6 - s6);
    }
  } else if (sp.model == PDX_PAIR_WCA) {
    p->rc2 = 1.2599211f * p->sig2;  // UniformWCA constant (PairModels.jl:16)
  } else if (sp.model == PDX_PAIR_SOFT) {
    p->rc2 = p->sig2;
  } else if (sp.model == PDX_PAIR_MIXED_LJ || sp.model == PDX_PAIR_MIXED_WCA) {
    // rc = factor sigma_ij: (rc/sigma_ij)^2 = factor^2, and the LJ shift u(rc) is one constant
    const float f = (float)sp.cutoff;
    p->rfac2 = f * f;
    if (sp.model == PDX_PAIR_MIXED_LJ && sp.shift) {
      const float s2 = 1.0f / (f * f), s6 = s2 * s2 * s2;
      p->eshift = 4.0f * eps * (s6 * s6 - s6);
    }
  }
  if (sp.coulomb) {
    const double rc = sp.coulomb_cutoff, rc2 = rc * rc, a = sp.alpha;
    // the split's long-range part 1/r - E_s/r and its force factor as functions of s = r^2:
    // Gaussian (erf(alpha r)/r) or prolate (a(t)/r by quadrature, Splits.jl:163-202)
    ProlateSplit ps;
    if (sp.coulomb == 2 && !ps.make(rc, sp.split_shape)) {
      delete p;
      return fail(PDX_ERR_ARGUMENT, "prolate split set-up failed");
    }
    auto correction = [&](double s, double &corr, double &fcorr) {
      if (sp.coulomb == 2) ps.correction(s, corr, fcorr);
      else ewald_correction(a, s, corr, fcorr);
    };
    p->cC = (float)sp.coulomb_C;
    p->crc2 = (float)rc2;
    p->csx = (float)(2.0 / rc2);
    // cutoff energy E_s(rc)/rc: erfc(alpha rc)/rc, exactly zero for the prolate split (Splits.jl:77-78)
    p->ceshift = (sp.coulomb_shift && sp.coulomb == 1) ? (float)(std::erfc(a * rc) / rc) : 0.0f;
    p->halfself = (float)(0.5 * sp.coulomb_C * (sp.coulomb == 2 ? ps.self_coefficient() : 2.0 * a / std::sqrt(M_PI)));
    const int nodes = 64;
    std::vector<double> fe(nodes), ff(nodes);
    for (int k = 0; k < nodes; ++k) {
      const double x = std::cos(M_PI * (k + 0.5) / nodes);
      double corr, fcorr;
      correction((x + 1.0) * rc2 / 2.0, corr, fcorr);
      fe[k] = -corr;
      ff[k] = fcorr;
    }
    // FP32 tolerances of coulomb_polynomial (PairFunctor.jl:58-61): 1e-8 energy, 1e-7 force
    std::vector<double> me = chebyshev_monomial(fe, 1e-8), mf = chebyshev_monomial(ff, 1e-7);
    if ((int)me.size() > MAXC || (int)mf.size() > MAXC) {
      delete p;
      return fail(PDX_ERR_ARGUMENT, "the split's long-range polynomial needs more than 24 terms (alpha*cutoff or the split shape too large)");
    }
    p->npe = (int)me.size();
    p->npf = (int)mf.size();
    for (int k = 0; k < p->npe; ++k) p->pe[k] = (float)me[k];
    for (int k = 0; k < p->npf; ++k) p->pf[k] = (float)mf[k];
    // measured fit error of the FP32 Horner form against FP64, relative to max|f|
    double emax = 0, fmax = 0, eerr = 0, ferr = 0;
    for (int k = 0; k <= 2000; ++k) {
      const double x = -1.0 + 2.0 * k / 2000.0;
      double corr, fcorr;
      correction((x + 1.0) * rc2 / 2.0, corr, fcorr);
      float he = p->pe[p->npe - 1], hf = p->pf[p->npf - 1];
      for (int q = p->npe - 2; q >= 0; --q) he = fmaf(he, (float)x, p->pe[q]);
      for (int q = p->npf - 2; q >= 0; --q) hf = fmaf(hf, (float)x, p->pf[q]);
      emax = std::max(emax, std::fabs(corr));
      fmax = std::max(fmax, std::fabs(fcorr));
      eerr = std::max(eerr, std::fabs((double)he + corr));
      ferr = std::max(ferr, std::fabs((double)hf - fcorr));
    }
    p->fit_err_e = eerr / emax;
    p->fit_err_f = ferr / fmax;
  }
  p->lanes = sp.lanes;
  *out = p;
  return PDX_OK;
}

extern "C" int pdx_pair_destroy(pdx_pair_t p) {
  delete p;
  return PDX_OK;
}

extern "C" int pdx_pair_info(pdx_pair_t p, double out[4]) {
  if (!p || !out) return fail(PDX_ERR_ARGUMENT, "null argument");
  out[0] = p->npe; out[1] = p->npf; out[2] = p->fit_err_e; out[3] = p->fit_err_f;
  return PDX_OK;
}

namespace {
// fixed_partial == nullptr: the model's own partial buffer, grown here when too small (a host
// boundary: it synchronises and allocates); otherwise that caller-provided workspace of
// fixed_blocks per-block slots, and a launch needing more is refused.
int pair_forces_impl(pdx_pair_t p, pdx_nl_t nl, float *fx, float *fy, float *fz, float *Epot, float *V,
                     double *totals, int32_t flags, pdx_stream_t stream, double *fixed_partial, int fixed_blocks) {
  if (!p || !nl) return fail(PDX_ERR_ARGUMENT, "null pair model or neighbor list");
  if (!fx || !fy || !fz) return fail(PDX_ERR_ARGUMENT, "null force array");
  const bool energy = (flags & PDX_ENERGY) != 0;
  const int N = nl->N;
  // lanes > 0: G lanes of a wave per particle; lanes < 0: the split layout with -lanes waves
  // per block of 64 particles; 0: automatic
  const bool acc_path = p->accumulate != PDX_ACC_FP32 || p->bonds != nullptr;
  const bool cells = p->traversal == PDX_TRAVERSAL_CELLS;
  const bool typed = typed_model(p->spec.model);
  if (typed) {
    if (acc_path || cells)
      return fail(PDX_ERR_ARGUMENT, "typed pair models use the rows traversal with FP32 sums and no bonds");
    if (p->typed_n != N)
      return fail(PDX_ERR_DIMENSION, p->typed_n == 0 ? "typed pair model without its per-particle data "
                                                       "(pdx_pair_set_sigmas / pdx_pair_set_types)"
                                                     : "typed pair data and neighbor list particle counts differ");
  }
  if (cells) {
    if (acc_path) return fail(PDX_ERR_ARGUMENT, "the cell traversal uses FP32 sums without bonds");
    if (nl->allpairs) return fail(PDX_ERR_ARGUMENT, "the cell traversal needs a cell grid (not all-pairs rows)");
  }
  if (acc_path) {
    if (p->spec.coulomb) return fail(PDX_ERR_ARGUMENT, "accumulation modes and bonds are not available with Coulomb");
    if (p->spec.model != PDX_PAIR_LJ && p->spec.model != PDX_PAIR_WCA && p->spec.model != PDX_PAIR_SOFT)
      return fail(PDX_ERR_ARGUMENT, "accumulation modes and bonds need the LJ, WCA or soft model");
    if (p->lanes < 0) return fail(PDX_ERR_ARGUMENT, "accumulation modes and bonds use the lanes layout (lanes >= 0)");
    if (p->bonds && p->bonds->N != nl->N) return fail(PDX_ERR_DIMENSION, "bonds and neighbor list particle counts differ");
  }
  int G = p->lanes;
  if (G == 0) {
    // about 2^18 threads: enough waves per SIMD to hide the neighbour gathers while a wave's
    // row slots stay in few cache lines (measured on the 64 000-ion system: 4 lanes beat 2,
    // 8 and 16, and every split layout)
    const int64_t want = std::max<int64_t>(1, 262144 / std::max(N, 1));
    G = 1;
    while (G * 2 <= want && G < 64) G <<= 1;
    // rows of 32 entries and more take four lanes however many particles there are: the lanes of a
    // particle gather from the same few cells, so a wave touches 16 rows' neighbourhoods instead of
    // 64 (256 000 LJ atoms, 82 entries: 58 -> 40 us; 512 000 ions, 187 entries: 423 -> 304 us, with
    // 2 lanes 46 and 338, with 8 lanes 45 and 310). Short rows leave such lanes idle (1 M beads, 14
    // entries: 60 us with one lane, 76 with four), and the accumulation modes keep their split. Around
    // the line, 500 000 LJ atoms with one and four lanes: 19 entries 23.4 and 21.6 us (forces) and 35.5
    // and 44.3 (energies), 33 entries 39.9 and 30.1, 52.2 and 50.6; LJ + Coulomb energies cross later,
    // 33 entries 57.7 and 63.0, 42 entries 63.4 and 63.5, 54 entries 76.6 and 75.8.
    const double rl = std::sqrt((double)nl->rl2);
    const double rows = 4.1887902 * rl * rl * rl * N / (nl->box[0] * nl->box[1] * nl->box[2]);
    if (!acc_path && rows >= 32.0) G = std::max(G, 4);
  }
  if (acc_path) G = std::min(G, 8);
  const int shape = p->wide && G > 0 ? 0 : walk_shape(G, N);  // 0: one lane with 64-bit addresses
  if (shape >= 0) G = std::max(shape, 1);
  const int blocks = cells ? nl->ncell
                           : (G < 0 ? (N + WAVE - 1) / WAVE : (int)(((int64_t)N * G + TPB - 1) / TPB));
  double *partial = fixed_partial;
  if (energy && totals) {
    if (fixed_partial) {
      if (blocks > fixed_blocks)
        return fail(PDX_ERR_ARGUMENT, std::to_string(blocks) + " workgroups exceed the fixed workspace of " +
                                          std::to_string(fixed_blocks) + " (fewer particles or lanes, or pdx_pair_forces)");
    } else if ((size_t)blocks * 7 > p->partial.n) {
      PDX_HIP(hipStreamSynchronize(as_stream(stream)));
      int rc = p->partial.alloc((size_t)blocks * 7);
      if (rc) return rc;
    }
  }
  if (!fixed_partial) partial = p->partial.p;
  PairArgs a{};
  a.N = N;
  a.packed = nl->packed.p;
  a.nbr = nl->neighbors_flat.p;
  a.counts = nl->counts.p;
  a.state = nl->state.p;
  a.geom = nl->geom.p;
  a.fx = fx; a.fy = fy; a.fz = fz;
  a.Epot = Epot; a.V = V;
  a.totals = totals;
  a.partial = partial;
  a.add = (flags & PDX_ADD) ? 1 : 0;
  a.eps = p->eps; a.sig2 = p->sig2; a.rc2 = p->rc2; a.eshift = p->eshift;
  a.cC = p->cC; a.crc2 = p->crc2; a.csx = p->csx; a.ceshift = p->ceshift; a.halfself = p->halfself;
  // a row entry was within the list radius at the build and both particles moved at most skin/2
  a.reach = 1.001f * (float)(std::sqrt((double)nl->rl2) + nl->skin);
  a.sigp = p->sigp.p; a.typ = p->typ.p; a.tab = p->tab.p; a.ntypes = p->ntypes; a.rfac2 = p->rfac2;
  for (int k = 0; k < MAXC; ++k) { a.pe[k] = p->pe[k]; a.pf[k] = p->pf[k]; }
  const bool coul = p->spec.coulomb != 0;
  const int np = std::max(p->npe, p->npf);
  hipStream_t st = as_stream(stream);
  if (p->nexc > 0) {
    if (p->exc_n != N) return fail(PDX_ERR_DIMENSION, "exceptions and neighbor list particle counts differ");
    if (G < 0 && !cells) return fail(PDX_ERR_ARGUMENT, "exceptions use the lanes layout (lanes >= 0)");
    a.exo = p->exc_off.p;
    a.exj = p->exc_j.p;
    a.exs = p->exc_s.p;
  }
  // FP64 totals: per-block partials, then one block adds them in block order
  auto finish = [&]() -> int {
    PDX_LAUNCH_CHECK();
    if (energy && totals) {
      hipLaunchKernelGGL(k_sum_partials<7>, dim3(1), dim3(SUM_THREADS), 0, st, (const double *)partial, blocks,
                         totals, a.add, (const int64_t *)nl->state.p);
      PDX_LAUNCH_CHECK();
    }
    return PDX_OK;
  };
  if (cells) {
    CellArgs c{};
    c.sortedq = nl->sortedq.p;
    c.ids = nl->particle_ids_sorted.p;
    c.offsets = nl->cell_offsets.p;
    c.nx = nl->nx; c.ny = nl->ny; c.nz = nl->nz;
    float cut2 = p->spec.model != PDX_PAIR_NONE ? p->rc2 : 0.0f;
    if (coul) cut2 = std::max(cut2, p->crc2);
    c.cut2 = cut2;
    hipLaunchKernelGGL(k_refresh_sorted, dim3((N + TPB - 1) / TPB), dim3(TPB), 0, st, N, nl->particle_ids_sorted.p,
                       nl->packed.p, nl->sortedq.p, nl->state.p);
    const dim3 grid(nl->ncell);
    switch (p->spec.model) {
      case PDX_PAIR_LJ: launch_cells<PDX_PAIR_LJ>(coul, energy, np, grid, st, a, c); break;
      case PDX_PAIR_WCA: launch_cells<PDX_PAIR_WCA>(coul, energy, np, grid, st, a, c); break;
      case PDX_PAIR_SOFT: launch_cells<PDX_PAIR_SOFT>(coul, energy, np, grid, st, a, c); break;
      default: launch_cells<PDX_PAIR_NONE>(coul, energy, np, grid, st, a, c); break;
    }
    return finish();
  }
  if (acc_path) {
    const int bonded = (p->bonds != nullptr ? 1 : 0) | (p->bonds != nullptr && p->exclude_bonded ? 2 : 0);
    if (bonded) {
      a.boff = p->bonds->offsets.p;
      a.bpart = p->bonds->partners.p;
      a.binvalid = p->bonds->invalid.p;
      a.bk = (float)p->bonds->k;
      a.bR02 = (float)(p->bonds->R0 * p->bonds->R0);
    }
    if (p->spec.model == PDX_PAIR_LJ) launch_acc<PDX_PAIR_LJ>(p->accumulate, energy, shape, dim3(blocks), st, a, bonded);
    else if (p->spec.model == PDX_PAIR_WCA) launch_acc<PDX_PAIR_WCA>(p->accumulate, energy, shape, dim3(blocks), st, a, bonded);
    else launch_acc<PDX_PAIR_SOFT>(p->accumulate, energy, shape, dim3(blocks), st, a, bonded);
    return finish();
  }
  switch (p->spec.model) {
    case PDX_PAIR_MIXED_LJ: launch_typed<PDX_PAIR_MIXED_LJ>(coul, energy, np, shape, dim3(blocks), st, a); break;
    case PDX_PAIR_MIXED_WCA: launch_typed<PDX_PAIR_MIXED_WCA>(coul, energy, np, shape, dim3(blocks), st, a); break;
    case PDX_PAIR_MATRIX_LJ: launch_typed<PDX_PAIR_MATRIX_LJ>(coul, energy, np, shape, dim3(blocks), st, a); break;
    case PDX_PAIR_MATRIX_WCA: launch_typed<PDX_PAIR_MATRIX_WCA>(coul, energy, np, shape, dim3(blocks), st, a); break;
    case PDX_PAIR_LJ: launch_model<PDX_PAIR_LJ>(coul, energy, np, shape, dim3(blocks), st, a); break;
    case PDX_PAIR_WCA: launch_model<PDX_PAIR_WCA>(coul, energy, np, shape, dim3(blocks), st, a); break;
    case PDX_PAIR_SOFT: launch_model<PDX_PAIR_SOFT>(coul, energy, np, shape, dim3(blocks), st, a); break;
    default: launch_model<PDX_PAIR_NONE>(coul, energy, np, shape, dim3(blocks), st, a); break;
  }
  return finish();
}
}  // namespace

extern "C" int pdx_pair_forces(pdx_pair_t p, pdx_nl_t nl, float *fx, float *fy, float *fz, float *Epot,
                               float *V, double *totals, int32_t flags, pdx_stream_t stream) {
  return pair_forces_impl(p, nl, fx, fy, fz, Epot, V, totals, flags, stream, nullptr, 0);
}

extern "C" int pdx_pair_compute(pdx_pair_t p, pdx_nl_t nl, const float *x, const float *y, const float *z,
                                const float *q, float *fx, float *fy, float *fz, float *Epot, float *V, double *totals,
                                int32_t flags, pdx_stream_t stream) {
  if (!p || !nl) return fail(PDX_ERR_ARGUMENT, "null pair model or neighbor list");
  if (!x || !y || (!z && nl->dim == 3)) return fail(PDX_ERR_ARGUMENT, "null coordinate array");
  if (nl->packed_src[0] != x || nl->packed_src[1] != y || nl->packed_src[2] != z || nl->packed_src[3] != q)
    return fail(PDX_ERR_STATE, "the coordinates (and charges) differ from those the list's last check packed; "
                               "call pdx_nl_update / pdx_nl_check with them first");
  return pair_forces_impl(p, nl, fx, fy, fz, Epot, V, totals, flags, stream, nullptr, 0);
}

extern "C" int pdx_pair_set_sigmas(pdx_pair_t p, int32_t n, const float *sigma) {
  if (!p || (!sigma && n > 0)) return fail(PDX_ERR_ARGUMENT, "null argument");
  if (p->spec.model != PDX_PAIR_MIXED_LJ && p->spec.model != PDX_PAIR_MIXED_WCA)
    return fail(PDX_ERR_ARGUMENT, "per-particle diameters belong to the mixed-sigma models");
  if (n <= 0) return fail(PDX_ERR_ARGUMENT, "particle count must be positive");
  float smax = 0.f;
  for (int32_t i = 0; i < n; ++i) {
    if (!(std::isfinite(sigma[i]) && sigma[i] > 0)) return fail(PDX_ERR_ARGUMENT, "diameters must be finite and positive");
    smax = std::max(smax, sigma[i]);
  }
  PDX_HIP(hipDeviceSynchronize());
  int rc = p->sigp.alloc(n);
  if (rc) return rc;
  PDX_HIP(hipMemcpy(p->sigp.p, sigma, sizeof(float) * n, hipMemcpyHostToDevice));
  p->typed_n = n;
  p->typed_rmax = p->spec.cutoff * smax;
  return PDX_OK;
}

extern "C" int pdx_pair_set_types(pdx_pair_t p, int32_t n, int32_t ntypes, const int32_t *typ, const double *sigma,
                                  const double *epsilon, const double *rcut) {
  if (!p || !typ || !sigma || !epsilon || !rcut) return fail(PDX_ERR_ARGUMENT, "null argument");
  if (p->spec.model != PDX_PAIR_MATRIX_LJ && p->spec.model != PDX_PAIR_MATRIX_WCA)
    return fail(PDX_ERR_ARGUMENT, "type tables belong to the pair-matrix models");
  if (n <= 0) return fail(PDX_ERR_ARGUMENT, "particle count must be positive");
  if (ntypes < 1 || ntypes > 64) return fail(PDX_ERR_ARGUMENT, "ntypes must be in 1..64");
  for (int32_t i = 0; i < n; ++i)
    if (typ[i] < 1 || typ[i] > ntypes) return fail(PDX_ERR_ARGUMENT, "type ids must lie in 1..ntypes");
  // rows a*ntypes + b of (sigma^2, epsilon, rc^2, u(rc) with the shift) in FP32, from the
  // column-major matrices (element (a, b) at a + ntypes b)
  std::vector<float4> tab((size_t)ntypes * ntypes);
  double rmax = 0;
  for (int a = 0; a < ntypes; ++a)
    for (int b = 0; b < ntypes; ++b) {
      const size_t k = (size_t)a + (size_t)ntypes * b;
      const double sg = sigma[k], ep = epsilon[k], rc = rcut[k];
      if (!(std::isfinite(sg) && sg > 0 && std::isfinite(ep) && std::isfinite(rc) && rc >= 0))
        return fail(PDX_ERR_ARGUMENT, "pair sigma must be positive, epsilon and rcut finite, rcut >= 0");
      const float s2 = (float)sg * (float)sg, r2 = (float)rc * (float)rc;
      float esh = 0.f;
      if (p->spec.model == PDX_PAIR_MATRIX_LJ && p->spec.shift && rc > 0) {
        // lj_cutoff_energy (PairModels.jl:20-25) per pair
        const float x2 = s2 / r2, x6 = x2 * x2 * x2;
        esh = 4.0f * (float)ep * (x6 * x6 - x6);
      }
      tab[(size_t)a * ntypes + b] = make_float4(s2, (float)ep, r2, esh);
      rmax = std::max(rmax, rc);
    }
  PDX_HIP(hipDeviceSynchronize());
  int rc;
  if ((rc = p->typ.alloc(n)) || (rc = p->tab.alloc(tab.size()))) return rc;
  PDX_HIP(hipMemcpy(p->typ.p, typ, sizeof(int32_t) * n, hipMemcpyHostToDevice));
  PDX_HIP(hipMemcpy(p->tab.p, tab.data(), sizeof(float4) * tab.size(), hipMemcpyHostToDevice));
  p->typed_n = n;
  p->ntypes = ntypes;
  p->typed_rmax = rmax;
  return PDX_OK;
}

extern "C" int pdx_pair_cutoff(pdx_pair_t p, double *rc) {
  if (!p || !rc) return fail(PDX_ERR_ARGUMENT, "null argument");
  double r = 0;
  switch (p->spec.model) {
    case PDX_PAIR_LJ: r = p->spec.cutoff; break;
    case PDX_PAIR_WCA: r = std::sqrt(1.2599211) * p->spec.sigma; break;
    case PDX_PAIR_SOFT: r = p->spec.sigma; break;
    case PDX_PAIR_NONE: r = 0; break;
    default:
      if (p->typed_n == 0) return fail(PDX_ERR_STATE, "typed pair model without its per-particle data");
      r = p->typed_rmax;
  }
  if (p->spec.coulomb) r = std::max(r, p->spec.coulomb_cutoff);
  *rc = r;
  return PDX_OK;
}

extern "C" int pdx_pair_set_bond_exclusion(pdx_pair_t p, int32_t exclude) {
  if (!p) return fail(PDX_ERR_ARGUMENT, "null pair model");
  if (exclude && p->spec.coulomb)
    return fail(PDX_ERR_ARGUMENT, "bonded exclusions of charged pairs go through the Coulomb exceptions");
  p->exclude_bonded = exclude != 0;
  return PDX_OK;
}

extern "C" int pdx_pair_set_accumulation(pdx_pair_t p, int32_t mode) {
  if (!p) return fail(PDX_ERR_ARGUMENT, "null pair model");
  if (mode != PDX_ACC_FP32 && mode != PDX_ACC_FIXED64 && mode != PDX_ACC_FP64)
    return fail(PDX_ERR_ARGUMENT, "accumulation mode must be PDX_ACC_FP32, PDX_ACC_FIXED64 or PDX_ACC_FP64");
  p->accumulate = mode;
  return PDX_OK;
}

extern "C" int pdx_bonds_create(int32_t n, int32_t nbond, const int32_t *bi, const int32_t *bj, double k, double R0,
                                pdx_bonds_t *out) {
  if (!out) return fail(PDX_ERR_ARGUMENT, "null argument");
  *out = nullptr;
  if (n < 1 || nbond < 0) return fail(PDX_ERR_ARGUMENT, "particle and bond counts must be positive");
  if (nbond > 0 && (!bi || !bj)) return fail(PDX_ERR_ARGUMENT, "null bond arrays");
  if (!(std::isfinite(k) && k >= 0)) return fail(PDX_ERR_ARGUMENT, "FENE k must be finite and nonnegative");
  if (!(std::isfinite(R0) && R0 > 0 && std::isfinite(R0 * R0)))
    return fail(PDX_ERR_ARGUMENT, "FENE R0 and its square must be finite and positive");
  std::vector<int32_t> cnt(n + 1, 0);
  for (int b = 0; b < nbond; ++b) {
    if (bi[b] < 0 || bi[b] >= n || bj[b] < 0 || bj[b] >= n || bi[b] == bj[b])
      return fail(PDX_ERR_ARGUMENT, "bond " + std::to_string(b) + " names an invalid particle pair");
    ++cnt[bi[b] + 1];
    ++cnt[bj[b] + 1];
  }
  for (int i = 0; i < n; ++i) cnt[i + 1] += cnt[i];
  std::vector<int32_t> part(2 * (size_t)nbond), fill(cnt.begin(), cnt.end() - 1);
  for (int b = 0; b < nbond; ++b) {
    part[fill[bi[b]]++] = bj[b];
    part[fill[bj[b]]++] = bi[b];
  }
  for (int i = 0; i < n; ++i) std::sort(part.begin() + cnt[i], part.begin() + cnt[i + 1]);  // fixed order
  auto *b = new pdx_bonds_s();
  b->N = n;
  b->nbond = nbond;
  b->k = k;
  b->R0 = R0;
  int rc;
  if ((rc = b->offsets.alloc(n + 1)) || (rc = b->partners.alloc(std::max<size_t>(1, part.size()))) ||
      (rc = b->invalid.alloc(1))) {
    delete b;
    return rc;
  }
  const int32_t none = INT32_MAX;
  if (hipMemcpy(b->offsets.p, cnt.data(), sizeof(int32_t) * (n + 1), hipMemcpyHostToDevice) != hipSuccess ||
      (nbond > 0 && hipMemcpy(b->partners.p, part.data(), sizeof(int32_t) * part.size(), hipMemcpyHostToDevice) != hipSuccess) ||
      hipMemcpy(b->invalid.p, &none, sizeof(int32_t), hipMemcpyHostToDevice) != hipSuccess) {
    delete b;
    return fail(PDX_ERR_DEVICE, "bond table upload failed");
  }
  *out = b;
  return PDX_OK;
}

extern "C" int pdx_bonds_destroy(pdx_bonds_t b) {
  delete b;
  return PDX_OK;
}

extern "C" int pdx_pair_set_bonds(pdx_pair_t p, pdx_bonds_t b) {
  if (!p) return fail(PDX_ERR_ARGUMENT, "null pair model");
  p->bonds = b;
  return PDX_OK;
}

extern "C" int pdx_bonds_status(pdx_bonds_t b, int32_t *first_invalid, int32_t reset, pdx_stream_t stream) {
  if (!b || !first_invalid) return fail(PDX_ERR_ARGUMENT, "null argument");
  hipStream_t st = as_stream(stream);
  int32_t v = INT32_MAX;
  PDX_HIP(hipMemcpyAsync(&v, b->invalid.p, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  PDX_HIP(hipStreamSynchronize(st));
  if (reset && v != INT32_MAX) {
    const int32_t none = INT32_MAX;
    PDX_HIP(hipMemcpyAsync(b->invalid.p, &none, sizeof(int32_t), hipMemcpyHostToDevice, st));
    PDX_HIP(hipStreamSynchronize(st));
  }
  *first_invalid = v == INT32_MAX ? -1 : v;
  if (v != INT32_MAX)
    return fail(PDX_ERR_COORDINATE, "FENE bond incident on particle " + std::to_string(v + 1) +
                                        " has nonfinite length or r >= R0=" + std::to_string(b->R0) +
                                        ". Reduce the timestep or correct the configuration; forces are not clamped.");
  return PDX_OK;
}

extern "C" int pdx_pair_set_exceptions(pdx_pair_t p, int32_t n, int32_t nexc, const int32_t *ei, const int32_t *ej,
                                       const double *scale) {
  if (!p) return fail(PDX_ERR_ARGUMENT, "null pair model");
  if (nexc < 0 || n < 1) return fail(PDX_ERR_ARGUMENT, "particle and exception counts must be positive");
  if (nexc > 0 && (!ei || !ej || !scale)) return fail(PDX_ERR_ARGUMENT, "null exception arrays");
  if (nexc > 0 && !p->spec.coulomb) return fail(PDX_ERR_ARGUMENT, "exceptions need the real-space Coulomb term");
  // validate and deduplicate (normalize_exceptions, Spec.jl:200-224); key (min, max)
  std::vector<std::pair<std::pair<int32_t, int32_t>, double>> items;
  items.reserve(nexc);
  for (int k = 0; k < nexc; ++k) {
    const int32_t a = ei[k], b = ej[k];
    const double s = scale[k];
    if (a < 0 || a >= n || b < 0 || b >= n)
      return fail(PDX_ERR_ARGUMENT, "Exception pair (" + std::to_string(a + 1) + ", " + std::to_string(b + 1) +
                                        ") is out of range for N=" + std::to_string(n) + ".");
    if (a == b)
      return fail(PDX_ERR_ARGUMENT, "Exception pair (" + std::to_string(a + 1) + ", " + std::to_string(b + 1) +
                                        ") refers to a single particle.");
    if (!(std::isfinite(s) && s >= 0))
      return fail(PDX_ERR_ARGUMENT, "Exception scale must be finite and nonnegative.");
    items.push_back({{std::min(a, b), std::max(a, b)}, s});
  }
  std::sort(items.begin(), items.end(), [](const auto &x, const auto &y) { return x.first < y.first; });
  std::vector<std::pair<std::pair<int32_t, int32_t>, double>> uniq;
  for (const auto &it : items) {
    if (!uniq.empty() && uniq.back().first == it.first) {
      if (uniq.back().second != it.second)
        return fail(PDX_ERR_ARGUMENT, "Exception pair (" + std::to_string(it.first.first + 1) + ", " +
                                          std::to_string(it.first.second + 1) + ") is listed with conflicting scales.");
      continue;
    }
    uniq.push_back(it);
  }
  std::vector<int32_t> off(n + 1, 0);
  size_t m = 0;
  for (const auto &it : uniq) {
    if (it.second == 1.0) continue;
    ++off[it.first.first + 1];
    ++off[it.first.second + 1];
    m += 2;
  }
  for (int i = 0; i < n; ++i) off[i + 1] += off[i];
  std::vector<int32_t> jj(std::max<size_t>(m, 1)), fill(off.begin(), off.end() - 1);
  std::vector<float> ss(std::max<size_t>(m, 1));
  for (const auto &it : uniq) {  // sorted by (i, j): each particle's list is in id order
    if (it.second == 1.0) continue;
    const int32_t a = it.first.first, b = it.first.second;
    jj[fill[a]] = b; ss[fill[a]++] = (float)it.second;
    jj[fill[b]] = a; ss[fill[b]++] = (float)it.second;
  }
  for (int i = 0; i < n; ++i) {  // partners of i in id order (the b-side entries arrive out of order)
    std::vector<std::pair<int32_t, float>> row;
    for (int t = off[i]; t < off[i + 1]; ++t) row.push_back({jj[t], ss[t]});
    std::sort(row.begin(), row.end());
    for (int t = off[i]; t < off[i + 1]; ++t) { jj[t] = row[t - off[i]].first; ss[t] = row[t - off[i]].second; }
  }
  p->nexc = 0;
  p->exc_n = n;
  if (m == 0) return PDX_OK;
  int rc;
  if ((rc = p->exc_off.alloc(n + 1)) || (rc = p->exc_j.alloc(m)) || (rc = p->exc_s.alloc(m))) return rc;
  PDX_HIP(hipMemcpy(p->exc_off.p, off.data(), sizeof(int32_t) * (n + 1), hipMemcpyHostToDevice));
  PDX_HIP(hipMemcpy(p->exc_j.p, jj.data(), sizeof(int32_t) * m, hipMemcpyHostToDevice));
  PDX_HIP(hipMemcpy(p->exc_s.p, ss.data(), sizeof(float) * m, hipMemcpyHostToDevice));
  p->nexc = (int32_t)(m / 2);
  return PDX_OK;
}

extern "C" int pdx_pair_set_lanes(pdx_pair_t p, int32_t lanes) {
  if (!p) return fail(PDX_ERR_ARGUMENT, "null pair model");
  if (lanes > 0 && (lanes > 64 || (lanes & (lanes - 1))))
    return fail(PDX_ERR_ARGUMENT, "lanes per particle must be a power of two in 1..64");
  if (lanes < 0 && !(lanes == -2 || lanes == -4 || lanes == -8 || lanes == -16))
    return fail(PDX_ERR_ARGUMENT, "split layouts use 2, 4, 8 or 16 waves (lanes = -2, -4, -8, -16)");
  if (lanes < 0 && (typed_model(p->spec.model) || p->nexc > 0 || p->bonds || p->accumulate != PDX_ACC_FP32))
    return fail(PDX_ERR_ARGUMENT, "typed models, exceptions, bonds and accumulation modes use the lanes layout (lanes >= 0)");
  p->lanes = lanes;
  return PDX_OK;
}

extern "C" int pdx_pair_set_traversal(pdx_pair_t p, int32_t mode) {
  if (!p) return fail(PDX_ERR_ARGUMENT, "null pair model");
  if (mode != PDX_TRAVERSAL_ROWS && mode != PDX_TRAVERSAL_CELLS)
    return fail(PDX_ERR_ARGUMENT, "traversal must be PDX_TRAVERSAL_ROWS or PDX_TRAVERSAL_CELLS");
  p->traversal = mode;
  return PDX_OK;
}

extern "C" int pdx_test_pair_wide(pdx_pair_t p, int32_t on) {
  if (!p) return fail(PDX_ERR_ARGUMENT, "null pair model");
  p->wide = on != 0;
  return PDX_OK;
}
