// Pair kernels over the list's rows and cells and their launches by model (pdx_pairs.hip calls the
// launches; one translation unit per model instantiates them, so that they compile side by side).
#pragma once

#include "pdx_internal.hpp"
#include "pdx_pairmath.hpp"
#include "pdx_rowwalk.hpp"

namespace pdx {
namespace pairk {

constexpr int TPB = 256;
constexpr int MAXC = 24;

struct PairArgs {
  int N;
  const float4 *packed;
  const int32_t *nbr;
  const int32_t *counts;
  const int64_t *state;
  const float *geom;
  float *fx, *fy, *fz, *Epot, *V;
  double *totals;
  double *partial;
  int add;
  float eps, sig2, rc2, eshift;   // LJ / WCA / soft
  float cC, crc2, csx, ceshift, halfself;
  float pe[MAXC];
  float pf[MAXC];
  // Coulomb exceptions (k_pair with COUL): CSR over particles, scale per entry
  const int32_t *exo, *exj;
  const float *exs;
  // FENE bonds (k_pair_acc only)
  const int32_t *boff, *bpart;
  int32_t *binvalid;
  float bk, bR02;
  // typed models (k_pair only): per-particle diameters, or 1-based types and the type-pair table
  const float *sigp;
  const int32_t *typ;
  const float4 *tab;  // (sig2, eps, rc2, eshift), row a*ntypes + b
  int ntypes;
  float rfac2;
  float reach;  // a particle further than this from every face has no row entry across the seam
};


// Writes of one particle's sums (lane that owns it; every STEP-th lane owns one) and the FP64 totals
// of the launch.
template <bool COUL, bool ENERGY, int STEP = 1>
__device__ __forceinline__ void pair_epilogue(const PairArgs &a, bool owner, int i, float qi, float ax, float ay,
                                              float az, float e, const float (&v)[6]) {
  float ei = 0.f, w[6] = {0, 0, 0, 0, 0, 0};
  if (owner) {
    if (a.add) {
      a.fx[i] += ax; a.fy[i] += ay; a.fz[i] += az;
    } else {
      a.fx[i] = ax; a.fy[i] = ay; a.fz[i] = az;
    }
    if (ENERGY) {
      // half of every pair (each is visited from both ends) plus the Coulomb self energy
      ei = 0.5f * e;
      if (COUL) ei -= a.halfself * qi * qi;
#pragma unroll
      for (int c = 0; c < 6; ++c) w[c] = 0.5f * v[c];
      if (a.Epot) a.Epot[i] = a.add ? a.Epot[i] + ei : ei;
      if (a.V) {
#pragma unroll
        for (int c = 0; c < 6; ++c) {
          float *p = a.V + (size_t)c * a.N + i;
          *p = a.add ? *p + w[c] : w[c];
        }
      }
    }
  }
  if (ENERGY && a.totals) {
    const double d[7] = {(double)ei, (double)w[0], (double)w[1], (double)w[2],
                         (double)w[3], (double)w[4], (double)w[5]};
    block_partials_every<7, STEP>(d, a.partial);
  }
}

// The row walk of the lanes layouts: lane `lane` of particle i's G lanes takes slots lane, lane + G,
// ... of its row, U at a time, and calls visit(jj, pj, dx, dy, dz) with U entries: U independent
// gathers in flight. Bound by VALU issue, so the visit's overhead is kept out of the vector unit:
//  - iterations that every lane of the wave has in full (counted once) take no bounds test, and the
//    next iteration's ids are loaded while this one is evaluated; only the ragged end tests (entries
//    past a row's end point at i itself, whose r^2 = 0 every model excludes);
//  - loads are buffer loads with a scalar base and a 32-bit lane offset: the row's is constant (the
//    base moves on), a gather's is its id shifted, so an address costs at most one instruction;
//  - a wave whose particles all lie further than a.reach from every face has no row entry across
//    the periodic seam and skips that test (row_deltas).
// With energies a visit of the LJ + Coulomb rows went from 93 to 78 vector instructions (66 of them
// pair terms; 486 400 ions, 4 lanes: 258 -> 242 us, 64 000 ions: 37 -> 32 us). Forces only it is 49,
// fewer than the gather's share of the L1 (75 clocks per wave and visit), which then bounds the walk
// (224 -> 220 us).
// Lists beyond the 32-bit offsets even with one lane (walk_shape) take 64-bit addresses: WIDE.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
constexpr int BUFFER_RAW = 0x00020000;  // word 3 of a raw buffer resource on gfx9
template <int G, int U, bool WIDE, class VISIT>
__device__ __forceinline__ void walk_rows(const PairArgs &a, const float4 &pi, int i, int lane, bool active, int n,
                                          float hx, float hy, float hz, float Lx, float Ly, float Lz, VISIT visit) {
  const int N = a.N;
  const bool near_face = active & ((fabsf(pi.x) > hx - a.reach) | (fabsf(pi.y) > hy - a.reach) |
                                   (fabsf(pi.z) > hz - a.reach));
  const bool seam = __ballot(near_face) != 0;
  // ids are 1-based: the resource starts one particle early
  const auto prs = __builtin_amdgcn_make_buffer_rsrc((void *)(a.packed - 1), 0, (int)walk_records(N), BUFFER_RAW);
  auto eval = [&](const int (&id)[U]) {
    float4 pj[U];
    int jj[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      jj[u] = id[u] - 1;
      if (WIDE) {
        pj[u] = a.packed[jj[u]];
      } else {
        const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(prs, (int)walk_gather(id[u]), 0, 0);
        pj[u] = make_float4(__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w));
      }
    }
    float dx[U], dy[U], dz[U];
    if (seam) {
      row_deltas<U>(pi, pj, hx, hy, hz, Lx, Ly, Lz, dx, dy, dz);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        dx[u] = pi.x - pj[u].x;
        dy[u] = pi.y - pj[u].y;
        dz[u] = pi.z - pj[u].z;
      }
    }
    visit(jj, pj, dx, dy, dz);
  };
  const int32_t *row = a.nbr + i;
  const int2 range = wave_range<G>(n);
  const int full = WIDE ? 0 : range.x / (U * G);
  const int its = (range.y + U * G - 1) / (U * G);
  const int vo = (int)walk_lane(lane, N, i);
  auto load = [&](int k, int (&id)[U]) {
    if (k < full) {
      const auto rrs = __builtin_amdgcn_make_buffer_rsrc((void *)(a.nbr + (size_t)k * (U * G) * N), 0, -1, BUFFER_RAW);
#pragma unroll
      for (int u = 0; u < U; ++u) id[u] = (int)__builtin_amdgcn_raw_buffer_load_b32(rrs, vo, (int)walk_step(u, G, N), 0);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int t = (k * U + u) * G + lane;
        id[u] = i + 1;
        if (t < n) id[u] = row[(size_t)t * N];
      }
    }
  };
  int nx[U];
  if (its > 0) load(0, nx);
  for (int k = 0; k < its; ++k) {
    int id[U];
#pragma unroll
    for (int u = 0; u < U; ++u) id[u] = nx[u];
    if (k + 1 < its) load(k + 1, nx);
    eval(id);
  }
}

// Waves a SIMD that the row kernels are held to. The row loop waits for its gathers, so it is the highest
// number that leaves the loop without scratch accesses: forces only 8 (64 registers), with energies 6 (80),
// less where the Coulomb polynomials meet per-pair coefficients or one lane's longer index arithmetic.
// Spilled at 8, pair matrices with Coulomb took 13.1 us (20 000 particles, forces) and 24.8 us (64 000),
// mixed diameters 11.6 and 20.8 us; at 7 waves 10.5 and 20.1, 9.5 and 18.5 us.
__host__ __device__ constexpr int pair_waves(int model, bool coul, bool energy, int G, int NP) {
  const bool typed = typed_model(model), soft = model == PDX_PAIR_SOFT;
  if (energy) return coul && G == 1 && (typed || (soft && NP > 16)) ? 5 : 6;
  if (G == 1) return coul && typed ? 6 : (coul || typed ? 7 : 8);
  return coul && (typed || soft) ? 7 : 8;
}

// Layout A: G lanes of one wave per particle, xor-shuffle reduction. Forces-only launches evaluate
// every pair with pair_terms in row order (at a given lane count the sums are then the same bits whatever
// the traversal's bookkeeping, which trajectories keep); energy launches use the joined terms.
template <int MODEL, bool COUL, bool ENERGY, int G, int NP, bool WIDE = false>
__global__ __launch_bounds__(TPB, pair_waves(MODEL, COUL, ENERGY, G, NP)) void k_pair(const PairArgs a) {
  const int64_t *s = a.state;
  const bool valid = s[PDX_DN_VALID] != 0 && s[PDX_DN_ERROR] == 0;  // uniform
  if (!valid) return;
  const int gid = blockIdx.x * TPB + threadIdx.x;
  const int i = gid / G;
  const int lane = gid % G;
  const int N = a.N;
  const bool active = i < N;
  const int ic = active ? i : N - 1;
  const float Lx = a.geom[0], Ly = a.geom[1], Lz = a.geom[2];
  const float hx = 0.5f * Lx, hy = 0.5f * Ly, hz = 0.5f * Lz;
  float ax = 0.f, ay = 0.f, az = 0.f, e = 0.f;
  float v[6] = {0, 0, 0, 0, 0, 0};
  float pe[NP], pf[NP];
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    pe[k] = a.pe[k];
    pf[k] = a.pf[k];
  }
  constexpr bool TYPED = typed_model(MODEL);
  constexpr bool MIXED = MODEL == PDX_PAIR_MIXED_LJ || MODEL == PDX_PAIR_MIXED_WCA;
  const float4 pi = a.packed[ic];
  const float qi = active ? pi.w : 0.f;
  const float cqi = a.cC * qi;
  if (COUL && ENERGY && !TYPED) pe[0] = a.pe[0] - a.ceshift;
  {
    // typed models: i's diameter, or its type's row of the table
    const float ci = MIXED ? a.sigp[ic] : 0.f;
    const int ti = (TYPED && !MIXED) ? (a.typ[ic] - 1) * a.ntypes : 0;
    constexpr int U = WALK_U;
    walk_rows<G, U, WIDE>(a, pi, ic, lane, active, active ? a.counts[ic] : 0, hx, hy, hz, Lx, Ly, Lz,
                    [&](const int (&jj)[U], const float4 (&pj)[U], const float (&ddx)[U], const float (&ddy)[U],
                        const float (&ddz)[U]) {
      float cj[U];
      int tj[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        cj[u] = MIXED ? a.sigp[jj[u]] : 0.f;
        tj[u] = (TYPED && !MIXED) ? a.typ[jj[u]] - 1 : 0;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float dx = ddx[u], dy = ddy[u], dz = ddz[u];
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        float f, uu;
        if (TYPED)
          pair_terms_c<MODEL, COUL, ENERGY, NP>(a, typed_coef<MODEL>(a, ci, cj[u], ti, tj[u]), pe, pf, qi, pj[u].w,
                                                r2, f, uu);
        else if (ENERGY)
          pair_terms_joint<MODEL, COUL, ENERGY, NP>(a, pe, pf, cqi, pj[u].w, r2, f, uu);
        else
          pair_terms<MODEL, COUL, ENERGY, NP>(a, pe, pf, qi, pj[u].w, r2, f, uu);
        ax = fmaf(f, dx, ax);
        ay = fmaf(f, dy, ay);
        az = fmaf(f, dz, az);
        if (ENERGY) {
          e += uu;
          const float fxij = f * dx, fyij = f * dy, fzij = f * dz;
          v[0] = fmaf(dx, fxij, v[0]); v[1] = fmaf(dy, fyij, v[1]); v[2] = fmaf(dz, fzij, v[2]);
          v[3] = fmaf(dx, fyij, v[3]); v[4] = fmaf(dx, fzij, v[4]); v[5] = fmaf(dy, fzij, v[5]);
        }
      }
    });
    if (COUL && a.exo && active && qi != 0.0f) {
      // exceptions: + C q_i q_j (s - 1) / r at the minimum image, no cutoff, no potential shift
      for (int p = a.exo[i] + lane; p < a.exo[i + 1]; p += G) {
        const float4 pj = a.packed[a.exj[p]];
        const float sc = a.cC * qi * pj.w * (a.exs[p] - 1.0f);
        const float dx = periodic_delta(pi.x, pj.x, hx, Lx);
        const float dy = periodic_delta(pi.y, pj.y, hy, Ly);
        const float dz = periodic_delta(pi.z, pj.z, hz, Lz);
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        const float invr = __builtin_amdgcn_rsqf(r2);
        const float f = sc * invr * invr * invr;
        ax = fmaf(f, dx, ax);
        ay = fmaf(f, dy, ay);
        az = fmaf(f, dz, az);
        if (ENERGY) {
          e += sc * invr + (r2 < a.crc2 ? a.cC * qi * pj.w * a.ceshift : 0.0f);
          const float fxij = f * dx, fyij = f * dy, fzij = f * dz;
          v[0] = fmaf(dx, fxij, v[0]); v[1] = fmaf(dy, fyij, v[1]); v[2] = fmaf(dz, fzij, v[2]);
          v[3] = fmaf(dx, fyij, v[3]); v[4] = fmaf(dx, fzij, v[4]); v[5] = fmaf(dy, fzij, v[5]);
        }
      }
    }
  }
  if (G > 1) {
    ax = wave_sum_width(ax, G);
    ay = wave_sum_width(ay, G);
    az = wave_sum_width(az, G);
    if (ENERGY) {
      e = wave_sum_width(e, G);
#pragma unroll
      for (int c = 0; c < 6; ++c) v[c] = wave_sum_width(v[c], G);
    }
  }
  pair_epilogue<COUL, ENERGY, G>(a, active && lane == 0, i, qi, ax, ay, az, e, v);
}

// Layout B (large systems): a block owns 64 consecutive particles and S waves; wave w walks
// slots w, w+S, ... of all 64 rows, so every row load is one contiguous 256-byte access of
// the slot-major table, and the S partial sums meet in LDS.
template <int MODEL, bool COUL, bool ENERGY, int S, int NP>
__global__ __launch_bounds__(64 * S) void k_pair_split(const PairArgs a) {
  const int64_t *st = a.state;
  const bool valid = st[PDX_DN_VALID] != 0 && st[PDX_DN_ERROR] == 0;  // uniform
  if (!valid) return;
  constexpr int NV = ENERGY ? 10 : 3;
  __shared__ float red[S][NV][WAVE];
  const int lane = threadIdx.x & (WAVE - 1);
  const int w = threadIdx.x / WAVE;
  const int i = blockIdx.x * WAVE + lane;
  const int N = a.N;
  const bool active = i < N;
  const float Lx = a.geom[0], Ly = a.geom[1], Lz = a.geom[2];
  const float hx = 0.5f * Lx, hy = 0.5f * Ly, hz = 0.5f * Lz;
  float acc[NV];
#pragma unroll
  for (int c = 0; c < NV; ++c) acc[c] = 0.f;
  float qi = 0.f;
  float pe[NP], pf[NP];
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    pe[k] = a.pe[k];
    pf[k] = a.pf[k];
  }
  if (active) {
    const float4 pi = a.packed[i];
    qi = pi.w;
    const float cqi = a.cC * qi;
    if (COUL && ENERGY) pe[0] = a.pe[0] - a.ceshift;
    const int n = a.counts[i];
    const int32_t *row = a.nbr + i;
    int jn = w < n ? row[(size_t)w * N] - 1 : 0;
    for (int t = w; t < n; t += S) {
      const int j = jn;
      if (t + S < n) jn = row[(size_t)(t + S) * N] - 1;
      const float4 pj = a.packed[j];
      const float dx = periodic_delta(pi.x, pj.x, hx, Lx);
      const float dy = periodic_delta(pi.y, pj.y, hy, Ly);
      const float dz = periodic_delta(pi.z, pj.z, hz, Lz);
      const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
      float f, u;
      if (ENERGY) pair_terms_joint<MODEL, COUL, ENERGY, NP>(a, pe, pf, cqi, pj.w, r2, f, u);
      else pair_terms<MODEL, COUL, ENERGY, NP>(a, pe, pf, qi, pj.w, r2, f, u);
      acc[0] = fmaf(f, dx, acc[0]);
      acc[1] = fmaf(f, dy, acc[1]);
      acc[2] = fmaf(f, dz, acc[2]);
      if (ENERGY) {
        acc[3] += u;
        const float fxij = f * dx, fyij = f * dy, fzij = f * dz;
        acc[4] = fmaf(dx, fxij, acc[4]); acc[5] = fmaf(dy, fyij, acc[5]); acc[6] = fmaf(dz, fzij, acc[6]);
        acc[7] = fmaf(dx, fyij, acc[7]); acc[8] = fmaf(dx, fzij, acc[8]); acc[9] = fmaf(dy, fzij, acc[9]);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < NV; ++c) red[w][c][lane] = acc[c];
  __syncthreads();
  float sum[NV];
#pragma unroll
  for (int c = 0; c < NV; ++c) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < S; ++k) t += red[k][c][lane];  // fixed order: deterministic
    sum[c] = t;
  }
  float v[6] = {0, 0, 0, 0, 0, 0};
  if (ENERGY) {
#pragma unroll
    for (int c = 0; c < 6; ++c) v[c] = sum[4 + c];
  }
  pair_epilogue<COUL, ENERGY>(a, active && w == 0, i, qi, sum[0], sum[1], sum[2], ENERGY ? sum[3] : 0.f, v);
}

// ---- cell traversal: no rows. One workgroup per home cell of the list's grid stages the
// current (x, y, z, q) of its 27 neighbour cells into LDS (cell order, 2048 candidates per
// chunk), then each wave takes home particles in turn: 64 candidates at a time are tested
// against the cutoff, the hits are ballot-compacted into a wave-private LDS queue in candidate
// order and evaluated 64 at a time with every lane busy. Candidate order (cells z, y, x, then
// ids inside a cell) and all sums are fixed, so results are deterministic.
struct CellArgs {
  const float4 *sortedq;          // current (x, y, z, q) in cell order
  const int32_t *ids;             // 1-based storage id of cell slot t
  const int32_t *offsets;         // 1-based cell offsets (ncell + 1)
  int nx, ny, nz;
  float cut2;                     // the largest cutoff^2 of the pair terms
};

constexpr int CSTAGE = 2048;  // staged candidates per chunk (32 KiB)
constexpr int CHOME = 192;    // home particles per pass (their partial sums live in LDS)

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int MODEL, bool COUL, bool ENERGY, int NP>
__global__ __launch_bounds__(TPB) void k_pair_cells(const PairArgs a, const CellArgs c) {
  const int64_t *st = a.state;
  const bool valid = st[PDX_DN_VALID] != 0 && st[PDX_DN_ERROR] == 0;  // uniform
  if (!valid) return;
  constexpr int WPB = TPB / WAVE;
  constexpr int NACC = ENERGY ? 10 : 3;
  __shared__ float4 stage[CSTAGE];
  __shared__ float4 queue[WPB][2 * WAVE];
  __shared__ float accs[CHOME][NACC];
  __shared__ int seg_start[27], seg_pre[28];
  const int w = threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
  const unsigned long long below = (1ull << lane) - 1ull;
  const int nx = c.nx, ny = c.ny, nz = c.nz;
  const int home = blockIdx.x;
  const int cx = home % nx, cy = (home / nx) % ny, cz = home / (nx * ny);
  const float Lx = a.geom[0], Ly = a.geom[1], Lz = a.geom[2];
  const float hx = 0.5f * Lx, hy = 0.5f * Ly, hz = 0.5f * Lz;
  float pe[NP], pf[NP];
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    pe[k] = a.pe[k];
    pf[k] = a.pf[k];
  }
  if (threadIdx.x < 27) {
    const int k = threadIdx.x;
    int z2 = cz + k / 9 - 1, y2 = cy + (k / 3) % 3 - 1, x2 = cx + k % 3 - 1;
    z2 += z2 < 0 ? nz : 0; z2 -= z2 >= nz ? nz : 0;
    y2 += y2 < 0 ? ny : 0; y2 -= y2 >= ny ? ny : 0;
    x2 += x2 < 0 ? nx : 0; x2 -= x2 >= nx ? nx : 0;
    const int cc = (z2 * ny + y2) * nx + x2;
    seg_start[k] = c.offsets[cc] - 1;
    seg_pre[k + 1] = c.offsets[cc + 1] - c.offsets[cc];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    seg_pre[0] = 0;
    for (int k = 1; k <= 27; ++k) seg_pre[k] += seg_pre[k - 1];
  }
  __syncthreads();
  const int total = seg_pre[27];
  const int hs = c.offsets[home] - 1, he = c.offsets[home + 1] - 1;
  float4 *Q = queue[w];
  double tot[7] = {0, 0, 0, 0, 0, 0, 0};
  for (int hg = hs; hg < he; hg += CHOME) {  // uniform
    const int hn = min(CHOME, he - hg);
    for (int k = threadIdx.x; k < hn * NACC; k += TPB) (&accs[0][0])[k] = 0.f;
    for (int c0 = 0; c0 < total; c0 += CSTAGE) {  // uniform
      const int nch = min(CSTAGE, total - c0);
      __syncthreads();  // the previous chunk is no longer read
      for (int f = threadIdx.x; f < nch; f += TPB) {
        const int g = c0 + f;
        int sg = 0;
        while (seg_pre[sg + 1] <= g) ++sg;
        stage[f] = c.sortedq[seg_start[sg] + (g - seg_pre[sg])];
      }
      __syncthreads();
      for (int p = w; p < hn; p += WPB) {
        const int t = hg + p;
        const float4 pi = c.sortedq[t];
        const float qi = pi.w;
        float ax = 0.f, ay = 0.f, az = 0.f, e = 0.f;
        float v[6] = {0, 0, 0, 0, 0, 0};
        auto evaluate = [&](int cnt) {
          if (lane < cnt) {
            const float4 d = Q[lane];
            const float r2 = fmaf(d.x, d.x, fmaf(d.y, d.y, d.z * d.z));
            float f, uu;
            pair_terms<MODEL, COUL, ENERGY, NP>(a, pe, pf, qi, d.w, r2, f, uu);
            ax = fmaf(f, d.x, ax);
            ay = fmaf(f, d.y, ay);
            az = fmaf(f, d.z, az);
            if (ENERGY) {
              e += uu;
              const float fxij = f * d.x, fyij = f * d.y, fzij = f * d.z;
              v[0] = fmaf(d.x, fxij, v[0]); v[1] = fmaf(d.y, fyij, v[1]); v[2] = fmaf(d.z, fzij, v[2]);
              v[3] = fmaf(d.x, fyij, v[3]); v[4] = fmaf(d.x, fzij, v[4]); v[5] = fmaf(d.y, fzij, v[5]);
            }
          }
        };
        int qn = 0;  // uniform
        for (int k0 = 0; k0 < nch; k0 += WAVE) {
          const int k = k0 + lane;
          bool hit = false;
          float4 d = make_float4(0.f, 0.f, 0.f, 0.f);
          if (k < nch) {  // the particle itself has r^2 = 0, which every pair term excludes
            const float4 pj = stage[k];
            d.x = periodic_delta(pi.x, pj.x, hx, Lx);
            d.y = periodic_delta(pi.y, pj.y, hy, Ly);
            d.z = periodic_delta(pi.z, pj.z, hz, Lz);
            d.w = pj.w;
            hit = fmaf(d.x, d.x, fmaf(d.y, d.y, d.z * d.z)) < c.cut2;
          }
          const unsigned long long m = __ballot(hit);
          if (hit) Q[qn + __popcll(m & below)] = d;
          qn += __popcll(m);
          if (qn >= WAVE) {
            wave_lds_sync();
            evaluate(WAVE);
            const float4 rest = lane < qn - WAVE ? Q[WAVE + lane] : make_float4(0.f, 0.f, 0.f, 0.f);
            wave_lds_sync();
            if (lane < qn - WAVE) Q[lane] = rest;
            qn -= WAVE;
            wave_lds_sync();
          }
        }
        wave_lds_sync();
        evaluate(qn);
        wave_lds_sync();
        if (COUL && a.exo && c0 == 0 && qi != 0.0f) {
          const int i = c.ids[t] - 1;
          for (int q = a.exo[i] + lane; q < a.exo[i + 1]; q += WAVE) {
            const float4 pj = a.packed[a.exj[q]];
            const float sc = a.cC * qi * pj.w * (a.exs[q] - 1.0f);
            const float dx = periodic_delta(pi.x, pj.x, hx, Lx);
            const float dy = periodic_delta(pi.y, pj.y, hy, Ly);
            const float dz = periodic_delta(pi.z, pj.z, hz, Lz);
            const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            const float invr = __builtin_amdgcn_rsqf(r2);
            const float f = sc * invr * invr * invr;
            ax = fmaf(f, dx, ax);
            ay = fmaf(f, dy, ay);
            az = fmaf(f, dz, az);
            if (ENERGY) {
              e += sc * invr + (r2 < a.crc2 ? a.cC * qi * pj.w * a.ceshift : 0.0f);
              const float fxij = f * dx, fyij = f * dy, fzij = f * dz;
              v[0] = fmaf(dx, fxij, v[0]); v[1] = fmaf(dy, fyij, v[1]); v[2] = fmaf(dz, fzij, v[2]);
              v[3] = fmaf(dx, fyij, v[3]); v[4] = fmaf(dx, fzij, v[4]); v[5] = fmaf(dy, fzij, v[5]);
            }
          }
        }
        ax = wave_sum_width(ax, WAVE);
        ay = wave_sum_width(ay, WAVE);
        az = wave_sum_width(az, WAVE);
        if (ENERGY) {
          e = wave_sum_width(e, WAVE);
#pragma unroll
          for (int k = 0; k < 6; ++k) v[k] = wave_sum_width(v[k], WAVE);
        }
        if (lane == 0) {  // only this wave touches particle p: chunk sums in chunk order
          accs[p][0] += ax; accs[p][1] += ay; accs[p][2] += az;
          if (ENERGY) {
            accs[p][3] += e;
#pragma unroll
            for (int k = 0; k < 6; ++k) accs[p][4 + k] += v[k];
          }
        }
      }
    }
    __syncthreads();
    // outputs of the pass: thread per home particle (half energies and half virials)
    for (int p = threadIdx.x; p < hn; p += TPB) {
      const int t = hg + p;
      const int i = c.ids[t] - 1;
      const float qi = c.sortedq[t].w;
      const float fx = accs[p][0], fy = accs[p][1], fz = accs[p][2];
      if (a.add) {
        a.fx[i] += fx; a.fy[i] += fy; a.fz[i] += fz;
      } else {
        a.fx[i] = fx; a.fy[i] = fy; a.fz[i] = fz;
      }
      if (ENERGY) {
        float ei = 0.5f * accs[p][3];
        if (COUL) ei -= a.halfself * qi * qi;
        float wv[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) wv[k] = 0.5f * accs[p][4 + k];
        if (a.Epot) a.Epot[i] = a.add ? a.Epot[i] + ei : ei;
        if (a.V) {
#pragma unroll
          for (int k = 0; k < 6; ++k) {
            float *q = a.V + (size_t)k * a.N + i;
            *q = a.add ? *q + wv[k] : wv[k];
          }
        }
        tot[0] += (double)ei;
#pragma unroll
        for (int k = 0; k < 6; ++k) tot[1 + k] += (double)wv[k];
      }
    }
  }
  if (ENERGY && a.totals) block_partials<7>(tot, a.partial);
}

template <int MODEL, bool COUL, bool ENERGY, int NP>
void launch_cells_np(dim3 grid, hipStream_t st, const PairArgs &a, const CellArgs &c) {
  hipLaunchKernelGGL((k_pair_cells<MODEL, COUL, ENERGY, NP>), grid, dim3(TPB), 0, st, a, c);
}

template <int MODEL>
void launch_cells(bool coul, bool energy, int np, dim3 grid, hipStream_t st, const PairArgs &a, const CellArgs &c) {
  if (coul) {
    if (np <= 16) {
      if (energy) launch_cells_np<MODEL, true, true, 16>(grid, st, a, c);
      else launch_cells_np<MODEL, true, false, 16>(grid, st, a, c);
    } else {
      if (energy) launch_cells_np<MODEL, true, true, 24>(grid, st, a, c);
      else launch_cells_np<MODEL, true, false, 24>(grid, st, a, c);
    }
  } else {
    if (energy) launch_cells_np<MODEL, false, true, 1>(grid, st, a, c);
    else launch_cells_np<MODEL, false, false, 1>(grid, st, a, c);
  }
}

// ---- per-particle sums in a chosen precision (the bead-spring precision study). The pair
// arithmetic is that of k_pair's forces-only launches (pair_terms in FP32), with energies too; only the
// accumulation of the row sums changes: FP32 (fma, as k_pair), 64-bit fixed point at 2^32 (exact, so
// independent of the order and of the lane split), or FP64 (exact products, rounded sums).
template <int ACC> struct Sum;
template <> struct Sum<PDX_ACC_FP32> {
  float v = 0.f;
  __device__ __forceinline__ void add_prod(float a, float b) { v = fmaf(a, b, v); }
  __device__ __forceinline__ void add(float a) { v += a; }
  __device__ __forceinline__ double value() const { return (double)v; }
  template <int G> __device__ __forceinline__ void combine() {
#pragma unroll
    for (int o = G >> 1; o >= 1; o >>= 1) v += __shfl_xor(v, o, G);
  }
};
template <> struct Sum<PDX_ACC_FIXED64> {
  long long v = 0;
  __device__ __forceinline__ void add_prod(float a, float b) { v += __float2ll_rn(a * b * 4294967296.0f); }
  __device__ __forceinline__ void add(float a) { v += __float2ll_rn(a * 4294967296.0f); }
  __device__ __forceinline__ double value() const { return (double)v * 2.3283064365386962890625e-10; }
  template <int G> __device__ __forceinline__ void combine() {
#pragma unroll
    for (int o = G >> 1; o >= 1; o >>= 1) v += __shfl_xor(v, o, G);
  }
};
template <> struct Sum<PDX_ACC_FP64> {
  double v = 0.0;
  __device__ __forceinline__ void add_prod(float a, float b) { v += (double)a * (double)b; }
  __device__ __forceinline__ void add(float a) { v += (double)a; }
  __device__ __forceinline__ double value() const { return v; }
  template <int G> __device__ __forceinline__ void combine() {
#pragma unroll
    for (int o = G >> 1; o >= 1; o >>= 1) v += __shfl_xor(v, o, G);
  }
};

template <int MODEL, bool ENERGY, int G, int ACC, bool WIDE = false>
__global__ __launch_bounds__(TPB, ACC == PDX_ACC_FP32 ? (ENERGY ? 6 : 7) : 1) void k_pair_acc(const PairArgs a,
                                                                                             int bonded) {
  const int64_t *s = a.state;
  const bool valid = s[PDX_DN_VALID] != 0 && s[PDX_DN_ERROR] == 0;  // uniform
  if (!valid) return;
  const int gid = blockIdx.x * TPB + threadIdx.x;
  const int i = gid / G;
  const int lane = gid % G;
  const int N = a.N;
  const bool active = i < N;
  const float Lx = a.geom[0], Ly = a.geom[1], Lz = a.geom[2];
  const float hx = 0.5f * Lx, hy = 0.5f * Ly, hz = 0.5f * Lz;
  Sum<ACC> ax, ay, az, e, v[6];
  const float none[1] = {0.f};
  const int ic = active ? i : N - 1;
  {
    const float4 pi = a.packed[ic];
    const int n = active ? a.counts[ic] : 0;
    // bonded exclusions (BondExclusionFeature, src/engine/Bonded.jl:60-92): a row entry that is
    // one of i's bond partners gets no pair term; the first four partners live in registers
    const bool excl = (bonded & 2) != 0;
    int bp[4] = {-1, -1, -1, -1};
    int bx0 = 0, nbx = 0;
    if (excl) {
      bx0 = a.boff[ic];
      nbx = a.boff[ic + 1] - bx0;
#pragma unroll
      for (int k = 0; k < 4; ++k) bp[k] = k < nbx ? a.bpart[bx0 + k] : -1;
    }
    constexpr int U = WALK_U;
    walk_rows<G, U, WIDE>(a, pi, ic, lane, active, n, hx, hy, hz, Lx, Ly, Lz,
                    [&](const int (&jj)[U], const float4 (&)[U], const float (&ddx)[U], const float (&ddy)[U],
                        const float (&ddz)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float dx = ddx[u], dy = ddy[u], dz = ddz[u];
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        float f, uu;
        pair_terms<MODEL, false, ENERGY, 1>(a, none, none, 0.f, 0.f, r2, f, uu);
        if (excl) {
          bool ex = (jj[u] == bp[0]) | (jj[u] == bp[1]) | (jj[u] == bp[2]) | (jj[u] == bp[3]);
          for (int k = 4; k < nbx; ++k) ex |= a.bpart[bx0 + k] == jj[u];
          f = ex ? 0.f : f;
          uu = ex ? 0.f : uu;
        }
        ax.add_prod(f, dx);
        ay.add_prod(f, dy);
        az.add_prod(f, dz);
        if (ENERGY) {
          e.add(uu);
          const float fxij = f * dx, fyij = f * dy, fzij = f * dz;
          v[0].add_prod(dx, fxij); v[1].add_prod(dy, fyij); v[2].add_prod(dz, fzij);
          v[3].add_prod(dx, fyij); v[4].add_prod(dx, fzij); v[5].add_prod(dy, fzij);
        }
      }
    });
    if ((bonded & 1) && active) {
      const int b0 = a.boff[i], nb = a.boff[i + 1] - b0;
      const float R02 = a.bR02;
      for (int t = lane; t < nb; t += G) {
        const float4 pj = a.packed[a.bpart[b0 + t]];
        const float dx = periodic_delta(pi.x, pj.x, hx, Lx);
        const float dy = periodic_delta(pi.y, pj.y, hy, Ly);
        const float dz = periodic_delta(pi.z, pj.z, hz, Lz);
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        if (!(r2 < R02)) {  // out of the FENE domain (or not finite): latch, add nothing
          atomicMin(a.binvalid, i);
          continue;
        }
        // subtraction before division keeps near-limit extensions; log1p for short bonds
        // (_fene_denom, _fene_log, src/bonded/FENEBondCUDA.jl)
        const float denom = (R02 - r2) / R02;
        const float f = -a.bk / denom;
        ax.add_prod(f, dx);
        ay.add_prod(f, dy);
        az.add_prod(f, dz);
        if (ENERGY) {
          const float lg = r2 < 0.5f * R02 ? log1pf(-r2 / R02) : logf(denom);
          e.add(-0.5f * a.bk * R02 * lg);
          const float fxij = f * dx, fyij = f * dy, fzij = f * dz;
          v[0].add_prod(dx, fxij); v[1].add_prod(dy, fyij); v[2].add_prod(dz, fzij);
          v[3].add_prod(dx, fyij); v[4].add_prod(dx, fzij); v[5].add_prod(dy, fzij);
        }
      }
    }
  }
  if (G > 1) {
    ax.template combine<G>();
    ay.template combine<G>();
    az.template combine<G>();
    if (ENERGY) {
      e.template combine<G>();
#pragma unroll
      for (int c = 0; c < 6; ++c) v[c].template combine<G>();
    }
  }
  // every pair and bond was visited from both ends: half energies and half virials
  const bool owner = active && lane == 0;
  double ei = 0.0, w[6] = {0, 0, 0, 0, 0, 0};
  if (owner) {
    const float fx = (float)ax.value(), fy = (float)ay.value(), fz = (float)az.value();
    if (a.add) {
      a.fx[i] += fx; a.fy[i] += fy; a.fz[i] += fz;
    } else {
      a.fx[i] = fx; a.fy[i] = fy; a.fz[i] = fz;
    }
    if (ENERGY) {
      ei = 0.5 * e.value();
#pragma unroll
      for (int c = 0; c < 6; ++c) w[c] = 0.5 * v[c].value();
      if (a.Epot) a.Epot[i] = a.add ? a.Epot[i] + (float)ei : (float)ei;
      if (a.V) {
#pragma unroll
        for (int c = 0; c < 6; ++c) {
          float *p = a.V + (size_t)c * a.N + i;
          *p = a.add ? *p + (float)w[c] : (float)w[c];
        }
      }
    }
  }
  if (ENERGY && a.totals) {
    const double d[7] = {ei, w[0], w[1], w[2], w[3], w[4], w[5]};
    block_partials<7>(d, a.partial);
  }
}

template <int MODEL, bool ENERGY, int ACC>
void launch_acc_g(int G /* 0: one lane, 64-bit addresses */, dim3 grid, hipStream_t st, const PairArgs &a,
                  int bonded) {
  switch (G) {
    case 0: hipLaunchKernelGGL((k_pair_acc<MODEL, ENERGY, 1, ACC, true>), grid, dim3(TPB), 0, st, a, bonded); break;
    case 1: hipLaunchKernelGGL((k_pair_acc<MODEL, ENERGY, 1, ACC>), grid, dim3(TPB), 0, st, a, bonded); break;
    case 2: hipLaunchKernelGGL((k_pair_acc<MODEL, ENERGY, 2, ACC>), grid, dim3(TPB), 0, st, a, bonded); break;
    case 4: hipLaunchKernelGGL((k_pair_acc<MODEL, ENERGY, 4, ACC>), grid, dim3(TPB), 0, st, a, bonded); break;
    default: hipLaunchKernelGGL((k_pair_acc<MODEL, ENERGY, 8, ACC>), grid, dim3(TPB), 0, st, a, bonded); break;
  }
}

template <int MODEL>
void launch_acc(int acc, bool energy, int G, dim3 grid, hipStream_t st, const PairArgs &a, int bonded) {
  if (acc == PDX_ACC_FIXED64) {
    if (energy) launch_acc_g<MODEL, true, PDX_ACC_FIXED64>(G, grid, st, a, bonded);
    else launch_acc_g<MODEL, false, PDX_ACC_FIXED64>(G, grid, st, a, bonded);
  } else if (acc == PDX_ACC_FP64) {
    if (energy) launch_acc_g<MODEL, true, PDX_ACC_FP64>(G, grid, st, a, bonded);
    else launch_acc_g<MODEL, false, PDX_ACC_FP64>(G, grid, st, a, bonded);
  } else {
    if (energy) launch_acc_g<MODEL, true, PDX_ACC_FP32>(G, grid, st, a, bonded);
    else launch_acc_g<MODEL, false, PDX_ACC_FP32>(G, grid, st, a, bonded);
  }
}

template <int MODEL, bool COUL, bool ENERGY, int NP>
void launch_g(int G, dim3 grid, hipStream_t st, const PairArgs &a) {
  if (G < 0) {  // split layout, S = -G waves per 64 particles
    const dim3 sg((a.N + WAVE - 1) / WAVE);
    switch (-G) {
      case 2: hipLaunchKernelGGL((k_pair_split<MODEL, COUL, ENERGY, 2, NP>), sg, dim3(128), 0, st, a); break;
      case 4: hipLaunchKernelGGL((k_pair_split<MODEL, COUL, ENERGY, 4, NP>), sg, dim3(256), 0, st, a); break;
      case 8: hipLaunchKernelGGL((k_pair_split<MODEL, COUL, ENERGY, 8, NP>), sg, dim3(512), 0, st, a); break;
      default: hipLaunchKernelGGL((k_pair_split<MODEL, COUL, ENERGY, 16, NP>), sg, dim3(1024), 0, st, a); break;
    }
    return;
  }
  switch (G) {
    case 0: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 1, NP, true>), grid, dim3(TPB), 0, st, a); break;
    case 1: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 1, NP>), grid, dim3(TPB), 0, st, a); break;
    case 2: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 2, NP>), grid, dim3(TPB), 0, st, a); break;
    case 4: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 4, NP>), grid, dim3(TPB), 0, st, a); break;
    case 8: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 8, NP>), grid, dim3(TPB), 0, st, a); break;
    case 16: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 16, NP>), grid, dim3(TPB), 0, st, a); break;
    case 32: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 32, NP>), grid, dim3(TPB), 0, st, a); break;
    default: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 64, NP>), grid, dim3(TPB), 0, st, a); break;
  }
}

// Typed models: the lanes layout only.
template <int MODEL, bool COUL, bool ENERGY, int NP>
void launch_typed_g(int G, dim3 grid, hipStream_t st, const PairArgs &a) {
  switch (G) {
    case 0: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 1, NP, true>), grid, dim3(TPB), 0, st, a); break;
    case 1: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 1, NP>), grid, dim3(TPB), 0, st, a); break;
    case 2: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 2, NP>), grid, dim3(TPB), 0, st, a); break;
    case 4: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 4, NP>), grid, dim3(TPB), 0, st, a); break;
    case 8: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 8, NP>), grid, dim3(TPB), 0, st, a); break;
    case 16: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 16, NP>), grid, dim3(TPB), 0, st, a); break;
    case 32: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 32, NP>), grid, dim3(TPB), 0, st, a); break;
    default: hipLaunchKernelGGL((k_pair<MODEL, COUL, ENERGY, 64, NP>), grid, dim3(TPB), 0, st, a); break;
  }
}

template <int MODEL>
void launch_typed(bool coul, bool energy, int np, int G, dim3 grid, hipStream_t st, const PairArgs &a) {
  if (coul) {
    if (np <= 16) {
      if (energy) launch_typed_g<MODEL, true, true, 16>(G, grid, st, a);
      else launch_typed_g<MODEL, true, false, 16>(G, grid, st, a);
    } else {
      if (energy) launch_typed_g<MODEL, true, true, 24>(G, grid, st, a);
      else launch_typed_g<MODEL, true, false, 24>(G, grid, st, a);
    }
  } else {
    if (energy) launch_typed_g<MODEL, false, true, 1>(G, grid, st, a);
    else launch_typed_g<MODEL, false, false, 1>(G, grid, st, a);
  }
}

// Coulomb polynomials are zero-padded to 14, 16 or 24 monomials (Horner over exact zeros); the
// 9-10 A real-space fits at 1e-5 take 13-14.
template <int MODEL>
void launch_model(bool coul, bool energy, int np, int G, dim3 grid, hipStream_t st, const PairArgs &a) {
  if (coul) {
    if (np <= 14) {
      if (energy) launch_g<MODEL, true, true, 14>(G, grid, st, a);
      else launch_g<MODEL, true, false, 14>(G, grid, st, a);
    } else if (np <= 16) {
      if (energy) launch_g<MODEL, true, true, 16>(G, grid, st, a);
      else launch_g<MODEL, true, false, 16>(G, grid, st, a);
    } else {
      if (energy) launch_g<MODEL, true, true, 24>(G, grid, st, a);
      else launch_g<MODEL, true, false, 24>(G, grid, st, a);
    }
  } else {
    if (energy) launch_g<MODEL, false, true, 1>(G, grid, st, a);
    else launch_g<MODEL, false, false, 1>(G, grid, st, a);
  }
}

// instantiated in pdx_pairs_lj.hip, pdx_pairs_wca.hip, pdx_pairs_soft.hip, pdx_pairs_coulomb.hip and
// pdx_pairs_typed.hip
#define PDX_UNIFORM(M)                                                                                          \
  extern template void launch_model<M>(bool, bool, int, int, dim3, hipStream_t, const PairArgs &);              \
  extern template void launch_cells<M>(bool, bool, int, dim3, hipStream_t, const PairArgs &, const CellArgs &);
#define PDX_ACC_OF(M) extern template void launch_acc<M>(int, bool, int, dim3, hipStream_t, const PairArgs &, int);
#define PDX_TYPED(M) extern template void launch_typed<M>(bool, bool, int, int, dim3, hipStream_t, const PairArgs &);
PDX_UNIFORM(PDX_PAIR_LJ) PDX_UNIFORM(PDX_PAIR_WCA) PDX_UNIFORM(PDX_PAIR_SOFT) PDX_UNIFORM(PDX_PAIR_NONE)
PDX_ACC_OF(PDX_PAIR_LJ) PDX_ACC_OF(PDX_PAIR_WCA) PDX_ACC_OF(PDX_PAIR_SOFT)
PDX_TYPED(PDX_PAIR_MIXED_LJ) PDX_TYPED(PDX_PAIR_MIXED_WCA) PDX_TYPED(PDX_PAIR_MATRIX_LJ) PDX_TYPED(PDX_PAIR_MATRIX_WCA)
#undef PDX_UNIFORM
#undef PDX_ACC_OF
#undef PDX_TYPED

}  // namespace pairk
}  // namespace pdx
