// Batched independent replica boxes (LJ / WCA), each advanced by velocity Verlet, all of them
// in one persistent launch: one workgroup owns one replica for every step, so replicas never
// synchronise with each other and a step costs no kernel launch. Per step, inside the
// workgroup:
//   B  exclusive scan of the cell counts (LDS);
//   C  scatter (x, y, z, id) into cell order in LDS;
//   D  each cell's slice put in atom-id order (stable order: the traversal, and with it the
//      FP32 force sums, depend only on the replica's own coordinates);
//   E  forces from the LDS-resident sorted coordinates over the (2S+1)^3 stencil of cells of
//      side >= rc/S (or over all atoms for boxes with fewer than 2S+1 cells a side, as the
//      reference's all-pairs rows, DenseNeighborCUDA.jl:128-151), then the closing kick
//      v += c f (_nve_kick3_kernel!, src/SimulationCore.jl:581-591), the next step's kick-drift
//      v += c f, x += dt v, wrap to [-L/2, L/2) (_nve_kick_drift3_kernel!,
//      src/simulation/NVEFusion.jl:3-24) and the drifted atom's cell count.
// Atom state (x, v) stays in HBM / L2 between phases; the sorted coordinates, the cell table and
// the next counts live in LDS (up to 8192 atoms: 128 KiB of float4, within gfx950's 160 KiB).
// The launch lasts as long as its largest replica, one workgroup alone on its CU (its coordinates
// fill the LDS) and bound by VALU issue in E, so E visits few candidates and spends little on each:
// a stencil is walked as (2S+1)^2 rows of cells, contiguous in LDS; a row further than rc is left
// out and the others are cut to the cells a sphere of rc reaches; a row's image shift is subtracted
// from the atom once instead of testing every pair. 512 boxes of 256..8192 atoms, 20 steps: 31.0 ms
// with 27-cell stencils, a separate kick-drift pass and 512 threads, 8.5 ms now (0.42 ms a step).
#include "pdx_internal.hpp"

#include <algorithm>
#include <cmath>
#include <numeric>
#include <vector>

using namespace pdx;

namespace {

constexpr int NMAX = 8192;   // atoms per replica (LDS-resident sorted coordinates)
constexpr int NCMAX = 6000;  // cells per replica (their 16-bit starts and counts, 24 KiB, fit beside NMAX atoms)
constexpr int RED_BYTES = 1024;

struct Rep {
  int off, n;
  int model;     // PDX_PAIR_LJ / PDX_PAIR_WCA
  int S;         // stencil half-width in cells; 0: all pairs
  int nc[3];     // cells per dimension
  float L[3], halfL[3], cinv[3], cw[3];  // box, half box, cells per unit length, cell width
  float slack;                           // bound of the rounding of a cell edge
  float eps, sig2, rc2, eshift;
};

__device__ __forceinline__ int cell_coord(float x, float halfL, float cinv, int nc) {
  int c = (int)((x + halfL) * cinv);
  return c < 0 ? 0 : (c >= nc ? nc - 1 : c);
}

__device__ __forceinline__ float wrap_centred(float x, float L) {
  x -= (x >= 0.5f * L) ? L : 0.0f;
  x += (x < -0.5f * L) ? L : 0.0f;
  return x;
}

// Coordinates outside the box are a caller's, or of an atom that crossed more than the box in one step,
// which wrap_centred shifts once. Cells and pair distances are then taken from the image in the box.
__device__ __forceinline__ bool outside_box(const Rep &R, float x, float y, float z) {
  return !(fabsf(x) <= R.halfL[0] && fabsf(y) <= R.halfL[1] && fabsf(z) <= R.halfL[2]);
}
__device__ __forceinline__ float into_box(float x, float halfL, float L) {
  return fabsf(x) <= halfL ? x : x - L * floorf((x + halfL) / L);
}

// Force factor f (force on i = f d) and energy u of one pair (same arithmetic as the ELL
// pair kernel: 24e(2s^12 - s^6)/r^2; u = 4e(s^12 - s^6) - u_c, or + e for WCA).
__device__ __forceinline__ void lj_terms(const Rep &R, float r2, float &f, float &u) {
  const bool in = (r2 > 0.f) & (r2 < R.rc2);
  const float invr2 = __builtin_amdgcn_rcpf(r2);
  const float s2 = R.sig2 * invr2;
  const float s6 = s2 * s2 * s2;
  const float s12 = s6 * s6;
  f = in ? 24.0f * R.eps * (2.0f * s12 - s6) * invr2 : 0.f;
  u = in ? 4.0f * R.eps * (s12 - s6) + (R.model == PDX_PAIR_WCA ? R.eps : -R.eshift) : 0.f;
}

template <int BS>
__device__ __forceinline__ double block_sum(double v, double *red) {
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < BS / WAVE; ++w) s += red[w];
  return s;
}

// Lanes per atom of the force phase: two share the atoms of a small box on all pairs (16 boxes of 200
// atoms, 10 steps: 316 -> 177 us), where each lane's half is as long. The rows of a stencil are cut to a
// sphere and share badly: with two and four lanes 16 boxes of 700 atoms took 785 and 1 256 us, with one
// 502. A function of the replica alone, as the lanes' partial sums are part of its arithmetic.
__host__ __device__ inline int atom_lanes(const Rep &R) { return R.S == 0 && R.n <= 256 ? 2 : 1; }

// Forces on the atom at p (slot s): every G-th atom from sub on of a box on all pairs, else the stencil's
// rows of cells in row order, every row in x order. ENERGY also sums the pair energies and r.F.
template <bool ENERGY>
__device__ __forceinline__ void atom_forces(const Rep &R, const float4 *spos, const unsigned short *cst, int n,
                                            const float4 &p, int s, int sub, int G, float &ax, float &ay, float &az,
                                            float &e, float &w) {
  auto pair = [&](float dx, float dy, float dz) {
    const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
    float f, u;
    lj_terms(R, r2, f, u);
    ax = fmaf(f, dx, ax); ay = fmaf(f, dy, ay); az = fmaf(f, dz, az);
    if (ENERGY) {
      e += u;
      w = fmaf(f, r2, w);
    }
  };
  if (R.S == 0) {
    for (int j = sub; j < n; j += G) {
      const float4 q = spos[j];
      pair(mic_fast(p.x - q.x, R.halfL[0], R.L[0]), mic_fast(p.y - q.y, R.halfL[1], R.L[1]),
           mic_fast(p.z - q.z, R.halfL[2], R.L[2]));
    }
    return;
  }
  const int S = R.S;
  const int nx = R.nc[0], ny = R.nc[1], nz = R.nc[2];
  const int cx = cell_coord(p.x, R.halfL[0], R.cinv[0], nx);
  const int cy = cell_coord(p.y, R.halfL[1], R.cinv[1], ny);
  const int cz = cell_coord(p.z, R.halfL[2], R.cinv[2], nz);
  // 0 <= ux <= L whatever the coordinate (one that no shift brings into the box, NaN): with it every
  // row has x0 <= nx - 1 and x1 >= 0, and no cell outside the table is read
  const float ux = __builtin_amdgcn_fmed3f(p.x + R.halfL[0], 0.f, R.L[0]);
  for (int oz = -S; oz <= S; ++oz) {
    // a row's distance from the atom in z and y, less a slack that covers the rounding of the edges
    const float gz = (float)(cz + oz) * R.cw[2] - R.halfL[2];
    float dz = oz > 0 ? gz - p.z : (oz < 0 ? p.z - (gz + R.cw[2]) : 0.f);
    dz = fmaxf(dz - R.slack, 0.f);
    const float remz = fmaf(-dz, dz, R.rc2);
    int z2 = cz + oz;
    float pz = p.z;
    if (z2 < 0) { z2 += nz; pz += R.L[2]; } else if (z2 >= nz) { z2 -= nz; pz -= R.L[2]; }
    for (int oy = -S; oy <= S; ++oy) {
      const float gy = (float)(cy + oy) * R.cw[1] - R.halfL[1];
      float dy = oy > 0 ? gy - p.y : (oy < 0 ? p.y - (gy + R.cw[1]) : 0.f);
      dy = fmaxf(dy - R.slack, 0.f);
      const float rem = fmaf(-dy, dy, remz);
      if (!(rem > 0.f)) continue;
      const float xr = __builtin_amdgcn_sqrtf(rem) + R.slack;  // (its ulp is within the slack)
      const int x0 = max((int)floorf((ux - xr) * R.cinv[0]), cx - S);
      const int x1 = min((int)floorf((ux + xr) * R.cinv[0]), cx + S);
      int y2 = cy + oy;
      float py = p.y;
      if (y2 < 0) { y2 += ny; py += R.L[1]; } else if (y2 >= ny) { y2 -= ny; py -= R.L[1]; }
      // cells x0..x1 of the row as at most two runs of slots, one per image; one loop over both, as
      // most waves hold atoms at both ends of a row. An odd last step pairs the atom with itself.
      const unsigned short *cs = cst + (z2 * ny + y2) * nx;
      const bool left = x0 < 0, right = x1 >= nx;
      const float p0 = left ? p.x + R.L[0] : p.x, p1 = left ? p.x : p.x - R.L[0];
      const int b0 = cs[left ? x0 + nx : x0], l0 = (int)cs[left || right ? nx : x1 + 1] - b0;
      int b1 = 0, tot = l0;
      if (left | right) {
        b1 = cs[0];
        tot += (int)cs[(left ? x1 : x1 - nx) + 1] - b1;
        b1 -= l0;
      }
      for (int k = 0; k < tot; k += 2) {
        const bool i0 = k < l0, i1 = k + 1 < l0;
        const float4 q0 = spos[k + (i0 ? b0 : b1)];
        const float4 q1 = spos[k + 1 < tot ? k + 1 + (i1 ? b0 : b1) : s];
        pair((i0 ? p0 : p1) - q0.x, py - q0.y, pz - q0.z);
        pair((i1 ? p0 : p1) - q1.x, py - q1.y, pz - q1.z);
      }
    }
  }
}

template <int BS>
__global__ __launch_bounds__(BS) void k_replicas(const Rep *__restrict__ reps, const int32_t *__restrict__ order,
                                                 float *x, float *y, float *z, float *vx, float *vy, float *vz,
                                                 float *fx, float *fy, float *fz, int32_t *key, float c, float dt,
                                                 float mass, int nsteps, int first_force, int energy, int reg0,
                                                 int reg1, int reg2, double *out) {
  extern __shared__ float4 smem[];
  float4 *spos = smem;
  char *base0 = reinterpret_cast<char *>(smem) + reg0;
  unsigned short *cst = reinterpret_cast<unsigned short *>(base0);     // cell starts
  unsigned *cnt = reinterpret_cast<unsigned *>(base0 + reg1);          // next counts, two 16-bit cells a word
  int *wsum = reinterpret_cast<int *>(base0 + reg1 + reg2);  // 16 wave sums
  int *outside = wsum + 16;                                  // an atom of the coming step is outside the box
  double *red = reinterpret_cast<double *>(base0 + reg1 + reg2 + 128);

  const int rid = order[blockIdx.x];
  const Rep R = reps[rid];
  const int t = threadIdx.x, lane = t & (WAVE - 1), wave = t / WAVE;
  const int n = R.n, off = R.off;
  const bool allpairs = R.S == 0;
  const int ncell = allpairs ? 0 : R.nc[0] * R.nc[1] * R.nc[2];
  const int chunk = (ncell + BS - 1) / BS;
  const int G = atom_lanes(R);
  double pe = 0.0, ke = 0.0, vir = 0.0;

  // the atom's cell for the next scatter: its rank among the cell's atoms so far
  auto bin = [&](int g, float px, float py, float pz) {
    if (allpairs) return;
    if (outside_box(R, px, py, pz)) {
      px = into_box(px, R.halfL[0], R.L[0]);
      py = into_box(py, R.halfL[1], R.L[1]);
      pz = into_box(pz, R.halfL[2], R.L[2]);
      *outside = 1;
    }
    const int cell = (cell_coord(pz, R.halfL[2], R.cinv[2], R.nc[2]) * R.nc[1] +
                      cell_coord(py, R.halfL[1], R.cinv[1], R.nc[1])) * R.nc[0] +
                     cell_coord(px, R.halfL[0], R.cinv[0], R.nc[0]);
    const int sh = 16 * (cell & 1);
    const unsigned r = (atomicAdd(&cnt[cell >> 1], 1u << sh) >> sh) & 0xffffu;
    key[g] = (int)((unsigned)cell | (r << 16));
  };
  // opening half kick, drift and wrap of one atom
  auto kick_drift = [&](int g, float ux, float uy, float uz, float px, float py, float pz) {
    vx[g] = ux; vy[g] = uy; vz[g] = uz;
    px = wrap_centred(fmaf(dt, ux, px), R.L[0]);
    py = wrap_centred(fmaf(dt, uy, py), R.L[1]);
    pz = wrap_centred(fmaf(dt, uz, pz), R.L[2]);
    x[g] = px; y[g] = py; z[g] = pz;
    bin(g, px, py, pz);
  };

  for (int k = t; k < (ncell + 1) / 2; k += BS) cnt[k] = 0u;
  if (t == 0) *outside = 0;
  __syncthreads();
  for (int i = t; i < n; i += BS) {
    const int g = off + i;
    if (first_force) bin(g, x[g], y[g], z[g]);
    else kick_drift(g, fmaf(c, fx[g], vx[g]), fmaf(c, fy[g], vy[g]), fmaf(c, fz[g], vz[g]), x[g], y[g], z[g]);
  }
  __syncthreads();
  for (int step = first_force ? 0 : 1; step <= nsteps; ++step) {
    const bool integrate = step > 0;
    const bool last = step == nsteps;
    bool images = false;  // some atom's coordinates are not its slot's
    if (!allpairs) {
      // ---- B: exclusive scan of the counts (contiguous chunk per thread, wave scans)
      const int k0 = min(t * chunk, ncell), k1 = min(k0 + chunk, ncell);
      auto count = [&](int k) { return (int)((cnt[k >> 1] >> (16 * (k & 1))) & 0xffffu); };
      int sum = 0;
      for (int k = k0; k < k1; ++k) sum += count(k);
      int v = sum;
#pragma unroll
      for (int o = 1; o < WAVE; o <<= 1) {
        const int u = __shfl_up(v, o, WAVE);
        if (lane >= o) v += u;
      }
      if (lane == WAVE - 1) wsum[wave] = v;
      __syncthreads();
      int base = v - sum;
      for (int w = 0; w < wave; ++w) base += wsum[w];
      for (int k = k0; k < k1; ++k) {
        cst[k] = (unsigned short)base;
        base += count(k);
      }
      if (t == 0) cst[ncell] = (unsigned short)n;
      __syncthreads();
      images = *outside != 0;
      // ---- C: scatter into cell order; the counts are cleared for E
      for (int k = t; k < (ncell + 1) / 2; k += BS) cnt[k] = 0u;
      for (int i = t; i < n; i += BS) {
        const int g = off + i;
        const unsigned kk = (unsigned)key[g];
        const int slot = cst[kk & 0xffffu] + (int)(kk >> 16);
        float4 p = make_float4(x[g], y[g], z[g], __int_as_float(i));
        if (images) {
          p.x = into_box(p.x, R.halfL[0], R.L[0]);
          p.y = into_box(p.y, R.halfL[1], R.L[1]);
          p.z = into_box(p.z, R.halfL[2], R.L[2]);
        }
        spos[slot] = p;
      }
      __syncthreads();
      if (t == 0) *outside = 0;
      // ---- D: atom-id order inside every cell
      for (int cell = t; cell < ncell; cell += BS) {
        const int b = cst[cell], e = cst[cell + 1];
        for (int a = b + 1; a < e; ++a) {
          const float4 p = spos[a];
          const int id = __float_as_int(p.w);
          int j = a - 1;
          while (j >= b && __float_as_int(spos[j].w) > id) {
            spos[j + 1] = spos[j];
            --j;
          }
          spos[j + 1] = p;
        }
      }
    } else {
      for (int i = t; i < n; i += BS) spos[i] = make_float4(x[off + i], y[off + i], z[off + i], __int_as_float(i));
    }
    __syncthreads();
    // ---- E: forces, the closing kick, and the next step's kick-drift and cell count
    const bool acc = last && energy;
    for (int q = t; q < n * G; q += BS) {
      const int s = q / G, sub = q - s * G;
      const float4 p = spos[s];
      float ax = 0.f, ay = 0.f, az = 0.f, e = 0.f, w = 0.f;
      if (acc) atom_forces<true>(R, spos, cst, n, p, s, sub, G, ax, ay, az, e, w);
      else atom_forces<false>(R, spos, cst, n, p, s, sub, G, ax, ay, az, e, w);
      for (int o = G >> 1; o >= 1; o >>= 1) {  // n G and the stride are multiples of G: whole groups
        ax += __shfl_xor(ax, o, WAVE);
        ay += __shfl_xor(ay, o, WAVE);
        az += __shfl_xor(az, o, WAVE);
      }
      if (acc) {
        pe += 0.5 * (double)e;
        vir += 0.5 * (double)w;
      }
      if (sub != 0) continue;
      const int g = off + __float_as_int(p.w);
      float ux = vx[g], uy = vy[g], uz = vz[g];
      if (integrate) { ux = fmaf(c, ax, ux); uy = fmaf(c, ay, uy); uz = fmaf(c, az, uz); }
      if (last) {
        fx[g] = ax; fy[g] = ay; fz[g] = az;
        if (integrate) { vx[g] = ux; vy[g] = uy; vz[g] = uz; }
        if (acc) ke += 0.5 * (double)mass * ((double)ux * ux + (double)uy * uy + (double)uz * uz);
      } else if (images) {
        kick_drift(g, fmaf(c, ax, ux), fmaf(c, ay, uy), fmaf(c, az, uz), x[g], y[g], z[g]);
      } else {
        kick_drift(g, fmaf(c, ax, ux), fmaf(c, ay, uy), fmaf(c, az, uz), p.x, p.y, p.z);
      }
    }
    __syncthreads();  // spos is rewritten by the next step; its x, key and counts are complete
  }
  if (energy) {
    const double a = block_sum<BS>(pe, red);
    const double b = block_sum<BS>(ke, red);
    const double d = block_sum<BS>(vir, red);
    if (t == 0) {
      out[4 * rid + 0] = a;
      out[4 * rid + 1] = b;
      out[4 * rid + 2] = d;
      out[4 * rid + 3] = (double)n;
    }
  }
}

size_t align16(size_t b) { return (b + 15) & ~(size_t)15; }

}  // namespace

struct pdx_rep_s {
  std::vector<pdx_replica_spec> specs;
  std::vector<Rep> host;
  std::vector<int64_t> offsets;
  int nrep = 0, nmax = 0, ncmax = 0, block = 1024, stencil = 0, nallpairs = 0;
  bool block_given = false;
  int64_t total = 0;
  size_t reg0 = 0, reg1 = 0, reg2 = 0, lds = 0;
  DevBuf<Rep> reps;
  DevBuf<int32_t> order, key;
};

namespace {

// The default workgroup: the smallest that gives every lane of the largest replica's atoms a thread, as
// idle waves keep other replicas off the CU (4 096 boxes of 64 atoms, 10 steps: 256 / 512 / 1024 threads
// 0.66 / 1.2 / 2.3 ms; 16 boxes of 700 atoms: 1.10 / 0.72 / 0.50 ms; 512 of 2 048: 2.9 / 2.0 / 2.1 ms).
// With more than two replicas a CU it is the mean replica's (512 at least beside larger ones): the
// largest one then shares the time with the others.
int default_block(const std::vector<Rep> &reps) {
  int64_t sum = 0;
  int largest = 0;
  for (const Rep &R : reps) {
    const int slots = R.n * atom_lanes(R);
    largest = std::max(largest, slots);
    sum += slots;
  }
  int slots = largest;
  if (reps.size() > 512) slots = std::max((int)(sum / (int64_t)reps.size()), largest > 512 ? 512 : 0);
  return slots <= 256 ? 256 : (slots <= 512 ? 512 : 1024);
}

// Cell tables for stencil half-width S (1 or 2; 0: per replica, 2 where its finer cells fit the
// table): cells of side >= rc / S, at least 2S + 1 a
// side (else S = 1, else all pairs), at most NCMAX cells (the widest dimension is coarsened).
int layout(pdx_rep_t r, int S) {
  r->host.resize(r->nrep);
  r->nmax = 0;
  r->ncmax = 0;
  r->nallpairs = 0;
  for (int k = 0; k < r->nrep; ++k) {
    const pdx_replica_spec &sp = r->specs[k];
    Rep R{};
    R.off = (int)r->offsets[k];
    R.n = sp.n;
    R.model = sp.model;
    const double rc = sp.model == PDX_PAIR_WCA ? std::pow(2.0, 1.0 / 6.0) * sp.sigma : sp.cutoff;
    const double rc2 = sp.model == PDX_PAIR_WCA ? 1.2599211 * sp.sigma * sp.sigma : sp.cutoff * sp.cutoff;
    R.eps = (float)sp.epsilon;
    R.sig2 = (float)(sp.sigma * sp.sigma);
    R.rc2 = (float)rc2;
    if (sp.model == PDX_PAIR_LJ && sp.shift) {
      const double s6 = std::pow(sp.sigma * sp.sigma / rc2, 3);
      R.eshift = (float)(4.0 * sp.epsilon * (s6 * s6 - s6));
    }
    for (int d = 0; d < 3; ++d) {
      R.L[d] = (float)sp.box[d];
      R.halfL[d] = (float)(0.5 * sp.box[d]);
    }
    int s = S;
    if (S == 0) {
      // halved cells cut the candidates of a sphere of rc (8192 LJ atoms: 430 -> about 150 with the
      // rows cut to the sphere); where they would have to be coarsened, whole cells are walked
      // (boxes with fewer than three whole cells a side take all pairs)
      double fine = 1.0, least = sp.box[0];
      for (int d = 0; d < 3; ++d) {
        fine *= std::floor(sp.box[d] * 2 / rc);
        least = std::min(least, sp.box[d]);
      }
      s = fine <= (double)NCMAX && least >= 3.0 * rc ? 2 : 1;
    }
    int nc[3];
    for (; s >= 1; --s) {
      bool ok = true;
      for (int d = 0; d < 3; ++d) {
        nc[d] = (int)std::floor(sp.box[d] * s / rc);
        ok &= nc[d] >= 2 * s + 1;
      }
      if (!ok) continue;
      while ((int64_t)nc[0] * nc[1] * nc[2] > NCMAX) {
        int dmax = 0;
        for (int d = 1; d < 3; ++d)
          if (nc[d] > nc[dmax]) dmax = d;
        --nc[dmax];
      }
      if (nc[0] >= 2 * s + 1 && nc[1] >= 2 * s + 1 && nc[2] >= 2 * s + 1) break;
    }
    if (s < 1) {
      R.S = 0;
      ++r->nallpairs;
      R.nc[0] = R.nc[1] = R.nc[2] = 1;
    } else {
      R.S = s;
      for (int d = 0; d < 3; ++d) {
        R.nc[d] = nc[d];
        R.cinv[d] = (float)(nc[d] / sp.box[d]);
        R.cw[d] = (float)(sp.box[d] / nc[d]);
        R.slack = std::max(R.slack, (float)(2e-6 * sp.box[d]));
      }
      r->ncmax = std::max(r->ncmax, nc[0] * nc[1] * nc[2]);
    }
    r->nmax = std::max(r->nmax, R.n);
    r->host[k] = R;
  }
  if (!r->block_given) r->block = default_block(r->host);
  r->reg0 = 16 * (size_t)r->nmax;
  r->reg1 = align16(2 * ((size_t)r->ncmax + 1));
  r->reg2 = align16(2 * ((size_t)r->ncmax + 1));
  r->lds = r->reg0 + r->reg1 + r->reg2 + 128 + RED_BYTES;
  if (r->lds > 160 * 1024) return fail(PDX_ERR_ARGUMENT, "replica tables exceed the 160 KiB of LDS");
  if (hipMemcpy(r->reps.p, r->host.data(), sizeof(Rep) * r->nrep, hipMemcpyHostToDevice) != hipSuccess)
    return fail(PDX_ERR_DEVICE, "replica table upload failed");
  // largest work first: the workgroups of the longest replicas start before the short ones
  std::vector<int32_t> ord(r->nrep);
  std::iota(ord.begin(), ord.end(), 0);
  auto work = [&](int k) {
    const Rep &R = r->host[k];
    const double cand = R.S == 0 ? (double)R.n : std::pow(2 * R.S + 1, 3) * R.n /
                                                     ((double)R.nc[0] * R.nc[1] * R.nc[2]);
    return (double)R.n * cand;
  };
  std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return work(a) > work(b); });
  if (hipMemcpy(r->order.p, ord.data(), sizeof(int32_t) * r->nrep, hipMemcpyHostToDevice) != hipSuccess)
    return fail(PDX_ERR_DEVICE, "replica order upload failed");
  r->stencil = S;
  return PDX_OK;
}

template <int BS>
int launch(pdx_rep_t r, float *x, float *y, float *z, float *vx, float *vy, float *vz, float *fx, float *fy,
           float *fz, float c, float dt, float mass, int nsteps, int first, int energy, double *out,
           hipStream_t st) {
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_replicas<BS>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    (void)hipGetLastError();
    attr = true;
  }
  hipLaunchKernelGGL(k_replicas<BS>, dim3(r->nrep), dim3(BS), r->lds, st, r->reps.p, r->order.p, x, y, z, vx, vy,
                     vz, fx, fy, fz, r->key.p, c, dt, mass, nsteps, first, energy, (int)r->reg0, (int)r->reg1,
                     (int)r->reg2, out);
  PDX_LAUNCH_CHECK();
  return PDX_OK;
}

}  // namespace

extern "C" int pdx_replicas_create(int32_t nrep, const pdx_replica_spec *specs, int32_t block, int32_t stencil,
                                   pdx_rep_t *out) {
  if (!out || !specs) return fail(PDX_ERR_ARGUMENT, "null argument");
  *out = nullptr;
  if (nrep < 1) return fail(PDX_ERR_ARGUMENT, "at least one replica is required");
  if (block != 0 && block != 256 && block != 512 && block != 1024) return fail(PDX_ERR_ARGUMENT, "block must be 256, 512 or 1024");
  if (stencil != 0 && stencil != 1 && stencil != 2) return fail(PDX_ERR_ARGUMENT, "stencil must be 1 or 2");
  int64_t total = 0;
  for (int k = 0; k < nrep; ++k) {
    const pdx_replica_spec &s = specs[k];
    if (s.n < 1 || s.n > NMAX)
      return fail(PDX_ERR_ARGUMENT, "replica " + std::to_string(k) + ": atom count must be in [1, 8192]");
    if (s.model != PDX_PAIR_LJ && s.model != PDX_PAIR_WCA)
      return fail(PDX_ERR_ARGUMENT, "replica " + std::to_string(k) + ": model must be LJ or WCA");
    if (!(s.sigma > 0) || !(s.epsilon >= 0))
      return fail(PDX_ERR_ARGUMENT, "replica " + std::to_string(k) + ": sigma must be > 0, epsilon >= 0");
    const double rc = s.model == PDX_PAIR_WCA ? std::pow(2.0, 1.0 / 6.0) * s.sigma : s.cutoff;
    if (!(rc > 0)) return fail(PDX_ERR_ARGUMENT, "replica " + std::to_string(k) + ": cutoff must be > 0");
    for (int d = 0; d < 3; ++d)
      if (!(s.box[d] >= 2.0 * rc))
        return fail(PDX_ERR_ARGUMENT, "replica " + std::to_string(k) +
                                          ": box lengths must be at least twice the cutoff (minimum image)");
    total += s.n;
  }
  if (total > INT32_MAX) return fail(PDX_ERR_ARGUMENT, "too many atoms in total");
  auto *r = new pdx_rep_s();
  r->nrep = nrep;
  r->specs.assign(specs, specs + nrep);
  r->offsets.resize(nrep + 1);
  r->offsets[0] = 0;
  for (int k = 0; k < nrep; ++k) r->offsets[k + 1] = r->offsets[k] + specs[k].n;
  r->total = total;
  r->block_given = block != 0;
  if (block) r->block = block;
  int rc;
  if ((rc = r->reps.alloc(nrep)) || (rc = r->order.alloc(nrep)) || (rc = r->key.alloc(total)) ||
      (rc = layout(r, stencil))) {
    delete r;
    return rc;
  }
  *out = r;
  return PDX_OK;
}

extern "C" int pdx_replicas_destroy(pdx_rep_t r) {
  delete r;
  return PDX_OK;
}

extern "C" int pdx_replicas_set_launch(pdx_rep_t r, int32_t block, int32_t stencil) {
  if (!r) return fail(PDX_ERR_ARGUMENT, "null handle");
  if (block != 0 && block != 256 && block != 512 && block != 1024)
    return fail(PDX_ERR_ARGUMENT, "block must be 256, 512 or 1024 (0: by the replicas' sizes)");
  if (stencil != 0 && stencil != 1 && stencil != 2)
    return fail(PDX_ERR_ARGUMENT, "stencil must be 1 or 2 (0: per replica)");
  r->block_given = block != 0;
  r->block = block ? block : default_block(r->host);
  return stencil == r->stencil ? PDX_OK : layout(r, stencil);
}

extern "C" int pdx_replicas_info(pdx_rep_t r, int64_t out[8]) {
  if (!r || !out) return fail(PDX_ERR_ARGUMENT, "null argument");
  out[0] = r->total;
  out[1] = r->nrep;
  out[2] = r->nmax;
  out[3] = (int64_t)r->lds;
  out[4] = r->block;
  out[5] = r->stencil;
  out[6] = r->nallpairs;
  out[7] = r->ncmax;
  return PDX_OK;
}

extern "C" int pdx_replicas_offsets(pdx_rep_t r, int64_t *offsets) {
  if (!r || !offsets) return fail(PDX_ERR_ARGUMENT, "null argument");
  std::copy(r->offsets.begin(), r->offsets.end(), offsets);
  return PDX_OK;
}

extern "C" int pdx_replicas_run(pdx_rep_t r, float *x, float *y, float *z, float *vx, float *vy, float *vz, float *fx,
                                float *fy, float *fz, double mass, double dt, int32_t nsteps, int32_t flags,
                                double *out, pdx_stream_t stream) {
  if (!r) return fail(PDX_ERR_ARGUMENT, "null handle");
  if (!x || !y || !z || !vx || !vy || !vz || !fx || !fy || !fz) return fail(PDX_ERR_ARGUMENT, "null array");
  if (nsteps < 0) return fail(PDX_ERR_ARGUMENT, "nsteps must be >= 0");
  if (!(mass > 0) || !(dt >= 0)) return fail(PDX_ERR_ARGUMENT, "mass must be > 0 and dt >= 0");
  const bool energy = (flags & PDX_ENERGY) != 0;
  if (energy && !out) return fail(PDX_ERR_ARGUMENT, "PDX_ENERGY needs the output array");
  const int first = (flags & PDX_VV_FORCES_VALID) ? 0 : 1;
  if (nsteps == 0 && !first) return PDX_OK;
  const float c = (float)(0.5 * dt / mass);
  hipStream_t st = as_stream(stream);
  switch (r->block) {
    case 256: return launch<256>(r, x, y, z, vx, vy, vz, fx, fy, fz, c, (float)dt, (float)mass, nsteps, first, energy, out, st);
    case 512: return launch<512>(r, x, y, z, vx, vy, vz, fx, fy, fz, c, (float)dt, (float)mass, nsteps, first, energy, out, st);
    default: return launch<1024>(r, x, y, z, vx, vy, vz, fx, fy, fz, c, (float)dt, (float)mass, nsteps, first, energy, out, st);
  }
}
