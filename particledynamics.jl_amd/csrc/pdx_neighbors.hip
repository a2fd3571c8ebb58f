// Cell-list binning and slot-major ELL row construction on gfx950.
//
// Pipeline of one predicated rebuild (all kernels are enqueued every time; each returns at
// once unless the device state requests a rebuild, so the sequence can be captured in a
// hipGraph — the "predicated reference path" of src/neighbors/DeviceNeighborCUDA.jl:413-420):
//   k_decide       coverage check: per-block max |dr|^2, packing of (x, y, z, q), zeroing of
//                  the cell histogram
//   k_decide_final max over the blocks vs skin^2/4, age, adaptive interval (one block); lists of up to
//                  DECIDE_BLOCKS check blocks and SCAN_FUSED_MAX cells decide in k_bin instead
//   k_bin          cell id + histogram; the atomic's return value is the particle's slot
//   k_scan_scatter exclusive scan -> 1-based cell_offsets, particle_ids_sorted (1-based)
//                  (k_scan_local / k_scan_blocks / k_scan_finish / k_scatter above SCAN_FUSED_MAX cells)
//   k_sort_cells   ascending id inside each cell (rows and traversal become reproducible),
//                  and the cell-ordered packed positions read by the row kernel
//   k_rows_auto    (or k_rows / k_rows_cells / k_rows_allpairs) 27-cell stencil, r^2 <= rlist^2,
//                  slot-major rows t*N + i, 1-based ids; per-block max row length and statistics
//   k_commit_refs  max row length vs cap, state words; reference positions of a successful build
#include "pdx_internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>

using namespace pdx;

namespace {

constexpr int TPB = 256;
// The longest row is kept in ROW_WORDS words, one a cache line: one word is a queue of atomics from all
// row workgroups (rebuilds of 10 240 particles on 8^3 cells 58 us, with them 52), and a workgroup that
// looked first would wait for it (rows of 256 000 LJ atoms 204 us against 200).
constexpr int ROW_WORDS = 64;
constexpr int ROW_LINE = 32;                       // words of a cache line
constexpr int ROW_CHOICE = ROW_WORDS * ROW_LINE;  // word of masks_pay's choice
constexpr int DECIDE_BLOCKS = 1024;  // check blocks of a list whose k_bin decides
constexpr int SCAN_BLOCK = 1024;  // cells per block of the local scan (256 threads x 4)

__device__ __forceinline__ bool rebuild_requested(const int64_t *s) {
  return s[PDX_DN_REQUEST] != 0 && s[PDX_DN_ERROR] == 0;
}

// ------------------------------------------------------------------ decide
// Velocity-Verlet prefix of a step, fused into the check: v += c_i f, x += dt v wrapped into
// [-L/2, L/2) (_nve_kick_drift3_kernel!, src/simulation/NVEFusion.jl:3-24; the reference fuses
// it with the displacement pass the same way, src/engine/Fusion.jl:1-6). Applied only while the
// list is valid (_device_if_valid!, DeviceNeighborCUDA.jl:157-162).
struct KickDrift {
  float *vx, *vy, *vz;
  const float *fx, *fy, *fz;
  const float *inv_mass;  // per particle, or null: c for every particle
  float c, half_dt, dt;
};

// Coverage check (_device_displacement_kernel! + _device_decide_kernel!,
// DeviceNeighborCUDA.jl:169-236): per-block maximum squared displacement (plus the float4
// packing and the histogram clearing), then k_decide_final or k_bin decides. With KD the
// step's kick-drift moves x, y, z (in place) first.
template <bool KD>
__global__ __launch_bounds__(TPB) void k_decide(int N, float *__restrict__ x,
                                                 float *__restrict__ y,
                                                 float *__restrict__ z,
                                                 const float *__restrict__ q,
                                                 const float *__restrict__ rref, float4 *packed,
                                                 int32_t *cell_counts, int32_t *row_max, int ncell, int allpairs,
                                                 const float *geom, const int64_t *state,
                                                 float *partial, const int32_t *__restrict__ offsets,
                                                 const int32_t *__restrict__ ids, int32_t *snap_offsets,
                                                 int32_t *snap_ids, int64_t *snap, KickDrift kd) {
  const int64_t err = state[PDX_DN_ERROR];
  if (err != 0) return;  // latched: every block leaves (uniform)
  const int i = blockIdx.x * TPB + threadIdx.x;
  // cell snapshot: the cells of a build completed since the last snapshot, copied before this
  // step's rebuild can overwrite them (the decision records the build); a spread on another
  // stream may then read them beside the rebuild
  if (!allpairs && state[PDX_DN_BUILDS] > 0 && state[PDX_DN_BUILDS] != snap[0]) {
    for (int c = i; c <= ncell; c += gridDim.x * TPB) snap_offsets[c] = offsets[c];
    if (i < N) snap_ids[i] = ids[i];
    if (i == 0) snap[2] = 0;  // valid once this launch completes (snap[0] is written with the decision)
  }
  const float L[3] = {geom[0], geom[1], geom[2]};
  const bool valid = state[PDX_DN_VALID] != 0;
  float value = 0.0f;
  if (i < N) {
    float c[3] = {x[i], y[i], z ? z[i] : 0.0f};  // 2-D lists: no z array, every z is 0
    if (KD && valid) {
      const float ci = kd.inv_mass ? kd.half_dt * kd.inv_mass[i] : kd.c;
      float *v[3] = {kd.vx, kd.vy, kd.vz};
      const float *f[3] = {kd.fx, kd.fy, kd.fz};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        if (d == 2 && !z) break;
        const float u = fmaf(ci, f[d][i], v[d][i]);
        v[d][i] = u;
        float p = fmaf(kd.dt, u, c[d]);
        p -= (p >= 0.5f * L[d]) ? L[d] : 0.0f;
        p += (p < -0.5f * L[d]) ? L[d] : 0.0f;
        c[d] = p;
      }
      x[i] = c[0];
      y[i] = c[1];
      if (z) z[i] = c[2];
    }
    // z, then y, then x: the nested muladd order of the reference (threshold ties included)
    for (int d = 2; d >= 0; --d) {
      const float h = 0.5f * L[d];
      if (!(isfinite(c[d]) && -h <= c[d] && c[d] <= h)) {
        value = INFINITY;
      } else if (valid && value != INFINITY) {
        float dx = mic_fast(c[d] - rref[(size_t)d * N + i], h, L[d]);
        value = fmaf(dx, dx, value);
      }
    }
    packed[i] = make_float4(c[0], c[1], c[2], q ? q[i] : 0.0f);
  }
  // histogram and largest row are scratch of the next rebuild: cleared here (one launch fewer)
  if (i < ROW_WORDS) row_max[i * ROW_LINE] = 0;
  if (!allpairs)
    for (int c = i; c < ncell; c += gridDim.x * TPB) cell_counts[c] = 0;

  __shared__ float smax[TPB / WAVE];
  float m = wave_max(value);
  if ((threadIdx.x & (WAVE - 1)) == 0) smax[threadIdx.x / WAVE] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    float b = smax[0];
    for (int w = 1; w < TPB / WAVE; ++w) b = fmaxf(b, smax[w]);
    // -1: not measured (no valid list to measure against); a snapshot spread reading these
    // maxima then cannot bound the motion since the snapshot's build
    partial[blockIdx.x] = (!valid && b != INFINITY) ? -1.0f : b;
  }
}

// Largest of the check blocks' maxima (every thread of the block).
__device__ __forceinline__ float largest_displacement(int nblocks, const float *__restrict__ partial) {
  __shared__ float smax[TPB / WAVE];
  float v = 0.0f;
  for (int b = threadIdx.x; b < nblocks; b += TPB) v = fmaxf(v, partial[b]);
  v = wave_max(v);
  if ((threadIdx.x & (WAVE - 1)) == 0) smax[threadIdx.x / WAVE] = v;
  __syncthreads();
  float largest = smax[0];
  for (int w = 1; w < TPB / WAVE; ++w) largest = fmaxf(largest, smax[w]);
  return largest;
}

// What the decision makes of the state words (read only).
struct Decision {
  int64_t active;  // 0: an error is latched, nothing changes
  int64_t request, valid, error, reason, interval;
};
__device__ __forceinline__ Decision decide(float largest, const int64_t *state, float threshold, int force) {
  Decision d{state[PDX_DN_ERROR] == 0, 0, state[PDX_DN_VALID], state[PDX_DN_ERROR], 0, state[PDX_DN_INTERVAL]};
  if (!isfinite(largest)) {
    d.error = PDX_DN_COORDINATE_ERROR;
    d.valid = 0;
    return d;
  }
  if (force || d.valid == 0) {
    d.request = 1;
    d.valid = 0;
    d.reason = PDX_DN_REASON_INVALID;
    return d;
  }
  const int64_t age = state[PDX_DN_STEP] - state[PDX_DN_LAST_BUILD];
  const bool disp = largest > threshold;
  const bool old = age >= d.interval;
  if (disp || old) {
    d.request = 1;
    d.valid = 0;
    d.reason = (disp ? PDX_DN_REASON_DISPLACEMENT : 0) | (old ? PDX_DN_REASON_AGE : 0);
    // adaptive interval: x0.9 on displacement, x1.1 when the list aged out early, in [5, 100]
    if (disp) {
      float t = rintf(0.9f * (float)d.interval);
      d.interval = t < 5.0f ? 5 : (int64_t)t;
    } else if (largest < 0.1f * threshold) {
      float t = rintf(1.1f * (float)d.interval);
      d.interval = t > 100.0f ? 100 : (int64_t)t;
    }
  }
  return d;
}
__device__ __forceinline__ void write_decision(const Decision &d, int64_t *state) {
  state[PDX_DN_CHECKS] += 1;
  state[PDX_DN_REQUEST] = d.request;
  if (state[PDX_DN_DIAGNOSTICS] != 0) state[PDX_DN_REASON] = d.reason;
  state[PDX_DN_ERROR] = d.error;
  state[PDX_DN_VALID] = d.valid;
  state[PDX_DN_INTERVAL] = d.interval;
}
// The check's snapshot (k_decide copied it) is of this build.
__device__ __forceinline__ void record_snapshot(const int64_t *state, int64_t *snap) {
  if (state[PDX_DN_BUILDS] > 0 && state[PDX_DN_BUILDS] != snap[0]) snap[0] = state[PDX_DN_BUILDS];
}

// The decision from the blocks' maxima (one block).
__global__ __launch_bounds__(TPB) void k_decide_final(int nblocks, const float *__restrict__ partial, int64_t *state,
                                                       float threshold, int force, int64_t *snap, int allpairs) {
  if (state[PDX_DN_ERROR] != 0) return;
  const float largest = largest_displacement(nblocks, partial);
  if (threadIdx.x != 0) return;
  if (!allpairs) record_snapshot(state, snap);
  write_decision(decide(largest, state, threshold, force), state);
}

// ------------------------------------------------------------------ binning
// Cell id from the current box, fractional binning floor(x n/L) (_kernel_cell_ids3g!,
// DeviceNeighborCUDA.jl:464-481) + histogram (_kernel_cell_histogram!, DenseNeighborCUDA.jl:50).
// DECIDE: every block takes the decision itself from the check's partials and the state words, which
// no block of this launch writes; block 0 hands it to k_scan_scatter, which writes the words. A launch
// that finds nothing to do is 4-5 us of a step: with this and k_scan_scatter's fusion a step of 256 000 LJ
// atoms went from 98 to 96 us, an eager evaluation of 4 000 atoms from 40 to 32 us.
template <bool DECIDE>
__global__ __launch_bounds__(TPB) void k_bin(int N, const float4 *__restrict__ packed,
                                              const float *geom, int nx, int ny, int nz,
                                              int32_t *cell_of_particle, int32_t *cell_counts,
                                              int32_t *cell_rank, const int64_t *state, int nblocks,
                                              const float *__restrict__ partial, float threshold, int force,
                                              int64_t *snap, Decision *decision) {
  if (DECIDE) {
    const Decision d = decide(largest_displacement(nblocks, partial), state, threshold, force);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      *decision = d;
      if (d.active) record_snapshot(state, snap);
    }
    if (!d.active || !d.request) return;
  } else if (!rebuild_requested(state)) {
    return;
  }
  const int i = blockIdx.x * TPB + threadIdx.x;
  if (i >= N) return;
  const float4 p = packed[i];
  const float Lx = geom[0], Ly = geom[1], Lz = geom[2];
  float xx = p.x + 0.5f * Lx; xx -= floorf(xx / Lx) * Lx;
  float yy = p.y + 0.5f * Ly; yy -= floorf(yy / Ly) * Ly;
  float zz = p.z + 0.5f * Lz; zz -= floorf(zz / Lz) * Lz;
  int cx = (int)floorf(xx * ((float)nx / Lx)); cx = min(max(cx, 0), nx - 1);
  int cy = (int)floorf(yy * ((float)ny / Ly)); cy = min(max(cy, 0), ny - 1);
  int cz = (int)floorf(zz * ((float)nz / Lz)); cz = min(max(cz, 0), nz - 1);
  const int c = (cz * ny + cy) * nx + cx;
  cell_of_particle[i] = c;
  cell_rank[i] = atomicAdd(&cell_counts[c], 1);
}

// Where mask_rows is the faster build, by how the particles fill the cells now (occupied cells, largest
// cell): a workgroup per cell needs cells enough for the CUs, and no cell far above the mean one, on which
// the launch would wait. Whole rebuilds in microseconds, masks against k_rows at its default lanes:
// random particles in cell order, 1 331 cells of 14, 30, 60, 72, 80: 56 / 91 / 284 / 428 / 504 against
// 76 / 109 / 337 / 427 / 407; 8 000 cells of 14, 60, 100, 120: 133 / 1 169 / 3 545 / 5 323 against
// 137 / 1 307 / 3 682 / 5 267; a droplet of 61 440 particles in 1 000 of 4 096 cells 256 against 197, in
// 2 742 of them 103 against 121; half of 43 904 in a blob of 350 a cell 1 888 against 426. Two-dimensional
// lists have a third of the stencil: 1 600 occupied cells of 43 and 60: 140 / 243 against 137 / 211;
// 2 500: 162 / 298 against 172 / 384.
__device__ __forceinline__ bool masks_pay(int N, int ncell, bool flat, int used, int largest) {
  const long long n = N;
  if (used < (flat ? 2048 : 1024) || (long long)largest * used > 2 * n + 16ll * used) return false;
  return n <= (long long)used * (used >= 4096 || flat ? 100 : (used == ncell ? 72 : 56));
}

// Occupied cells and the largest one of a wave's lanes.
__device__ __forceinline__ int2 occupancy(int used, int largest) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) used += __shfl_xor(used, off, WAVE);
  return make_int2(used, wave_max(largest));
}

// Cell offsets (1-based, last entry N+1: _device_offsets_kernel!, DeviceNeighborCUDA.jl:280-289) and
// the particles' scatter in one launch for grids of up to SCAN_FUSED_MAX cells: every workgroup scans
// all counts in its LDS (1024 threads, a contiguous run of at most 16 cells each, wave scans of the
// run totals; the counts come from the caches) and places its share of the particles; workgroup 0
// stores the offsets and, with DECIDE, writes k_bin's decision into the state words, which the other
// workgroups do not read.
constexpr int SCAN_FUSED_MAX = 16384;  // 64 KiB of LDS
constexpr int SCAN_THREADS = 1024;
constexpr int SCAN_GRID = 64;  // 16 and 256 are 1% slower (256 000 LJ atoms), 1 is 10%
template <bool DECIDE>
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_scatter(int ncell, int N, const int32_t *__restrict__ counts,
                                                               int32_t *offsets,
                                                               const int32_t *__restrict__ cell_of_particle,
                                                               const int32_t *__restrict__ cell_rank,
                                                               int32_t *ids_sorted, int32_t *row_max, int flat,
                                                               int64_t *state,
                                                               const Decision *__restrict__ decision) {
  if (DECIDE) {
    const Decision d = *decision;
    if (!d.active) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) write_decision(d, state);
    if (!d.request) return;
  } else if (!rebuild_requested(state)) {
    return;
  }
  extern __shared__ int32_t first[];  // ncell
  __shared__ int32_t wtot[SCAN_THREADS / WAVE];
  __shared__ int2 wocc[SCAN_THREADS / WAVE];
  int used = 0, largest = 0;
  for (int c = threadIdx.x; c < ncell; c += SCAN_THREADS) first[c] = counts[c];
  __syncthreads();
  const int per = (ncell + SCAN_THREADS - 1) / SCAN_THREADS;
  const int c0 = min((int)threadIdx.x * per, ncell), c1 = min(c0 + per, ncell);
  int32_t run = 0;
  for (int c = c0; c < c1; ++c) {
    const int n = first[c];
    run += n;
    used += n != 0;
    largest = max(largest, n);
  }
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const bool choose = blockIdx.x == gridDim.x - 1;  // (workgroup 0 stores the offsets)
  if (choose) {
    const int2 o = occupancy(used, largest);
    if (lane == 0) wocc[w] = o;
  }
  int32_t v = run;
#pragma unroll
  for (int o = 1; o < WAVE; o <<= 1) {
    const int32_t u = __shfl_up(v, o, WAVE);
    if (lane >= o) v += u;
  }
  if (lane == WAVE - 1) wtot[w] = v;
  __syncthreads();
  int32_t base = v - run + 1;
  for (int k = 0; k < w; ++k) base += wtot[k];
  for (int c = c0; c < c1; ++c) {
    const int32_t n = first[c];
    first[c] = base;
    base += n;
  }
  __syncthreads();
  if (blockIdx.x == 0) {
    for (int c = threadIdx.x; c < ncell; c += SCAN_THREADS) offsets[c] = first[c];
    if (threadIdx.x == 0) offsets[ncell] = N + 1;
  }
  if (choose && w == 0) {
    const int2 o = lane < SCAN_THREADS / WAVE ? wocc[lane] : make_int2(0, 0), all = occupancy(o.x, o.y);
    if (lane == 0) row_max[ROW_CHOICE] = masks_pay(N, ncell, flat != 0, all.x, all.y);
  }
  for (int i = blockIdx.x * SCAN_THREADS + threadIdx.x; i < N; i += gridDim.x * SCAN_THREADS)
    ids_sorted[first[cell_of_particle[i]] - 1 + cell_rank[i]] = i + 1;
}

// The largest grids pass the 64 KiB a launch may take unasked.
void allow_scan_lds() {
  static std::once_flag once;
  std::call_once(once, [] {
    const int most = sizeof(int32_t) * SCAN_FUSED_MAX;
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_scan_scatter<false>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, most);
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_scan_scatter<true>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, most);
    (void)hipGetLastError();
  });
}

// Exclusive scan of cell_counts, SCAN_BLOCK cells per block (block-local part).
__global__ __launch_bounds__(TPB) void k_scan_local(int ncell, const int32_t *counts,
                                                     int32_t *offsets, int32_t *block_totals,
                                                     int2 *block_occ, const int64_t *state) {
  if (!rebuild_requested(state)) return;
  __shared__ int32_t sh[TPB];
  __shared__ int2 wocc[TPB / WAVE];
  int used = 0, largest = 0;
  const int base = blockIdx.x * SCAN_BLOCK + threadIdx.x * 4;
  int32_t v[4];
  int32_t run = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[k] = (base + k < ncell) ? counts[base + k] : 0;
    run += v[k];
    used += v[k] != 0;
    largest = max(largest, v[k]);
  }
  const int2 o = occupancy(used, largest);
  if ((threadIdx.x & (WAVE - 1)) == 0) wocc[threadIdx.x / WAVE] = o;
  sh[threadIdx.x] = run;
  __syncthreads();
  for (int off = 1; off < TPB; off <<= 1) {
    int32_t a = threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
    __syncthreads();
    sh[threadIdx.x] += a;
    __syncthreads();
  }
  int32_t excl = sh[threadIdx.x] - run;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (base + k < ncell) offsets[base + k] = excl;
    excl += v[k];
  }
  if (threadIdx.x == TPB - 1) {
    block_totals[blockIdx.x] = sh[TPB - 1];
    int2 t = wocc[0];
    for (int k = 1; k < TPB / WAVE; ++k) t = make_int2(t.x + wocc[k].x, max(t.y, wocc[k].y));
    block_occ[blockIdx.x] = t;
  }
}

// Exclusive scan of the block totals (one block, sequential over chunks of 1024), and the grid's occupancy.
__global__ __launch_bounds__(1024) void k_scan_blocks(int nblocks, int32_t *block_totals,
                                                       const int2 *__restrict__ block_occ, int32_t *row_max,
                                                       int N, int ncell, int flat,
                                                       const int64_t *state) {
  if (!rebuild_requested(state)) return;
  __shared__ int32_t sh[1024];
  __shared__ int2 wocc[1024 / WAVE];
  int used = 0, largest = 0;
  for (int k = threadIdx.x; k < nblocks; k += 1024) {
    used += block_occ[k].x;
    largest = max(largest, block_occ[k].y);
  }
  const int2 o = occupancy(used, largest);
  if ((threadIdx.x & (WAVE - 1)) == 0) wocc[threadIdx.x / WAVE] = o;
  __syncthreads();
  if (threadIdx.x < WAVE) {
    const int2 t = threadIdx.x < 1024 / WAVE ? wocc[threadIdx.x] : make_int2(0, 0), all = occupancy(t.x, t.y);
    if (threadIdx.x == 0) row_max[ROW_CHOICE] = masks_pay(N, ncell, flat != 0, all.x, all.y);
  }
  int32_t carry = 0;
  for (int base = 0; base < nblocks; base += 1024) {
    const int k = base + threadIdx.x;
    const int32_t v = k < nblocks ? block_totals[k] : 0;
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      int32_t a = threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
      __syncthreads();
      sh[threadIdx.x] += a;
      __syncthreads();
    }
    if (k < nblocks) block_totals[k] = carry + sh[threadIdx.x] - v;
    const int32_t tot = sh[1023];
    __syncthreads();
    carry += tot;
  }
}

// 1-based offsets with last entry N+1 (_device_offsets_kernel!, DeviceNeighborCUDA.jl:280-289).
__global__ __launch_bounds__(TPB) void k_scan_finish(int ncell, int N, int32_t *offsets,
                                                      const int32_t *block_totals,
                                                      const int64_t *state) {
  if (!rebuild_requested(state)) return;
  const int c = blockIdx.x * TPB + threadIdx.x;
  if (c < ncell) offsets[c] += block_totals[c / SCAN_BLOCK] + 1;
  if (c == ncell) offsets[ncell] = N + 1;
}

__global__ __launch_bounds__(TPB) void k_scatter(int N, const int32_t *__restrict__ cell_of_particle,
                                                  const int32_t *__restrict__ cell_rank,
                                                  const int32_t *__restrict__ offsets, int32_t *ids_sorted,
                                                  const int64_t *state) {
  if (!rebuild_requested(state)) return;
  const int i = blockIdx.x * TPB + threadIdx.x;
  if (i >= N) return;
  const int c = cell_of_particle[i];
  ids_sorted[offsets[c] - 1 + cell_rank[i]] = i + 1;
}

// Stable order inside each cell (ascending id) and the cell-ordered packed copy (x, y, z, id)
// the row kernel streams through. One wave per cell: the cell's ids are staged in LDS and each
// lands at its rank (ids are distinct); cells beyond the LDS stage are sorted by one lane.
constexpr int SORT_STAGE = 2048;
__global__ __launch_bounds__(WAVE) void k_sort_cells(int ncell, const int32_t *offsets, int32_t *ids_sorted,
                                                     const float4 *__restrict__ packed, float4 *sorted,
                                                     const int64_t *state) {
  if (!rebuild_requested(state)) return;
  __shared__ int32_t sh[SORT_STAGE];
  // grid-stride over the cells (a bounded grid: on a check without rebuild the launch is cheap
  // however many cells there are)
  for (int c = blockIdx.x; c < ncell; c += gridDim.x) {
    const int s = offsets[c] - 1, e = offsets[c + 1] - 1, n = e - s;
    __syncthreads();  // the previous cell's ranks are read
    if (n <= SORT_STAGE) {
      for (int k = threadIdx.x; k < n; k += WAVE) sh[k] = ids_sorted[s + k];
      __syncthreads();
      for (int k = threadIdx.x; k < n; k += WAVE) {
        const int32_t key = sh[k];
        int rank = 0;
        for (int m = 0; m < n; ++m) rank += sh[m] < key;
        ids_sorted[s + rank] = key;
        const float4 p = packed[key - 1];
        sorted[s + rank] = make_float4(p.x, p.y, p.z, __int_as_float(key - 1));
      }
      continue;
    }
    if (threadIdx.x == 0) {
      for (int a = s + 1; a < e; ++a) {
        const int32_t key = ids_sorted[a];
        int b = a - 1;
        while (b >= s && ids_sorted[b] > key) {
          ids_sorted[b + 1] = ids_sorted[b];
          --b;
        }
        ids_sorted[b + 1] = key;
      }
    }
    __syncthreads();
    for (int k = s + threadIdx.x; k < e; k += WAVE) {
      const int i = ids_sorted[k] - 1;
      const float4 p = packed[i];
      sorted[k] = make_float4(p.x, p.y, p.z, __int_as_float(i));
    }
  }
}

// ------------------------------------------------------------------ rows
// Commit data of a block's rows (_device_capacity_partial_kernel!, DeviceNeighborCUDA.jl:291-310): the
// largest row into a word of its group, candidates and accepted entries per block; called by every thread.
__device__ __forceinline__ void row_partials(int longest, long long tested, long long accepted, int32_t *row_max,
                                             int64_t *stat_partial) {
  __shared__ int smax[TPB / WAVE];
  __shared__ long long ssum[2][TPB / WAVE];
  longest = wave_max(longest);
  for (int off = 32; off >= 1; off >>= 1) {
    tested += __shfl_xor(tested, off, WAVE);
    accepted += __shfl_xor(accepted, off, WAVE);
  }
  const int w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  if ((threadIdx.x & (WAVE - 1)) == 0) { smax[w] = longest; ssum[0][w] = tested; ssum[1][w] = accepted; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < nw; ++k) { longest = max(longest, smax[k]); tested += ssum[0][k]; accepted += ssum[1][k]; }
    atomicMax(&row_max[(blockIdx.x % ROW_WORDS) * ROW_LINE], longest);
    stat_partial[2 * blockIdx.x] = tested;
    stat_partial[2 * blockIdx.x + 1] = accepted;
  }
}

// G lanes per particle, particles in cell order (the groups of a wave share their home cell,
// so candidate loads are broadcast). The group walks the 27-cell stencil G candidates at a
// time; accepted neighbours are placed with a wave64 ballot + popcount in candidate order, so
// every row is identical whatever G is. Distance test as the reference: mic_fast differences,
// r^2 = muladd(dx,dx,muladd(dy,dy,dz^2)) <= rl^2 (_kernel_neighbors3!, DenseNeighborCUDA.jl:153-206;
// cooperative placement as _cooperative_rows3_kernel!, src/engine/Builder.jl:39-129). Slots are
// written slot-major at t*N + i with 1-based ids; the count keeps growing past cap so the
// commit can report the required capacity.
// STAGE (opt-in): the workgroup's rows are kept in LDS as [slot][particle] (TPB/G particles, cap
// slots, at most 64 KiB) and written out slot by slot after the search, so a row slot of
// consecutive particles is one contiguous store; written straight from the search, the slots of
// a wave's particles advance at different rates and the 4-byte stores land in partially filled
// lines (measured: 8.6x the row bytes at 486 400 ions, 2.0x staged). Same rows either way.
constexpr size_t ROW_STAGE_BYTES = 65536;
// The rows of the vb-th TPB / G particles; longest, all_tested and all_found take this thread's rows.
template <int G, bool STAGE>
__device__ __forceinline__ void search_rows(int vb, int N, int cap, int nx, int ny, int nz,
                                            const float4 *__restrict__ sorted, const int32_t *__restrict__ offsets,
                                            const int32_t *__restrict__ cell_of_particle, const float *geom, float rl2,
                                            int32_t *nbr, int32_t *counts, int64_t *candidates, int &longest,
                                            long long &all_tested, long long &all_found) {
  constexpr int PB = TPB / G;  // particles per workgroup
  extern __shared__ int32_t srow[];  // STAGE: [cap][PB]
  const int t = vb * PB + threadIdx.x / G;
  const int lg = threadIdx.x % G;
  const int pb = threadIdx.x / G;
  const int wl = threadIdx.x & (WAVE - 1);
  const unsigned long long gmask = (G == WAVE) ? ~0ull : (((1ull << G) - 1ull) << (wl - lg));
  const unsigned long long below = (1ull << wl) - 1ull;
  const bool active = t < N;  // whole groups are active or not (G divides the block)
  const float Lx = geom[0], Ly = geom[1], Lz = geom[2];
  const float hx = 0.5f * Lx, hy = 0.5f * Ly, hz = 0.5f * Lz;
  int found = 0, i = -1;
  int64_t tested = 0;
  if (active) {
    const float4 pi = sorted[t];
    i = __float_as_int(pi.w);
    const int c0 = cell_of_particle[i];
    const int cx = c0 % nx, cy = (c0 / nx) % ny, cz = c0 / (nx * ny);
    for (int oz = -1; oz <= 1; ++oz) {
      int cz2 = cz + oz; cz2 -= (cz2 >= nz) ? nz : 0; cz2 += (cz2 < 0) ? nz : 0;
      for (int oy = -1; oy <= 1; ++oy) {
        int cy2 = cy + oy; cy2 -= (cy2 >= ny) ? ny : 0; cy2 += (cy2 < 0) ? ny : 0;
        for (int ox = -1; ox <= 1; ++ox) {
          int cx2 = cx + ox; cx2 -= (cx2 >= nx) ? nx : 0; cx2 += (cx2 < 0) ? nx : 0;
          const int c = (cz2 * ny + cy2) * nx + cx2;
          const int s = offsets[c] - 1, e = offsets[c + 1] - 1;
          for (int k0 = s; k0 < e; k0 += G) {
            const int k = k0 + lg;
            bool acc = false, cand = false;
            int j = 0;
            if (k < e) {
              const float4 pj = sorted[k];
              j = __float_as_int(pj.w);
              cand = j != i;
              const float dx = mic_fast(pj.x - pi.x, hx, Lx);
              const float dy = mic_fast(pj.y - pi.y, hy, Ly);
              const float dz = mic_fast(pj.z - pi.z, hz, Lz);
              const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
              acc = cand && (r2 <= rl2);
            }
            if (G == 1) {
              tested += cand;
              if (acc) {
                if (found < cap) {
                  if (STAGE) srow[found * PB + pb] = j + 1;
                  else nbr[(size_t)found * N + i] = j + 1;
                }
                ++found;
              }
            } else {
              const unsigned long long am = __ballot(acc) & gmask;
              tested += __popcll(__ballot(cand) & gmask);
              if (acc) {
                const int slot = found + __popcll(am & below);
                if (slot < cap) {
                  if (STAGE) srow[slot * PB + pb] = j + 1;
                  else nbr[(size_t)slot * N + i] = j + 1;
                }
              }
              found += __popcll(am);
            }
          }
        }
      }
    }
  }
  if (STAGE) {
    __shared__ int sfound[PB], sid[PB];
    __shared__ int smax;
    if (lg == 0) {
      sfound[pb] = active ? min(found, cap) : 0;
      sid[pb] = i;
    }
    if (threadIdx.x == 0) smax = 0;
    __syncthreads();
    if (lg == 0 && active) atomicMax(&smax, min(found, cap));
    __syncthreads();
    const int ns = smax;
    for (int e = threadIdx.x; e < ns * PB; e += TPB) {
      const int sl = e / PB, q = e - sl * PB;
      if (sl < sfound[q]) nbr[(size_t)sl * N + sid[q]] = srow[sl * PB + q];
    }
  }
  if (active && lg == 0) {
    counts[i] = found;
    if (candidates) candidates[i] = tested;
    longest = max(longest, found);
    all_tested += tested;
    all_found += found;
  }
}

template <int G, bool STAGE>
__global__ __launch_bounds__(TPB) void k_rows(int N, int cap, int nx, int ny, int nz,
                                               const float4 *__restrict__ sorted,
                                               const int32_t *__restrict__ offsets,
                                               const int32_t *__restrict__ cell_of_particle,
                                               const float *geom, float rl2, int32_t *nbr,
                                               int32_t *counts, int64_t *candidates, int32_t *row_max,
                                               int64_t *stat_partial, const int64_t *state) {
  if (!rebuild_requested(state)) return;  // uniform over the grid
  int longest = 0;
  long long all_tested = 0, all_found = 0;
  search_rows<G, STAGE>(blockIdx.x, N, cap, nx, ny, nz, sorted, offsets, cell_of_particle, geom, rl2, nbr, counts,
                        candidates, longest, all_tested, all_found);
  row_partials(longest, all_tested, all_found, row_max, stat_partial);
}

// Rows from LDS-staged candidates: one workgroup per cell. Wave 0 lists the cell's 27 stencil cells
// in k_rows' order (z, y, x offsets -1..1, each cell's particles in sorted order) with the
// inclusive scan of their sizes; the flattened candidate list is staged into LDS RC_CHUNK float4s
// at a time, and the cell's particles, G lanes each (TPB/G per pass), test them from LDS. The
// ballot + popcount placement over the flattened order writes exactly k_rows' rows (the
// accepted candidates in stencil order), whatever G or the chunking.
constexpr int RC_CHUNK = 2048;
template <int G>
__global__ __launch_bounds__(TPB) void k_rows_cells(int N, int cap, int ncell, int nx, int ny, int nz,
                                                    const float4 *__restrict__ sorted,
                                                    const int32_t *__restrict__ offsets, const float *geom,
                                                    float rl2, int32_t *nbr, int32_t *counts,
                                                    int64_t *candidates, int32_t *row_max,
                                                    int64_t *stat_partial, const int64_t *state) {
  constexpr int PB = TPB / G;  // particles per pass
  __shared__ float4 cand[RC_CHUNK];
  __shared__ int cstart[27], cpre[28];
  if (!rebuild_requested(state)) return;  // uniform over the grid
  int longest = 0;
  long long all_tested = 0, all_found = 0;
  for (int c = blockIdx.x; c < ncell; c += gridDim.x) {  // grid-stride over the cells
    const int p0 = offsets[c] - 1, np = offsets[c + 1] - offsets[c];
    if (np <= 0) continue;  // uniform over the workgroup
    const int cx = c % nx, cy = (c / nx) % ny, cz = c / (nx * ny);
    __syncthreads();  // the previous cell's stencil and candidates are no longer read
    if (threadIdx.x < WAVE) {
      int cnt = 0;
      if (threadIdx.x < 27) {
        const int o = threadIdx.x;
        int cz2 = cz + o / 9 - 1; cz2 -= (cz2 >= nz) ? nz : 0; cz2 += (cz2 < 0) ? nz : 0;
        int cy2 = cy + (o / 3) % 3 - 1; cy2 -= (cy2 >= ny) ? ny : 0; cy2 += (cy2 < 0) ? ny : 0;
        int cx2 = cx + o % 3 - 1; cx2 -= (cx2 >= nx) ? nx : 0; cx2 += (cx2 < 0) ? nx : 0;
        const int cc = (cz2 * ny + cy2) * nx + cx2;
        cstart[o] = offsets[cc] - 1;
        cnt = offsets[cc + 1] - offsets[cc];
      }
#pragma unroll
      for (int d = 1; d < WAVE; d <<= 1) {
        const int u = __shfl_up(cnt, d, WAVE);
        if ((int)threadIdx.x >= d) cnt += u;
      }
      if (threadIdx.x < 27) cpre[threadIdx.x + 1] = cnt;
      if (threadIdx.x == 0) cpre[0] = 0;
    }
    __syncthreads();
    const int total = cpre[27];
    const float Lx = geom[0], Ly = geom[1], Lz = geom[2];
    const float hx = 0.5f * Lx, hy = 0.5f * Ly, hz = 0.5f * Lz;
    const int lg = threadIdx.x % G, pl = threadIdx.x / G;
    const int wl = threadIdx.x & (WAVE - 1);
    const unsigned long long gmask = (G == WAVE) ? ~0ull : (((1ull << G) - 1ull) << (wl - lg));
    const unsigned long long below = (1ull << wl) - 1ull;
    for (int pb = 0; pb < np; pb += PB) {
      const bool active = pb + pl < np;
      float4 pi = make_float4(0.f, 0.f, 0.f, 0.f);
      int i = -1;
      if (active) {
        pi = sorted[p0 + pb + pl];
        i = __float_as_int(pi.w);
      }
      int found = 0;
      int64_t tested = 0;
      for (int ch = 0; ch < total; ch += RC_CHUNK) {
        const int nch = min(RC_CHUNK, total - ch);
        __syncthreads();  // the previous chunk (or pass) is no longer read
        for (int f = threadIdx.x; f < nch; f += TPB) {
          const int g = ch + f;
          int cc = 0;
#pragma unroll
          for (int h = 16; h >= 1; h >>= 1)
            if (cc + h < 27 && cpre[cc + h] <= g) cc += h;
          cand[f] = sorted[cstart[cc] + (g - cpre[cc])];
        }
        __syncthreads();
        if (active) {
          for (int k0 = 0; k0 < nch; k0 += G) {
            const int k = k0 + lg;
            bool acc = false, cnd = false;
            int j = 0;
            if (k < nch) {
              const float4 pj = cand[k];
              j = __float_as_int(pj.w);
              cnd = j != i;
              const float dx = mic_fast(pj.x - pi.x, hx, Lx);
              const float dy = mic_fast(pj.y - pi.y, hy, Ly);
              const float dz = mic_fast(pj.z - pi.z, hz, Lz);
              const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
              acc = cnd && (r2 <= rl2);
            }
            if (G == 1) {
              tested += cnd;
              if (acc) {
                if (found < cap) nbr[(size_t)found * N + i] = j + 1;
                ++found;
              }
            } else {
              const unsigned long long am = __ballot(acc) & gmask;
              tested += __popcll(__ballot(cnd) & gmask);
              if (acc) {
                const int slot = found + __popcll(am & below);
                if (slot < cap) nbr[(size_t)slot * N + i] = j + 1;
              }
              found += __popcll(am);
            }
          }
        }
      }
      if (active && lg == 0) {
        counts[i] = found;
        if (candidates) candidates[i] = tested;
        longest = max(longest, found);
        all_tested += tested;
        all_found += found;
      }
    }
  }
  row_partials(longest, all_tested, all_found, row_max, stat_partial);
}

// ---- the build of many evenly filled cells: one workgroup per cell, lanes = candidates, particles one
// after the other in scalar registers (four waves, a chunk of 64 candidates each in turn). A distance test
// of 64 candidates is then seven vector instructions (three more per dimension where the stencil crosses
// the seam), its ballot goes into lane p of a register pair (particle p of the cell), and the cell's tests
// end as bit masks in LDS. The rows are written in a second pass with lanes = particles, each wave a quarter
// of the masks from the slot its earlier ones add up to: every lane takes its next set bit, so a store
// writes neighbouring slots of the cell's rows, lines that fill up within a few steps where the
// cell's particles are contiguous in storage (spatial order). Candidates are numbered in stencil
// order (z, y, x cells, then the cells' order), so rows are k_rows' rows.
// Bound by vector issue in both passes (about 9 instructions per 64 tests and 12 per step of the row
// writes). k_rows spends 38 on 64 tests (per-lane image, ballots, predicated 4-byte stores that each
// touch their own line). Whole rebuilds with it at its best lane count and with this kernel: 326 and
// 264 us (256 000 LJ atoms, 21 a cell), 1 224 and 1 020 us (486 400 ions, 61 a cell).
// v_writelane_b32: old with lane `lane` = value, both uniform. This compiler has the intrinsic but no
// builtin for it; a compiler without it refuses the name.
extern "C" __device__ __attribute__((const)) int pdx_writelane(int value, int lane,
                                                               int old) __asm("llvm.amdgcn.writelane.i32");
constexpr int RM_CHUNKS = 28;  // candidate chunks of 64 per pass (21 KiB of LDS: seven workgroups per CU)
constexpr int RM_WAVES = TPB / WAVE;
__device__ __forceinline__ void mask_rows(int N, int cap, int ncell, int nx, int ny, int nz,
                                          const float4 *__restrict__ sorted, const int32_t *__restrict__ offsets,
                                          const float *__restrict__ geom, float rl2, int32_t *__restrict__ nbr,
                                          int32_t *__restrict__ counts, int64_t *candidates, int &longest,
                                          long long &all_tested, long long &all_found) {
  __shared__ uint2 mask[RM_CHUNKS][WAVE];
  __shared__ int32_t cid[RM_CHUNKS * WAVE];
  __shared__ int cstart[27], cpre[28], ends[WAVE];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE);
  const float Lx = geom[0], Ly = geom[1], Lz = geom[2];
  const float hx = 0.5f * Lx, hy = 0.5f * Ly, hz = 0.5f * Lz;
  for (int c = blockIdx.x; c < ncell; c += gridDim.x) {
    const int p0 = offsets[c] - 1, np = offsets[c + 1] - 1 - p0;  // uniform
    if (np <= 0) continue;
    const int cx = c % nx, cy = (c / nx) % ny, cz = c / (nx * ny);
    __syncthreads();  // the previous cell's LDS is no longer read
    if (wv == 0) {
      int cnt = 0;
      if (lane < 27) {
        int cz2 = cz + lane / 9 - 1; cz2 -= (cz2 >= nz) ? nz : 0; cz2 += (cz2 < 0) ? nz : 0;
        int cy2 = cy + (lane / 3) % 3 - 1; cy2 -= (cy2 >= ny) ? ny : 0; cy2 += (cy2 < 0) ? ny : 0;
        int cx2 = cx + lane % 3 - 1; cx2 -= (cx2 >= nx) ? nx : 0; cx2 += (cx2 < 0) ? nx : 0;
        const int cc = (cz2 * ny + cy2) * nx + cx2;
        cstart[lane] = offsets[cc] - 1;
        cnt = offsets[cc + 1] - offsets[cc];
      }
#pragma unroll
      for (int d = 1; d < WAVE; d <<= 1) {
        const int u = __shfl_up(cnt, d, WAVE);
        if (lane >= d) cnt += u;
      }
      if (lane < 27) cpre[lane + 1] = cnt;
      if (lane == 0) cpre[0] = 0;
    }
    __syncthreads();
    const int total = __builtin_amdgcn_readfirstlane(cpre[27]);
    const int self0 = __builtin_amdgcn_readfirstlane(cpre[13]);  // the home cell's first candidate
    // no cell of the stencil lies across the seam, and two cells apart is less than half the box
    const bool plain = cx > 0 && cx < nx - 1 && cy > 0 && cy < ny - 1 && cz > 0 && cz < nz - 1 && nx > 4 && ny > 4 &&
                       nz > 4;
    for (int pg = 0; pg < np; pg += WAVE) {
      const int ng = min(WAVE, np - pg);
      const float4 *home = sorted + p0 + pg;
      const int i = lane < ng ? __float_as_int(home[lane].w) : 0;
      int found = 0;
      for (int ch0 = 0; ch0 < total; ch0 += RM_CHUNKS * WAVE) {
        const int nch = min(RM_CHUNKS, (total - ch0 + WAVE - 1) / WAVE);
        for (int cc = wv; cc < nch; cc += RM_WAVES) {
          const int g = ch0 + cc * WAVE + lane;
          int sc = 0;
#pragma unroll
          for (int h = 16; h >= 1; h >>= 1)
            if (sc + h < 27 && cpre[sc + h] <= g) sc += h;
          // lanes past the last candidate sit too far from everything to be accepted
          float4 q = make_float4(1e30f, 0.f, 0.f, 0.f);
          if (g < total) q = sorted[cstart[sc] + (g - cpre[sc])];
          cid[cc * WAVE + lane] = __float_as_int(q.w) + 1;
          int mlo = 0, mhi = 0;
          auto test = [&](int p, const float4 &pi, auto image) {
            float dx = q.x - pi.x, dy = q.y - pi.y, dz = q.z - pi.z;
            image(dx, dy, dz);
            const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            const unsigned long long m = __ballot(r2 <= rl2);
            mlo = pdx_writelane((int)(unsigned)m, p, mlo);
            mhi = pdx_writelane((int)(unsigned)(m >> 32), p, mhi);
          };
          // four particles' scalar loads in flight (lanes past ng - 1 of the masks are not read)
          auto tests = [&](auto image) {
            for (int p = 0; p < ng; p += 4) {
              float4 pi[4];
#pragma unroll
              for (int u = 0; u < 4; ++u) pi[u] = home[min(p + u, ng - 1)];
#pragma unroll
              for (int u = 0; u < 4; ++u) test(p + u, pi[u], image);
            }
          };
          // k_bin puts a particle at the very face +L/2 into cell 0: next to it, in cell 1, its
          // distance still needs the image
          const bool face = g < total && ((cx == 1 && q.x > 0.5f * hx) || (cy == 1 && q.y > 0.5f * hy) ||
                                          (cz == 1 && q.z > 0.5f * hz));
          if (plain && __ballot(face) == 0) {
            tests([](float &, float &, float &) {});
          } else {
            tests([&](float &dx, float &dy, float &dz) {
              dx = mic_fast(dx, hx, Lx);
              dy = mic_fast(dy, hy, Ly);
              dz = mic_fast(dz, hz, Lz);
            });
          }
          // the particle itself is among the home cell's candidates
          const int b = self0 + pg + lane - ch0 - cc * WAVE;
          if (b >= 0 && b < 32) mlo &= (int)~(1u << b);
          if (b >= 32 && b < WAVE) mhi &= (int)~(1u << (b - 32));
          mask[cc][lane] = make_uint2((unsigned)mlo, (unsigned)mhi);
        }
        __syncthreads();
        auto word = [&](int k) {
          const uint2 m = mask[k][lane];
          return lane < ng ? ((unsigned long long)m.y << 32) | m.x : 0ull;
        };
        const int w0 = nch * wv / RM_WAVES, w1 = nch * (wv + 1) / RM_WAVES;
        for (int k = 0; k < w0; ++k) found += (int)__popcll(word(k));
        int w = w0;
        unsigned long long m = w0 < w1 ? word(w0) : 0ull, nextm = w0 + 1 < w1 ? word(w0 + 1) : 0ull;
        int32_t *out = nbr + (size_t)found * N + i;
        while (__ballot(m != 0ull || w < w1 - 1) != 0) {
          if (m == 0ull && w < w1 - 1) {
            ++w;
            m = nextm;
            nextm = w + 1 < w1 ? word(w + 1) : 0ull;
          }
          if (m != 0ull) {
            const int b = __ffsll((long long)m) - 1;
            m &= m - 1ull;
            const int j = cid[w * WAVE + b];
            if (found < cap) *out = j;
            out += N;
            ++found;
          }
        }
        if (wv == RM_WAVES - 1) ends[lane] = found;
        __syncthreads();
        found = ends[lane];
      }
      if (wv == 0 && lane < ng) {
        counts[i] = found;
        if (candidates) candidates[i] = total - 1;
        longest = max(longest, found);
        all_tested += total - 1;
        all_found += found;
      }
    }
  }
}

template <int G>  // seven waves a SIMD: what the masks' LDS allows
__global__ __launch_bounds__(TPB, 7) void k_rows_auto(int N, int cap, int ncell, int nx, int ny, int nz,
                                                   const float4 *__restrict__ sorted,
                                                   const int32_t *__restrict__ offsets,
                                                   const int32_t *__restrict__ cell_of_particle,
                                                   const float *__restrict__ geom, float rl2,
                                                   int32_t *__restrict__ nbr, int32_t *__restrict__ counts,
                                                   int64_t *candidates, int32_t *row_max, int64_t *stat_partial,
                                                   const int64_t *state) {
  const bool masks = row_max[ROW_CHOICE] != 0;  // (read beside the request)
  if (!rebuild_requested(state)) return;  // uniform over the grid
  int longest = 0;
  long long all_tested = 0, all_found = 0;
  if (__builtin_expect(masks, 1)) {
    mask_rows(N, cap, ncell, nx, ny, nz, sorted, offsets, geom, rl2, nbr, counts, candidates, longest, all_tested,
              all_found);
  } else {
    for (int vb = blockIdx.x; (long long)vb * (TPB / G) < N; vb += gridDim.x)
      search_rows<G, false>(vb, N, cap, nx, ny, nz, sorted, offsets, cell_of_particle, geom, rl2, nbr, counts,
                            candidates, longest, all_tested, all_found);
  }
  row_partials(longest, all_tested, all_found, row_max, stat_partial);
}

// All-pairs rows for small boxes, one image (_kernel_neighbors_allpairs!, DenseNeighborCUDA.jl:128-151).
__global__ __launch_bounds__(TPB) void k_rows_allpairs(int N, int cap,
                                                        const float4 *__restrict__ packed,
                                                        const float *geom, float rl2,
                                                        int32_t *nbr, int32_t *counts,
                                                        int64_t *candidates, int32_t *row_max,
                                                        int64_t *stat_partial, const int64_t *state) {
  if (!rebuild_requested(state)) return;
  const int i = blockIdx.x * TPB + threadIdx.x;
  const bool active = i < N;
  int found = 0;
  if (active) {
    const float Lx = geom[0], Ly = geom[1], Lz = geom[2];
    const float4 pi = packed[i];
    for (int j = 0; j < N; ++j) {
      if (j == i) continue;
      const float4 pj = packed[j];
      // dimension order of the reference's loop: r2 = muladd(dd, dd, r2) for d = 1..D
      float r2 = 0.0f;
      float dd = mic_fast(pj.x - pi.x, 0.5f * Lx, Lx); r2 = fmaf(dd, dd, r2);
      dd = mic_fast(pj.y - pi.y, 0.5f * Ly, Ly); r2 = fmaf(dd, dd, r2);
      dd = mic_fast(pj.z - pi.z, 0.5f * Lz, Lz); r2 = fmaf(dd, dd, r2);
      if (r2 <= rl2) {
        if (found < cap) nbr[(size_t)found * N + i] = j + 1;
        ++found;
      }
    }
    counts[i] = found;
    if (candidates) candidates[i] = N - 1;
  }
  row_partials(found, active ? N - 1 : 0, found, row_max, stat_partial);
}

// ------------------------------------------------------------------ commit
// Capacity commit (_device_commit_kernel!, DeviceNeighborCUDA.jl:291-388) and, when every row fitted,
// the reference positions of the build. Every block reads the largest row; block 0 also adds the
// statistics and writes the state words (the others need only the request and an error word that no
// successful commit changes).
__global__ __launch_bounds__(TPB) void k_commit_refs(int N, int nblocks, int cap, const int32_t *__restrict__ row_max,
                                                     const int64_t *__restrict__ stat_partial,
                                                     const float4 *__restrict__ packed, float *rref, int64_t *state) {
  if (!rebuild_requested(state)) return;
  static_assert(ROW_WORDS == WAVE, "one word a lane");
  const int largest = wave_max(row_max[(threadIdx.x & (WAVE - 1)) * ROW_LINE]);
  const int i = blockIdx.x * TPB + threadIdx.x;
  if (largest <= cap && i < N) {
    const float4 p = packed[i];
    rref[i] = p.x;
    rref[(size_t)N + i] = p.y;
    rref[(size_t)2 * N + i] = p.z;
  }
  if (blockIdx.x != 0) return;
  __shared__ long long ssum[2][TPB / WAVE];
  long long ctot = 0, atot = 0;
  for (int b = threadIdx.x; b < nblocks; b += TPB) {
    ctot += stat_partial[2 * b];
    atot += stat_partial[2 * b + 1];
  }
  for (int off = 32; off >= 1; off >>= 1) {
    ctot += __shfl_xor(ctot, off, WAVE);
    atot += __shfl_xor(atot, off, WAVE);
  }
  const int w = threadIdx.x / WAVE;
  if ((threadIdx.x & (WAVE - 1)) == 0) { ssum[0][w] = ctot; ssum[1][w] = atot; }
  __syncthreads();
  for (int k = 1; k < TPB / WAVE; ++k) { ctot += ssum[0][k]; atot += ssum[1][k]; }
  if (threadIdx.x != 0) return;
  state[PDX_DN_REQUIRED] = largest;
  const bool diag = state[PDX_DN_DIAGNOSTICS] != 0;
  if (diag) {
    state[PDX_DN_ATTEMPTS] += 1;
    state[PDX_DN_LAST_CANDIDATES] = ctot;
    state[PDX_DN_TOTAL_CANDIDATES] += ctot;
    state[PDX_DN_LAST_ACCEPTED] = atot;
    state[PDX_DN_TOTAL_ACCEPTED] += atot;
    if (largest > state[PDX_DN_MAX_ROW]) state[PDX_DN_MAX_ROW] = largest;
  }
  if (largest > cap) {
    state[PDX_DN_ERROR] = PDX_DN_CAPACITY_ERROR;
    state[PDX_DN_VALID] = 0;
    return;
  }
  state[PDX_DN_VALID] = 1;
  state[PDX_DN_LAST_BUILD] = state[PDX_DN_STEP];
  state[PDX_DN_BUILDS] += 1;
  if (diag) {
    const int64_t reason = state[PDX_DN_REASON];
    if (reason & PDX_DN_REASON_INVALID) state[PDX_DN_INVALID_BUILDS] += 1;
    else if (reason & PDX_DN_REASON_DISPLACEMENT) state[PDX_DN_DISPLACEMENT_BUILDS] += 1;
    else state[PDX_DN_AGE_BUILDS] += 1;
    if ((reason & (PDX_DN_REASON_DISPLACEMENT | PDX_DN_REASON_AGE)) ==
        (PDX_DN_REASON_DISPLACEMENT | PDX_DN_REASON_AGE))
      state[PDX_DN_OVERLAP_BUILDS] += 1;
  }
}


__global__ void k_advance(int64_t *state) {
  if (state[PDX_DN_VALID] != 0 && state[PDX_DN_ERROR] == 0) state[PDX_DN_STEP] += 1;
}

// Closing kick of a velocity-Verlet step, v += c_i f (_nve_kick3_kernel!, SimulationCore.jl:
// 581-591), while the list is valid; the first thread also advances the step counter (the
// reference folds advance_device_neighbor_step! into the kick, Run.jl:281-285).
__global__ __launch_bounds__(TPB) void k_kick(int N, KickDrift kd, int dim, int64_t *state) {
  if (!(state[PDX_DN_VALID] != 0 && state[PDX_DN_ERROR] == 0)) return;
  const int i = blockIdx.x * TPB + threadIdx.x;
  if (i < N) {
    const float ci = kd.inv_mass ? kd.half_dt * kd.inv_mass[i] : kd.c;
    kd.vx[i] = fmaf(ci, kd.fx[i], kd.vx[i]);
    kd.vy[i] = fmaf(ci, kd.fy[i], kd.vy[i]);
    if (dim == 3) kd.vz[i] = fmaf(ci, kd.fz[i], kd.vz[i]);
  }
  if (i == 0) state[PDX_DN_STEP] += 1;
}

__global__ void k_rearm(int64_t *state) {
  state[PDX_DN_ERROR] = 0;
  state[PDX_DN_REQUEST] = 1;
}

__global__ void k_invalidate(int64_t *state) { state[PDX_DN_VALID] = 0; }

// Spatial order of the last build (the permutation of OrderingWorkspace, src/engine/Ordering.jl:
// 19-79): slots in cell order (cells z, y, x), inside a cell by position (x, then y, then z, then
// the id for coincident particles), so the order depends on the configuration and not on the
// particles' labels. One wave per cell ranks its particles (cells hold a few dozen); perm[slot] =
// 0-based particle id. Cells beyond the LDS stage rank from global memory.
__global__ __launch_bounds__(WAVE) void k_spatial_order(int ncell, const int32_t *__restrict__ offsets,
                                                        const int32_t *__restrict__ ids,
                                                        const float4 *__restrict__ packed, int32_t *perm) {
  __shared__ float4 sh[SORT_STAGE / 2];
  const int c = blockIdx.x;
  const int s = offsets[c] - 1, e = offsets[c + 1] - 1, n = e - s;
  auto key = [&](int k) {
    const int i = ids[s + k] - 1;
    const float4 p = packed[i];
    return make_float4(p.x, p.y, p.z, __int_as_float(i));
  };
  const bool staged = n <= SORT_STAGE / 2;
  if (staged) {
    for (int k = threadIdx.x; k < n; k += WAVE) sh[k] = key(k);
    __syncthreads();
  }
  auto before = [](const float4 a, const float4 b) {
    if (a.x != b.x) return a.x < b.x;
    if (a.y != b.y) return a.y < b.y;
    if (a.z != b.z) return a.z < b.z;
    return __float_as_int(a.w) < __float_as_int(b.w);
  };
  for (int k = threadIdx.x; k < n; k += WAVE) {
    const float4 me = staged ? sh[k] : key(k);
    int rank = 0;
    for (int m = 0; m < n; ++m) rank += before(staged ? sh[m] : key(m), me);
    perm[s + rank] = __float_as_int(me.w);
  }
}

// Cell snapshot: offsets and ids of a build that completed since the last snapshot (the build
// counter moved), then the recorded count. Run after every step's evaluation, so that a spread
// running beside the next step's rebuild reads cells no rebuild is writing.
__global__ __launch_bounds__(TPB) void k_snap_copy(int N, int ncell, const int32_t *__restrict__ offsets,
                                                   const int32_t *__restrict__ ids, int32_t *so, int32_t *sid,
                                                   const int64_t *state, const int64_t *snap) {
  if (state[PDX_DN_ERROR] != 0 || state[PDX_DN_BUILDS] == snap[0]) return;
  const int k = blockIdx.x * TPB + threadIdx.x;
  if (k <= ncell) so[k] = offsets[k];
  if (k < N) sid[k] = ids[k];
}
__global__ void k_snap_mark(const int64_t *state, int64_t *snap) {
  if (state[PDX_DN_ERROR] != 0 || state[PDX_DN_BUILDS] == snap[0]) return;
  snap[0] = state[PDX_DN_BUILDS];
  snap[2] = 0;
}

inline int blocks_for(int64_t n, int tpb) { return (int)((n + tpb - 1) / tpb); }

int grid_for_box(const double box[3], double rl, int32_t out[3]) {
  for (int d = 0; d < 3; ++d) {
    if (!(std::isfinite(box[d]) && box[d] > 0))
      return fail(PDX_ERR_ARGUMENT, "Neighbor box lengths must be finite and positive.");
    // floor(L / cell) in the list precision, as _choose_grid (NeighborTypes.jl:52-63)
    const float n = std::floor((float)box[d] / (float)rl);
    out[d] = n < 1 ? 1 : (int32_t)n;
  }
  return PDX_OK;
}

// The decision from the check's partial maxima (and the snapshot's record), then the predicated
// rebuild.
int enqueue_decide_build(pdx_nl_t nl, hipStream_t st) {
  const int N = nl->N;
  const int nb = blocks_for(N, TPB);
  int64_t *s = nl->state.p;
  const float *geom = nl->geom.p;
  const float skin = (float)nl->skin;
  const float threshold = (0.25f * skin) * skin;
  int row_blocks = nb;  // workgroups of the row kernel, one commit partial each
  // k_bin decides where its workgroups reread at most 1 024 partials each (4 KB, from the caches) and
  // k_scan_scatter follows to write the decision down; else a launch of its own does. Forty steps in
  // k_bin and apart: LJ atoms 6 912 1.15 and 1.22 ms, 62 500 1.79 and 1.87, 256 000 (1 000 blocks) 3.68 and
  // 3.74, 500 000 6.13 both; ions beside a mesh 27 000 4.64 and 4.66, 64 000 5.14 and 5.17, 262 144 (1 024
  // blocks) 22.23 and 22.14, 486 400 23.2 and 22.9. Single evaluations beside a mesh: 7 600 ions 78 and
  // 82 us, 64 000 124 and 125.5. (With the scan apart too, 64 000 ions take 123 us, but 5.24 ms for forty
  // steps: the chain's launches then end after the spread instead of beside it.)
  const bool scan_fused = !nl->allpairs && nl->ncell <= SCAN_FUSED_MAX;
  const bool decide_fused = scan_fused && nb <= DECIDE_BLOCKS;
  Decision *dec = (Decision *)nl->decision.p;
  if (!decide_fused)
    hipLaunchKernelGGL(k_decide_final, dim3(1), dim3(TPB), 0, st, nb, nl->disp_partial.p, s, threshold,
                       nl->check_force, nl->snap_state.p, (int)nl->allpairs);
  if (!nl->allpairs) {
    const int sblocks = blocks_for(nl->ncell, SCAN_BLOCK);
    const int flat = nl->dim == 2;
    auto bin = decide_fused ? k_bin<true> : k_bin<false>;
    hipLaunchKernelGGL(bin, dim3(nb), dim3(TPB), 0, st, N, nl->packed.p, geom, nl->nx, nl->ny, nl->nz,
                       nl->cell_of_particle.p, nl->cell_counts.p, nl->cell_rank.p, s, nb, nl->disp_partial.p,
                       threshold, nl->check_force, nl->snap_state.p, dec);
    if (scan_fused) {
      auto scan = decide_fused ? k_scan_scatter<true> : k_scan_scatter<false>;
      hipLaunchKernelGGL(scan, dim3(std::min(blocks_for(N, SCAN_THREADS), SCAN_GRID)), dim3(SCAN_THREADS),
                         sizeof(int32_t) * (size_t)nl->ncell, st, nl->ncell, N, nl->cell_counts.p, nl->cell_offsets.p,
                         nl->cell_of_particle.p, nl->cell_rank.p, nl->particle_ids_sorted.p, nl->row_max.p, flat,
                         s, dec);
    } else {
      hipLaunchKernelGGL(k_scan_local, dim3(sblocks), dim3(TPB), 0, st, nl->ncell, nl->cell_counts.p,
                         nl->cell_offsets.p, nl->scan_block.p, nl->scan_occ.p, s);
      hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(1024), 0, st, sblocks, nl->scan_block.p,
                         nl->scan_occ.p, nl->row_max.p, N, nl->ncell, flat, s);
      hipLaunchKernelGGL(k_scan_finish, dim3(blocks_for(nl->ncell + 1, TPB)), dim3(TPB), 0, st, nl->ncell, N,
                         nl->cell_offsets.p, nl->scan_block.p, s);
      hipLaunchKernelGGL(k_scatter, dim3(nb), dim3(TPB), 0, st, N, nl->cell_of_particle.p, nl->cell_rank.p,
                         nl->cell_offsets.p, nl->particle_ids_sorted.p, s);
    }
    hipLaunchKernelGGL(k_sort_cells, dim3(std::min(nl->ncell, 8192)), dim3(WAVE), 0, st, nl->ncell, nl->cell_offsets.p,
                       nl->particle_ids_sorted.p, nl->packed.p, nl->sorted.p, s);
    // Lists of 14 to 100 particles a cell on at least 1 024 cells choose between the mask build and
    // k_rows on the device (masks_pay); k_rows also takes a caller's lane count and the opt-in forms below.
    // Lanes per particle of k_rows: the list's row lanes; with PDX_ROW_STAGE=1 the rows are staged in LDS and
    // the lanes raised until the workgroup's rows fit the 64 KiB stage. Staging cuts the build's HBM
    // writes at 486 400 ions from 3.97 GB to 0.93 GB but not its time (1.13 ms at 32 lanes against
    // 1.12 ms written straight at 8), so the default writes straight from the search.
    int G = nl->row_lanes;
    bool stage = false;
    if (const char *v = std::getenv("PDX_ROW_STAGE")) stage = std::atoi(v) != 0;
    // the cell-staged build (k_rows_cells, PDX_ROW_CELLS=1): at 486 400 ions (8 000 cells, one
    // workgroup each) 1.06-1.09 ms against 1.12 ms for k_rows in spatial storage order, 1.33 against
    // 1.55 ms in lattice order; a whole rebuild with mask_rows takes 1.02 ms, with k_rows 1.22
    bool cells = false;
    if (const char *v = std::getenv("PDX_ROW_CELLS")) cells = std::atoi(v) != 0;
    if (stage) cells = false;
    if (!stage && !cells && !nl->row_lanes_given && nl->ncell >= 1024 && N >= 14 * (int64_t)nl->ncell &&
        N <= 100 * (int64_t)nl->ncell) {
      row_blocks = std::min(nl->ncell, 4096);
#define PDX_ROWA(GG)                                                                                            \
  hipLaunchKernelGGL((k_rows_auto<GG>), dim3(row_blocks), dim3(TPB), 0, st, N, nl->cap, nl->ncell, nl->nx,      \
                     nl->ny, nl->nz, nl->sorted.p, nl->cell_offsets.p, nl->cell_of_particle.p, geom, nl->rl2,   \
                     nl->neighbors_flat.p, nl->counts.p, nl->diagnostics ? nl->candidates.p : nullptr,          \
                     nl->row_max.p, nl->stat_partial.p, s);
      switch (G) {
        case 1: PDX_ROWA(1) break;
        case 2: PDX_ROWA(2) break;
        case 4: PDX_ROWA(4) break;
        case 8: PDX_ROWA(8) break;
        case 16: PDX_ROWA(16) break;
        default: PDX_ROWA(32) break;
      }
#undef PDX_ROWA
    } else if (cells) {
      row_blocks = std::min(nl->ncell, 8192);
#define PDX_ROWC(GG)                                                                                        \
  hipLaunchKernelGGL((k_rows_cells<GG>), dim3(row_blocks), dim3(TPB), 0, st, N, nl->cap, nl->ncell, \
                     nl->nx, nl->ny, nl->nz, \
                     nl->sorted.p, nl->cell_offsets.p, geom, nl->rl2, nl->neighbors_flat.p, nl->counts.p,     \
                     nl->diagnostics ? nl->candidates.p : nullptr, nl->row_max.p, nl->stat_partial.p, s);
      switch (G) {
        case 1: PDX_ROWC(1) break;
        case 2: PDX_ROWC(2) break;
        case 4: PDX_ROWC(4) break;
        case 8: PDX_ROWC(8) break;
        case 16: PDX_ROWC(16) break;
        default: PDX_ROWC(32) break;
      }
#undef PDX_ROWC
    } else {
    if (stage) {
      int g = G;
      while (g < 32 && (size_t)(TPB / g) * nl->cap * sizeof(int32_t) > ROW_STAGE_BYTES) g <<= 1;
      if ((size_t)(TPB / g) * nl->cap * sizeof(int32_t) <= ROW_STAGE_BYTES) G = g;
      else stage = false;
    }
    const int rb = (int)(((int64_t)N * G + TPB - 1) / TPB);
    row_blocks = rb;
    const size_t lds = stage ? (size_t)(TPB / G) * nl->cap * sizeof(int32_t) : 0;
#define PDX_ROWS(GG)                                                                                       \
  if (stage)                                                                                               \
    hipLaunchKernelGGL((k_rows<GG, true>), dim3(rb), dim3(TPB), lds, st, N, nl->cap, nl->nx, nl->ny, nl->nz, \
                       nl->sorted.p, nl->cell_offsets.p, nl->cell_of_particle.p, geom, nl->rl2,            \
                       nl->neighbors_flat.p, nl->counts.p, nl->diagnostics ? nl->candidates.p : nullptr,   \
                       nl->row_max.p, nl->stat_partial.p, s);                                          \
  else                                                                                                     \
    hipLaunchKernelGGL((k_rows<GG, false>), dim3(rb), dim3(TPB), 0, st, N, nl->cap, nl->nx, nl->ny, nl->nz, \
                       nl->sorted.p, nl->cell_offsets.p, nl->cell_of_particle.p, geom, nl->rl2,            \
                       nl->neighbors_flat.p, nl->counts.p, nl->diagnostics ? nl->candidates.p : nullptr,   \
                       nl->row_max.p, nl->stat_partial.p, s);
    switch (G) {
      case 1: PDX_ROWS(1) break;
      case 2: PDX_ROWS(2) break;
      case 4: PDX_ROWS(4) break;
      case 8: PDX_ROWS(8) break;
      case 16: PDX_ROWS(16) break;
      default: PDX_ROWS(32) break;
    }
#undef PDX_ROWS
    }
  } else {
    hipLaunchKernelGGL(k_rows_allpairs, dim3(nb), dim3(TPB), 0, st, N, nl->cap, nl->packed.p, geom,
                       nl->rl2, nl->neighbors_flat.p, nl->counts.p,
                       nl->diagnostics ? nl->candidates.p : nullptr, nl->row_max.p, nl->stat_partial.p, s);
  }
  hipLaunchKernelGGL(k_commit_refs, dim3(nb), dim3(TPB), 0, st, N, row_blocks, nl->cap, nl->row_max.p,
                     nl->stat_partial.p, nl->packed.p, nl->rref.p, s);
  PDX_LAUNCH_CHECK();
  return PDX_OK;
}

int enqueue_check(pdx_nl_t nl, const float *x, const float *y, const float *z, const float *q, hipStream_t st,
                  int force, const KickDrift *kd = nullptr) {
  if (!nl) return fail(PDX_ERR_ARGUMENT, "null neighbor list");
  if (!x || !y || (!z && nl->dim == 3)) return fail(PDX_ERR_ARGUMENT, "null coordinate array");
  const int N = nl->N;
  const int nb = blocks_for(N, TPB);
  nl->packed_src[0] = x; nl->packed_src[1] = y; nl->packed_src[2] = z; nl->packed_src[3] = q;
  float *xw = const_cast<float *>(x), *yw = const_cast<float *>(y), *zw = const_cast<float *>(z);
  if (kd)
    hipLaunchKernelGGL(k_decide<true>, dim3(nb), dim3(TPB), 0, st, N, xw, yw, zw, q, nl->rref.p, nl->packed.p,
                       nl->cell_counts.p, nl->row_max.p, nl->ncell, (int)nl->allpairs, nl->geom.p, nl->state.p,
                       nl->disp_partial.p,
                       (const int32_t *)nl->cell_offsets.p, (const int32_t *)nl->particle_ids_sorted.p,
                       nl->snap_offsets.p, nl->snap_ids.p, nl->snap_state.p, *kd);
  else
    hipLaunchKernelGGL(k_decide<false>, dim3(nb), dim3(TPB), 0, st, N, xw, yw, zw, q, nl->rref.p, nl->packed.p,
                       nl->cell_counts.p, nl->row_max.p, nl->ncell, (int)nl->allpairs, nl->geom.p, nl->state.p,
                       nl->disp_partial.p,
                       (const int32_t *)nl->cell_offsets.p, (const int32_t *)nl->particle_ids_sorted.p,
                       nl->snap_offsets.p, nl->snap_ids.p, nl->snap_state.p, KickDrift{});
  PDX_LAUNCH_CHECK();
  // the first check after creation / a box change builds; the second one snapshots that build
  if (nl->snap_host < 2) nl->snap_host += 1;
  nl->check_force = force;
  return PDX_OK;
}

int enqueue_update(pdx_nl_t nl, const float *x, const float *y, const float *z, const float *q,
                   hipStream_t st, int force) {
  int rc = enqueue_check(nl, x, y, z, q, st, force);
  if (rc) return rc;
  return enqueue_decide_build(nl, st);
}

}  // namespace

extern "C" int pdx_nl_create(int32_t n, const double box[3], double cutoff, double skin, int32_t cap,
                             int32_t interval, int32_t flags, pdx_nl_t *out) {
  if (!out || !box) return fail(PDX_ERR_ARGUMENT, "null argument");
  *out = nullptr;
  if (!(n > 0 && n < INT32_MAX)) return fail(PDX_ERR_ARGUMENT, "Neighbor builders require 0 < N < typemax(Int32).");
  if (cap <= 0) return fail(PDX_ERR_ARGUMENT, "Neighbor capacity must be positive.");
  if (!(std::isfinite(cutoff) && cutoff >= 0)) return fail(PDX_ERR_ARGUMENT, "Neighbor cutoff must be finite and nonnegative.");
  if (!(std::isfinite(skin) && skin >= 0)) return fail(PDX_ERR_ARGUMENT, "Neighbor skin must be finite and nonnegative.");
  if (interval < 1 || interval > 100) return fail(PDX_ERR_ARGUMENT, "Rebuild interval must be between 1 and 100");
  if ((int64_t)n * cap > INT32_MAX)
    return fail(PDX_ERR_ARGUMENT, "Neighbor table of N particles x cap exceeds the Int32 index range; lower `cap`.");
  auto *nl = new pdx_nl_s();
  nl->N = n;
  nl->cap = cap;
  nl->interval = interval;
  nl->cutoff = cutoff;
  nl->skin = skin;
  nl->allpairs = (flags & PDX_NL_ALLPAIRS) != 0;
  nl->diagnostics = (flags & PDX_NL_DIAGNOSTICS) != 0;
  nl->dim = (flags & PDX_NL_2D) ? 2 : 3;
  for (int d = 0; d < 3; ++d) nl->box[d] = box[d];
  const float rlf = std::max(1e-6f, (float)cutoff + (float)skin);
  nl->rl2 = rlf * rlf;
  // 2-D (DenseNeighborCUDA.jl:77, D = 2): every z is 0 and the list's z extent is three list
  // radii, so the z layers of the stencil beside the particles' own are empty and no pair has a
  // z image: the 3-D kernels then build the 2-D rows, which equal the 9-cell 2-D stencil's
  double box3[3] = {box[0], box[1], box[2]};
  if (nl->dim == 2) {
    box3[2] = 3.0 * (double)rlf * (1.0 + 1e-6);
    nl->box[2] = box3[2];
  }
  int32_t g[3];
  int rc = grid_for_box(box3, rlf, g);
  if (rc) { delete nl; return rc; }
  if (nl->allpairs) {
    const double mn = std::min(box3[0], std::min(box3[1], box3[2]));
    if (!(2.0 * rlf <= mn)) {
      delete nl;
      return fail(PDX_ERR_ARGUMENT, "All-pairs neighbor rows need cutoff+skin <= L/2 (minimum image).");
    }
    g[0] = g[1] = g[2] = 1;
  } else if (g[0] < 3 || g[1] < 3 || g[2] < 3) {
    delete nl;
    return fail(PDX_ERR_ARGUMENT,
                "Dense cell-list neighbor builder requires at least 3 cells per periodic dimension to avoid "
                "duplicate neighbor-cell visits. Increase the box size, reduce cutoff+skin, or use all-pairs rows.");
  }
  nl->nx = g[0]; nl->ny = g[1]; nl->nz = g[2];
  nl->ncell = g[0] * g[1] * g[2];
  // lanes per particle of the row build: enough to fill ~2^19 resident threads (256 CUs x 2048),
  // and at least one lane per ~256 candidates (27 cells of the mean occupancy): measured at 486 400
  // ions (1 700 candidates per particle), 8 lanes build in 1.12 ms against 1.65 ms for 2; at most
  // 32; PDX_ROW_LANES overrides (tuning)
  {
    int G = 1;
    while ((int64_t)n * G < 524288 && G < 32) G <<= 1;
    const double cand = 27.0 * (double)n / (double)std::max(1, nl->ncell);
    while (G < 32 && cand > 256.0 * G) G <<= 1;
    if (const char *v = std::getenv("PDX_ROW_LANES")) {
      const int e = std::atoi(v);
      if (e == 1 || e == 2 || e == 4 || e == 8 || e == 16 || e == 32) {
        G = e;
        nl->row_lanes_given = true;
      }
    }
    nl->row_lanes = nl->row_lanes_auto = G;
    nl->row_lanes_env = nl->row_lanes_given;
  }
  allow_scan_lds();
  const int nb = blocks_for(n, TPB);
  nl->ndisp = nb;
  const int cb = std::max(blocks_for((int64_t)n * 32, TPB), 8192);  // the row kernels' largest grids
  const int sblocks = blocks_for(nl->ncell, SCAN_BLOCK);
  if ((rc = nl->state.alloc(PDX_DN_NSTATE)) || (rc = nl->geom.alloc(3)) ||
      (rc = nl->neighbors_flat.alloc((size_t)n * cap)) || (rc = nl->counts.alloc(n)) ||
      (rc = nl->cell_offsets.alloc(nl->ncell + 1)) || (rc = nl->cell_counts.alloc(nl->ncell)) ||
      (rc = nl->particle_ids_sorted.alloc(n)) || (rc = nl->cell_of_particle.alloc(n)) ||
      (rc = nl->cell_rank.alloc(n)) || (rc = nl->rref.alloc((size_t)3 * n)) || (rc = nl->packed.alloc(n)) ||
      (rc = nl->sorted.alloc(n)) || (rc = nl->sortedq.alloc(n)) || (rc = nl->disp_partial.alloc(nb)) ||
      (rc = nl->row_max.alloc(ROW_CHOICE + 1)) ||
      (rc = nl->decision.alloc(sizeof(Decision) / sizeof(int64_t))) ||
      (rc = nl->stat_partial.alloc((size_t)2 * cb)) || (rc = nl->scan_block.alloc(sblocks)) ||
      (rc = nl->scan_occ.alloc(sblocks)) ||
      (rc = nl->candidates.alloc(nl->diagnostics ? n : 1)) ||
      (rc = nl->snap_offsets.alloc((size_t)nl->ncell + 1)) || (rc = nl->snap_ids.alloc(n)) ||
      (rc = nl->snap_state.alloc(4))) {
    delete nl;
    return rc;
  }
  int64_t st[PDX_DN_NSTATE] = {0};
  st[PDX_DN_INTERVAL] = interval;
  st[PDX_DN_DIAGNOSTICS] = nl->diagnostics ? 1 : 0;
  const float geomf[3] = {(float)box3[0], (float)box3[1], (float)box3[2]};
  std::vector<int32_t> ones(nl->ncell + 1, 1);
  // identity traversal order until the first build (mesh kernels may read it before then)
  std::vector<int32_t> ident(n);
  for (int32_t k = 0; k < n; ++k) ident[k] = k + 1;
  hipError_t e = hipSuccess;
  if (e == hipSuccess) e = hipMemcpy(nl->state.p, st, sizeof(st), hipMemcpyHostToDevice);
  const int64_t snap0[4] = {-1, 0, 1, 0};
  if (e == hipSuccess) e = hipMemcpy(nl->snap_state.p, snap0, sizeof(snap0), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(nl->geom.p, geomf, sizeof(geomf), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(nl->neighbors_flat.p, 0xff, sizeof(int32_t) * (size_t)n * cap);  // -1 padding
  if (e == hipSuccess) e = hipMemset(nl->counts.p, 0, sizeof(int32_t) * n);
  if (e == hipSuccess) e = hipMemset(nl->cell_counts.p, 0, sizeof(int32_t) * nl->ncell);
  if (e == hipSuccess) e = hipMemcpy(nl->cell_offsets.p, ones.data(), sizeof(int32_t) * (nl->ncell + 1), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(nl->particle_ids_sorted.p, ident.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(nl->cell_of_particle.p, 0, sizeof(int32_t) * n);
  if (e == hipSuccess) e = hipMemset(nl->packed.p, 0, sizeof(float4) * n);
  if (e == hipSuccess) e = hipMemset(nl->rref.p, 0, sizeof(float) * 3 * (size_t)n);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    delete nl;
    return fail(PDX_ERR_DEVICE, std::string("neighbor list initialisation failed: ") + hipGetErrorString(e));
  }
  *out = nl;
  return PDX_OK;
}

extern "C" int pdx_nl_destroy(pdx_nl_t nl) {
  delete nl;
  return PDX_OK;
}

extern "C" int pdx_nl_info(pdx_nl_t nl, int32_t out[8]) {
  if (!nl || !out) return fail(PDX_ERR_ARGUMENT, "null argument");
  out[0] = nl->N; out[1] = nl->cap; out[2] = nl->nx; out[3] = nl->ny; out[4] = nl->nz;
  out[5] = nl->ncell; out[6] = nl->allpairs; out[7] = nl->diagnostics;
  return PDX_OK;
}

extern "C" int pdx_nl_arrays_get(pdx_nl_t nl, pdx_nl_arrays *out) {
  if (!nl || !out) return fail(PDX_ERR_ARGUMENT, "null argument");
  out->neighbors_flat = nl->neighbors_flat.p;
  out->counts = nl->counts.p;
  out->cell_offsets = nl->cell_offsets.p;
  out->particle_ids_sorted = nl->particle_ids_sorted.p;
  out->cell_of_particle = nl->cell_of_particle.p;
  out->rref_x = nl->rref.p;
  out->rref_y = nl->rref.p + nl->N;
  out->rref_z = nl->rref.p + 2 * (size_t)nl->N;
  out->packed = reinterpret_cast<float *>(nl->packed.p);
  out->state = nl->state.p;
  return PDX_OK;
}

extern "C" int pdx_nl_update(pdx_nl_t nl, const float *x, const float *y, const float *z, const float *q,
                             pdx_stream_t stream) {
  return enqueue_update(nl, x, y, z, q, as_stream(stream), 0);
}

extern "C" int pdx_nl_rebuild(pdx_nl_t nl, const float *x, const float *y, const float *z, const float *q,
                              pdx_stream_t stream) {
  return enqueue_update(nl, x, y, z, q, as_stream(stream), 1);
}

extern "C" int pdx_nl_check(pdx_nl_t nl, const float *x, const float *y, const float *z, const float *q,
                            pdx_stream_t stream) {
  return enqueue_check(nl, x, y, z, q, as_stream(stream), 0);
}

namespace {
int make_kick_drift(pdx_nl_t nl, float *vx, float *vy, float *vz, const float *fx, const float *fy,
                    const float *fz, double dt, double mass, const float *inv_mass, KickDrift &kd) {
  if (!nl) return fail(PDX_ERR_ARGUMENT, "null neighbor list");
  if (!vx || !vy || !fx || !fy || (nl->dim == 3 && (!vz || !fz)))
    return fail(PDX_ERR_ARGUMENT, "null velocity or force array");
  if (!(std::isfinite(dt) && dt > 0)) return fail(PDX_ERR_ARGUMENT, "dt must be finite and positive");
  if (!inv_mass && !(std::isfinite(mass) && mass > 0))
    return fail(PDX_ERR_ARGUMENT, "Inertial integrators require mass > 0");
  kd.vx = vx; kd.vy = vy; kd.vz = vz;
  kd.fx = fx; kd.fy = fy; kd.fz = fz;
  kd.inv_mass = inv_mass;
  kd.dt = (float)dt;
  kd.half_dt = (float)(0.5 * dt);
  kd.c = inv_mass ? 0.0f : (float)dt / 2.0f / (float)mass;  // (dt / 2) / m in FP32, as Run.jl:249
  return PDX_OK;
}
}  // namespace

extern "C" int pdx_nl_check_kick_drift(pdx_nl_t nl, float *x, float *y, float *z, const float *q, float *vx,
                                       float *vy, float *vz, const float *fx, const float *fy, const float *fz,
                                       double dt, double mass, const float *inv_mass, pdx_stream_t stream) {
  KickDrift kd{};
  int rc = make_kick_drift(nl, vx, vy, vz, fx, fy, fz, dt, mass, inv_mass, kd);
  if (rc) return rc;
  return enqueue_check(nl, x, y, z, q, as_stream(stream), 0, &kd);
}

extern "C" int pdx_nve_kick(pdx_nl_t nl, float *vx, float *vy, float *vz, const float *fx, const float *fy,
                            const float *fz, double dt, double mass, const float *inv_mass, pdx_stream_t stream) {
  KickDrift kd{};
  int rc = make_kick_drift(nl, vx, vy, vz, fx, fy, fz, dt, mass, inv_mass, kd);
  if (rc) return rc;
  hipLaunchKernelGGL(k_kick, dim3(blocks_for(nl->N, TPB)), dim3(TPB), 0, as_stream(stream), nl->N, kd, nl->dim,
                     nl->state.p);
  PDX_LAUNCH_CHECK();
  return PDX_OK;
}

extern "C" int pdx_nl_spatial_order(pdx_nl_t nl, int32_t *perm, pdx_stream_t stream) {
  if (!nl || !perm) return fail(PDX_ERR_ARGUMENT, "null argument");
  if (nl->allpairs) return fail(PDX_ERR_ARGUMENT, "all-pairs lists have no cells to order by");
  int64_t st[PDX_DN_NSTATE];
  hipStream_t s = as_stream(stream);
  PDX_HIP(hipStreamSynchronize(s));
  PDX_HIP(hipMemcpy(st, nl->state.p, sizeof(st), hipMemcpyDeviceToHost));
  if (st[PDX_DN_ERROR] != 0 || st[PDX_DN_VALID] == 0)
    return fail(PDX_ERR_STATE, "spatial order needs a valid list (update it first)");
  hipLaunchKernelGGL(k_spatial_order, dim3(nl->ncell), dim3(WAVE), 0, s, nl->ncell,
                     (const int32_t *)nl->cell_offsets.p, (const int32_t *)nl->particle_ids_sorted.p,
                     (const float4 *)nl->packed.p, perm);
  PDX_LAUNCH_CHECK();
  return PDX_OK;
}

extern "C" int pdx_nl_invalidate(pdx_nl_t nl, pdx_stream_t stream) {
  if (!nl) return fail(PDX_ERR_ARGUMENT, "null neighbor list");
  hipStream_t s = as_stream(stream);
  PDX_HIP(hipStreamSynchronize(s));
  const int64_t snap0[4] = {-1, 0, 1, 0};
  PDX_HIP(hipMemcpy(nl->snap_state.p, snap0, sizeof(snap0), hipMemcpyHostToDevice));
  nl->snap_host = 0;
  hipLaunchKernelGGL(k_invalidate, dim3(1), dim3(1), 0, s, nl->state.p);
  PDX_LAUNCH_CHECK();
  PDX_HIP(hipStreamSynchronize(s));
  return PDX_OK;
}

extern "C" int pdx_nl_build(pdx_nl_t nl, pdx_stream_t stream) {
  if (!nl) return fail(PDX_ERR_ARGUMENT, "null neighbor list");
  return enqueue_decide_build(nl, as_stream(stream));
}

extern "C" int pdx_nl_snapshot(pdx_nl_t nl, pdx_stream_t stream) {
  if (!nl) return fail(PDX_ERR_ARGUMENT, "null neighbor list");
  if (nl->allpairs) return fail(PDX_ERR_ARGUMENT, "all-pairs lists have no cells to snapshot");
  hipStream_t st = as_stream(stream);
  const int n = std::max(nl->N, nl->ncell + 1);
  hipLaunchKernelGGL(k_snap_copy, dim3(blocks_for(n, TPB)), dim3(TPB), 0, st, nl->N, nl->ncell,
                     (const int32_t *)nl->cell_offsets.p, (const int32_t *)nl->particle_ids_sorted.p,
                     nl->snap_offsets.p, nl->snap_ids.p, (const int64_t *)nl->state.p,
                     (const int64_t *)nl->snap_state.p);
  hipLaunchKernelGGL(k_snap_mark, dim3(1), dim3(1), 0, st, (const int64_t *)nl->state.p, nl->snap_state.p);
  PDX_LAUNCH_CHECK();
  if (nl->snap_host >= 1) nl->snap_host = 2;
  return PDX_OK;
}

extern "C" int pdx_nl_advance(pdx_nl_t nl, pdx_stream_t stream) {
  if (!nl) return fail(PDX_ERR_ARGUMENT, "null neighbor list");
  hipLaunchKernelGGL(k_advance, dim3(1), dim3(1), 0, as_stream(stream), nl->state.p);
  PDX_LAUNCH_CHECK();
  return PDX_OK;
}

extern "C" int pdx_nl_rearm(pdx_nl_t nl, pdx_stream_t stream) {
  if (!nl) return fail(PDX_ERR_ARGUMENT, "null neighbor list");
  hipLaunchKernelGGL(k_rearm, dim3(1), dim3(1), 0, as_stream(stream), nl->state.p);
  PDX_LAUNCH_CHECK();
  return PDX_OK;
}

extern "C" int pdx_nl_resize_capacity(pdx_nl_t nl, int32_t cap) {
  if (!nl) return fail(PDX_ERR_ARGUMENT, "null neighbor list");
  if (cap <= 0) return fail(PDX_ERR_ARGUMENT, "Invalid ELL capacity");
  if ((int64_t)nl->N * cap > INT32_MAX) return fail(PDX_ERR_ARGUMENT, "Neighbor table exceeds the Int32 index range");
  PDX_HIP(hipDeviceSynchronize());
  int rc = nl->neighbors_flat.alloc((size_t)nl->N * cap);
  if (rc) return rc;
  PDX_HIP(hipMemset(nl->neighbors_flat.p, 0xff, sizeof(int32_t) * (size_t)nl->N * cap));
  nl->cap = cap;
  hipLaunchKernelGGL(k_invalidate, dim3(1), dim3(1), 0, 0, nl->state.p);
  PDX_HIP(hipDeviceSynchronize());
  return PDX_OK;
}

extern "C" int pdx_nl_set_box(pdx_nl_t nl, const double box[3], pdx_stream_t stream) {
  if (!nl || !box) return fail(PDX_ERR_ARGUMENT, "null argument");
  const float rlf = std::sqrt(nl->rl2);
  double box3[3] = {box[0], box[1], nl->dim == 2 ? nl->box[2] : box[2]};  // 2-D: z extent kept
  int32_t g[3];
  int rc = grid_for_box(box3, rlf, g);
  if (rc) return rc;
  if (nl->allpairs) {
    const double mn = std::min(box3[0], std::min(box3[1], box3[2]));
    if (!(2.0 * rlf <= mn)) return fail(PDX_ERR_ARGUMENT, "All-pairs neighbor rows need cutoff+skin <= L/2.");
  } else {
    if (g[0] < 3 || g[1] < 3 || g[2] < 3)
      return fail(PDX_ERR_ARGUMENT, "The box became too small for the device cell grid (3 cells per dimension).");
    if (g[0] != nl->nx || g[1] != nl->ny || g[2] != nl->nz) {
      PDX_HIP(hipStreamSynchronize(as_stream(stream)));
      const int ncell = g[0] * g[1] * g[2];
      if ((rc = nl->cell_offsets.alloc(ncell + 1)) || (rc = nl->cell_counts.alloc(ncell)) ||
          (rc = nl->scan_block.alloc(blocks_for(ncell, SCAN_BLOCK))) ||
          (rc = nl->scan_occ.alloc(blocks_for(ncell, SCAN_BLOCK))) || (rc = nl->snap_offsets.alloc(ncell + 1)))
        return rc;
      std::vector<int32_t> ones(ncell + 1, 1);
      PDX_HIP(hipMemcpy(nl->cell_offsets.p, ones.data(), sizeof(int32_t) * (ncell + 1), hipMemcpyHostToDevice));
      PDX_HIP(hipMemset(nl->cell_counts.p, 0, sizeof(int32_t) * ncell));
      nl->nx = g[0]; nl->ny = g[1]; nl->nz = g[2]; nl->ncell = ncell;
    }
  }
  for (int d = 0; d < 3; ++d) nl->box[d] = box3[d];
  {  // cells of the old box are no cover for the new one: no snapshot until the next build
    PDX_HIP(hipStreamSynchronize(as_stream(stream)));
    const int64_t snap0[4] = {-1, 0, 1, 0};
    PDX_HIP(hipMemcpy(nl->snap_state.p, snap0, sizeof(snap0), hipMemcpyHostToDevice));
    nl->snap_host = 0;
  }
  const float geomf[3] = {(float)box3[0], (float)box3[1], (float)box3[2]};
  PDX_HIP(hipMemcpyAsync(nl->geom.p, geomf, sizeof(geomf), hipMemcpyHostToDevice, as_stream(stream)));
  hipLaunchKernelGGL(k_invalidate, dim3(1), dim3(1), 0, as_stream(stream), nl->state.p);
  PDX_HIP(hipStreamSynchronize(as_stream(stream)));
  return PDX_OK;
}

extern "C" int pdx_nl_status(pdx_nl_t nl, int64_t state[PDX_DN_NSTATE], int32_t check, pdx_stream_t stream) {
  if (!nl || !state) return fail(PDX_ERR_ARGUMENT, "null argument");
  PDX_HIP(hipStreamSynchronize(as_stream(stream)));
  PDX_HIP(hipMemcpy(state, nl->state.p, sizeof(int64_t) * PDX_DN_NSTATE, hipMemcpyDeviceToHost));
  if (!check) return PDX_OK;
  if (state[PDX_DN_ERROR] == PDX_DN_CAPACITY_ERROR)
    return fail(PDX_ERR_CAPACITY, "Neighbor capacity " + std::to_string(nl->cap) + " is insufficient; at least " +
                                      std::to_string(state[PDX_DN_REQUIRED]) +
                                      " entries per particle are required. Rebuild with a larger cap.");
  if (state[PDX_DN_ERROR] == PDX_DN_COORDINATE_ERROR)
    return fail(PDX_ERR_COORDINATE,
                "Device ELL requires finite, centered coordinates; execution stopped before rebuilding/forces");
  if (state[PDX_DN_ERROR] != 0) return fail(PDX_ERR_STATE, "Device list stopped with an unknown error code");
  if (state[PDX_DN_VALID] == 0) return fail(PDX_ERR_STATE, "Device ELL has no valid list");
  return PDX_OK;
}

extern "C" int pdx_nl_set_row_lanes(pdx_nl_t nl, int32_t lanes) {
  if (!nl) return fail(PDX_ERR_ARGUMENT, "null neighbor list");
  if (lanes != 0 && lanes != 1 && lanes != 2 && lanes != 4 && lanes != 8 && lanes != 16 && lanes != 32)
    return fail(PDX_ERR_ARGUMENT, "row-build lanes must be 1, 2, 4, 8, 16 or 32 (0: automatic)");
  nl->row_lanes = lanes ? lanes : nl->row_lanes_auto;
  nl->row_lanes_given = lanes ? true : nl->row_lanes_env;
  return PDX_OK;
}
