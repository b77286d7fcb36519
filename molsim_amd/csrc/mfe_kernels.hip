// mfe_kernels.hip -- device kernels of the force engine except the FFT.
//
//   neighbour list ...... SetVListMD / NList skin test (Src/nlist.F90)
//   pair forces ......... UTwoBodyA / UTwoBodyACellList (Src/energy.F90)
//   SPME ................ UEwaldRecSPM spreading and gather
//   standard Ewald ...... UEwaldRecStd
//   bonds ............... UBond
//   integrator .......... VelVer (Src/md.F90), BDStep (Src/bd.F90)
//
// No global floating-point atomics anywhere: charge spreading owns its
// output bricks and accumulates in LDS; energies and virials are reduced
// per block into partial sums that one block adds up in a fixed order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "mfe_device.h"
#include "mfe_fft_device.h"
#include "mfe_internal.h"

namespace mfe {
namespace {

__global__ void k_fill_int(int *p, int n, int v) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_fill_double(double *p, int n, double v) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Exclusive scan of count[0..n) into start[0..n], zeroing count for the
// next use; one block of 1024 threads per replica, each thread owning a
// contiguous chunk; the chunk sums are scanned inside each wavefront with
// shuffles and across the 16 wavefronts through LDS (one barrier).
// which: 0 = cells of the neighbour list, 1 = SPME bricks.
__device__ __forceinline__ void ph_scan(int *count, int *start, int n) {
  __shared__ int wsum[16];
  const int per = (n + blockDim.x - 1) / blockDim.x;
  const int lo = threadIdx.x * per, hi = min(n, lo + per);
  // the chunk in batches of 16 loads in flight
  constexpr int kU = 16;
  int s = 0;
  for (int i0 = lo; i0 < hi; i0 += kU) {
    int v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) v[u] = i0 + u < hi ? count[i0 + u] : 0;
#pragma unroll
    for (int u = 0; u < kU; ++u) s += v[u];
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int x = s;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[wave] = x;
  __syncthreads();
  int wpre = 0;
  for (int w = 0; w < wave; ++w) wpre += wsum[w];
  int run = wpre + x - s;
  for (int i0 = lo; i0 < hi; i0 += kU) {
    int v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) v[u] = i0 + u < hi ? count[i0 + u] : 0;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (i0 + u < hi) {
        start[i0 + u] = run;
        count[i0 + u] = 0;
      }
      run += v[u];
    }
  }
  if (threadIdx.x == blockDim.x - 1) start[n] = wpre + x;
}

// The scan of the cell counts split over kScanBlocks contiguous ranges:
// each range's exclusive prefix is left in place of its counts and its
// total in c_bsum (this phase); after a barrier the scatter adds the totals
// of the earlier ranges (scan_bases) to what it reads.
__device__ __forceinline__ int scan_range(const SysDev &V) {
  return (V.cg.ncells + kScanBlocks - 1) / kScanBlocks;
}

__device__ __forceinline__ void ph_scan_local(const SysDev &V, int blk, int nblk) {
  __shared__ int wsum[16];
  int *count = V.c_count;
  const int n = V.cg.ncells, C = scan_range(V);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int sb = blk; sb < kScanBlocks; sb += nblk) {
    const int lo = min(n, sb * C), hi = min(n, lo + C);
    int carry = 0;
    for (int base = lo; base < hi; base += blockDim.x) {
      const int i = base + threadIdx.x;
      const int v = i < hi ? count[i] : 0;
      int x = v;
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
      }
      if (lane == 63) wsum[wave] = x;
      __syncthreads();
      int wpre = 0, tot = 0;
      for (int w = 0; w < nw; ++w) {
        wpre += w < wave ? wsum[w] : 0;
        tot += wsum[w];
      }
      if (i < hi) count[i] = carry + wpre + x - v;
      carry += tot;
      __syncthreads();
    }
    if (threadIdx.x == 0) V.c_bsum[sb] = carry;
  }
}

// the totals before each range, base[0..kScanBlocks), by the whole block
__device__ __forceinline__ void scan_bases(const SysDev &V, int *base) {
  __shared__ int wsum[kScanBlocks / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int v = 0, x = 0;
  if (threadIdx.x < kScanBlocks) {
    v = V.c_bsum[threadIdx.x];
    x = v;
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) wsum[wave] = x;
  }
  __syncthreads();
  if (threadIdx.x < kScanBlocks) {
    int pre = 0;
    for (int w = 0; w < wave; ++w) pre += wsum[w];
    base[threadIdx.x] = pre + x - v;
  }
  __syncthreads();
}

// ------------------------------------------------------- neighbour lists
// Cells of edge >= rcut + drnlist; a particle's cell is
// floor((x + L/2) * cinv), clamped to the grid.
__device__ __forceinline__ int cell_of(const double *r, const CellGeom &g,
                                       const Box &b, int c[3]) {
  for (int m = 0; m < 3; ++m) {
    int k = (int)floor((r[m] + b.L2[m]) * g.cinv[m]);
    c[m] = min(max(k, 0), g.n[m] - 1);
  }
  return c[0] + g.n[0] * (c[1] + g.n[1] * c[2]);
}

// The mixed path's FP32 position of a particle at x (FP64) in cell c,
// relative to the cell's reference point -L/2 + (c + 1/2) hf per axis and
// taken into [-L/2, L/2] (the particle may have crossed the box edge since
// the list was built), with its type in the fourth word.
__device__ __forceinline__ float4 rel_pos(const SysDev &V, const double *x, int c, int type) {
  const CellGeom &g = V.cg;
  const int cc[3] = {c % g.n[0], (c / g.n[0]) % g.n[1], c / (g.n[0] * g.n[1])};
  float r[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const double o = -V.box.L2[m] + (cc[m] + 0.5) * g.hf[m];
    double d = x[m] - o;
    if (d > V.box.L2[m]) d -= V.box.L[m];
    else if (d < -V.box.L2[m]) d += V.box.L[m];
    r[m] = (float)d;
  }
  return make_float4(r[0], r[1], r[2], __int_as_float(type));
}

// The rebuild's phases, each over threads t0, t0 + nt, ...: run as five
// kernels (batches, explicit builds) or as the phases of k_rebuild.
__device__ __forceinline__ void ph_cell_count(const SysDev &V, int t0, int nt) {
  const double *__restrict__ ro = V.ro;
  const CellGeom g = V.cg;
  const Box b = V.box;
  for (int i = t0; i < V.np; i += nt) {
    int c3[3];
    const int c = cell_of(ro + 3 * i, g, b, c3);
    V.c_of[i] = c;
    V.c_slot[i] = atomicAdd(&V.c_count[c], 1);
  }
}

// Particles placed into their cells in the order of the count's atomics,
// in c_pos (free until the list build writes it); base: the ranges' totals
// (scan_bases), with the final cell starts written here, or null when
// c_start already holds them.
__device__ __forceinline__ void ph_cell_scatter(const SysDev &V, int t0, int nt,
                                                const int *base) {
  const int C = scan_range(V), nc = V.cg.ncells;
  for (int i = t0; i < V.np; i += nt) {
    const int c = V.c_of[i];
    const int st = base ? V.c_count[c] + base[c / C] : V.c_start[c];
    V.c_pos[st + V.c_slot[i]] = i;
  }
  if (!base) return;
  for (int c = t0; c < nc; c += nt) V.c_start[c] = V.c_count[c] + base[c / C];
  if (t0 == 0) V.c_start[nc] = V.np;
}

// Members of each cell in ascending particle index (deterministic lists),
// and the positions and types in that order.  A particle's place is the
// number of its cell's members with a smaller index: a thread per particle
// counts them, so a crowded cell (a box of fewer than three cells per axis
// is one cell) costs its occupancy, not a serial sort by one thread:
// 1000 ions in one cell 31 ms -> 27 us.  Also clears the counts.
__device__ __forceinline__ void ph_cell_rank(const SysDev &V, int t0, int nt) {
  const int *__restrict__ tmp = V.c_pos;
  const int *__restrict__ start = V.c_start;
  for (int t = t0; t < V.np; t += nt) {
    const int i = tmp[t];
    const int c = V.c_of[i];
    const double x = V.ro[3 * i], y = V.ro[3 * i + 1], z = V.ro[3 * i + 2];
    const int ty = V.type[i];
    const int lo = start[c], hi = start[c + 1];
    int rank = 0;
    int k = lo;
    for (; k + 8 <= hi; k += 8) {
      int v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = tmp[k + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) rank += v[u] < i ? 1 : 0;
    }
    for (; k < hi; ++k) rank += tmp[k] < i ? 1 : 0;
    const int p = lo + rank;
    V.c_sorted[p] = i;
    V.ro_s[3 * p] = x;
    V.ro_s[3 * p + 1] = y;
    V.ro_s[3 * p + 2] = z;
    V.type_s[p] = ty;
    if (V.pos_f) {
      const double r[3] = {x, y, z};
      V.pos_f[p] = rel_pos(V, r, c, ty);
    }
  }
  for (int c = t0; c < V.cg.ncells; c += nt) V.c_count[c] = 0;
}

// positions and types in cell order (ro_s, type_s)
__device__ __forceinline__ void ph_sort_pos(const SysDev &V, int t0, int nt) {
  for (int t = t0; t < V.np; t += nt) {
    const int i = V.c_sorted[t];
    // every load before the first store
    const double x = V.ro[3 * i], y = V.ro[3 * i + 1], z = V.ro[3 * i + 2];
    const int ty = V.type[i];
    V.ro_s[3 * t] = x;
    V.ro_s[3 * t + 1] = y;
    V.ro_s[3 * t + 2] = z;
    V.type_s[t] = ty;
    if (V.pos_f) {
      const double r[3] = {x, y, z};
      V.pos_f[t] = rel_pos(V, r, V.c_of[i], ty);
    }
  }
}

// Full Verlet list: every j != i with r2 < (rcut+drnlist)^2 (SetVListMD's
// test, Src/nlist.F90:746-750).  Particles are taken in cell order
// (t -> i = sorted[t], positions from ro_s) and partners stored by their
// cell-order position, so the pair kernel reads neighbouring positions from
// neighbouring memory; the list is column-major, nbr[k*np + t].  The half
// list the reference keeps is the checkerboard subset of this set.
//
// 1 << lsh lanes share a particle: of each row of cells they test 4 << lsh
// candidates at a time and append the hits in candidate order (ballot
// prefix), so the list is the same for any lsh.  The test is a dependent
// load and some 20 FP64 operations, and one lane per particle leaves
// crowded cells to a few wavefronts (list_lsh_for chooses).
__device__ __forceinline__ void ph_nlist_build(const SysDev &V, int t0, int nt, int lsh) {
  const double *__restrict__ ros = V.ro_s;
  const int np = V.np;
  const CellGeom g = V.cg;
  const Box b = V.box;
  const int *__restrict__ cof = V.c_of;
  const int *__restrict__ start = V.c_start;
  const int *__restrict__ sorted = V.c_sorted;
  const double rs2 = V.rs2;
  const int maxnn = V.maxnn;
  int *__restrict__ nn = V.nn;
  int *__restrict__ nbr = V.nbr;
  int *flags = V.flags;
  double *drosum = V.drosum;
  const int lanes = 1 << lsh, sub = t0 & (lanes - 1);
  const int gsh = (threadIdx.x & 63) & ~(lanes - 1);
  const unsigned gmask = lanes == 1 ? 1u : ((1u << lanes) - 1u);
  const unsigned below = (1u << sub) - 1u;
  for (int t = t0 >> lsh; t < np; t += nt >> lsh) {
    const int i = sorted[t];
    const double xi = ros[3 * t], yi = ros[3 * t + 1], zi = ros[3 * t + 2];
    const int c = cof[i];
    const int cx = c % g.n[0], cy = (c / g.n[0]) % g.n[1], cz = c / (g.n[0] * g.n[1]);
    const int rx = g.n[0] > 1 ? 1 : 0, ry = g.n[1] > 1 ? 1 : 0, rz = g.n[2] > 1 ? 1 : 0;
    int n = 0;
    for (int dz = -rz; dz <= rz; ++dz) {
      const int z = (cz + dz + g.n[2]) % g.n[2];
      // the pair's offset code per axis (see CellGeom): -d inside the box,
      // +-2 across its edge, 0 on an axis of one cell
      const int kz = rz ? (cz + dz < 0 ? 2 : (cz + dz >= g.n[2] ? -2 : -dz)) : 0;
      for (int dy = -ry; dy <= ry; ++dy) {
        const int y = (cy + dy + g.n[1]) % g.n[1];
        const int ky = ry ? (cy + dy < 0 ? 2 : (cy + dy >= g.n[1] ? -2 : -dy)) : 0;
        // the row's cells x-1, x, x+1 (one on an axis of one cell): their
        // bounds loaded together, then their particles taken as one
        // sequence in the same order (cell by cell, p ascending), four
        // positions per lane in flight at a time
        int cs[3] = {0, 0, 0}, cn[3] = {0, 0, 0};
        unsigned cd[3] = {0u, 0u, 0u};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const int dx = k - 1;
          if (rx || dx == 0) {
            const int x = (cx + dx + g.n[0]) % g.n[0];
            const int kx = rx ? (cx + dx < 0 ? 2 : (cx + dx >= g.n[0] ? -2 : -dx)) : 0;
            cd[k] = (unsigned)((kx + 2) + 5 * (ky + 2) + 25 * (kz + 2)) << kNbrCodeShift;
            const int cc = x + g.n[0] * (y + g.n[1] * z);
            cs[k] = start[cc];
            cn[k] = start[cc + 1];
          }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) cn[k] -= cs[k];
        const int n01 = cn[0] + cn[1], tot = n01 + cn[2];
        for (int q0 = 0; q0 < tot; q0 += 4 << lsh) {
          int pp[4], kk[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int q = q0 + (u << lsh) + sub;
            const int k = q < cn[0] ? 0 : (q < n01 ? 1 : 2);
            kk[u] = k;
            // past the row's end: the particle itself (skipped below)
            pp[u] = q < tot ? cs[k] + q - (k == 0 ? 0 : (k == 1 ? cn[0] : n01)) : t;
          }
          double xj[4], yj[4], zj[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            xj[u] = ros[3 * pp[u]];
            yj[u] = ros[3 * pp[u] + 1];
            zj[u] = ros[3 * pp[u] + 2];
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            double ddx = xi - xj[u], ddy = yi - yj[u], ddz = zi - zj[u];
            const double r2 = pbcr2(ddx, ddy, ddz, b);
            const bool hit = pp[u] != t && r2 < rs2;
            const unsigned m = lanes == 1 ? (hit ? 1u : 0u)
                                          : (unsigned)(__ballot(hit) >> gsh) & gmask;
            if (hit) {
              const int at = n + __popc(m & below);
              const unsigned code = kk[u] == 0 ? cd[0] : (kk[u] == 1 ? cd[1] : cd[2]);
              if (at < maxnn) nbr[(size_t)at * np + t] = (int)((unsigned)pp[u] | code);
            }
            n += __popc(m);
          }
        }
      }
    }
    if (sub == 0) {
      // on overflow only the stored maxnn partners are visible to the pair
      // kernel; the call reports MFE_E_NEIGH_CAPACITY
      nn[t] = min(n, maxnn);
      if (n > maxnn) atomicOr(&flags[0], ERR_CAPACITY);
      // k_move keeps the cell-ordered positions current through c_pos
      // until the next rebuild
      V.c_pos[i] = t;
      if (drosum) {
        drosum[3 * i] = 0.0;
        drosum[3 * i + 1] = 0.0;
        drosum[3 * i + 2] = 0.0;
      }
    }
  }
}

#define MFE_GATE                                \
  const SysDev &V = sys[blockIdx.z];           \
  if (gated && V.flags[1] == 0) return;        \
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;

__global__ void k_cell_count(const SysDev *__restrict__ sys, int gated) {
  MFE_GATE
  ph_cell_count(V, t0, nt);
}

__global__ void __launch_bounds__(1024) k_cell_scan(const SysDev *__restrict__ sys, int gated) {
  const SysDev &V = sys[blockIdx.z];
  if (gated && V.flags[1] == 0) return;
  ph_scan_local(V, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(kBlock) k_cell_scatter(const SysDev *__restrict__ sys,
                                                         int gated) {
  MFE_GATE
  __shared__ int base[kScanBlocks];
  scan_bases(V, base);
  ph_cell_scatter(V, t0, nt, base);
}

__global__ void k_cell_rank(const SysDev *__restrict__ sys, int gated) {
  MFE_GATE
  ph_cell_rank(V, t0, nt);
}

__global__ void __launch_bounds__(kBlock) k_nlist_build(const SysDev *__restrict__ sys,
                                                        int gated) {
  MFE_GATE
  ph_nlist_build(V, t0, nt, V.list_lsh);
  if (t0 == 0 && gated) V.flags[2] += 1;
}
#undef MFE_GATE

// Grid-wide barrier of k_rebuild, whose blocks are all resident (one per
// CU), in two levels: the blocks arrive on kBarGroups group counters
// (block b on counter b % kBarGroups, each counter on a line of its own,
// so arrivals on different counters do not queue behind one another), the
// last block of each group on the top counter, and the last of those
// advances the generation.  Each wave waits for its stores (in L2), the
// block meets at s_barrier; thread 0 then arrives with acquire-release
// increments (a release writes the XCD's L2 back, so the other XCDs see
// the block's data; a group's last block has acquired its group's data
// before it releases on the top counter), the last arrival at each level
// resets that level's counter, the final one advances the generation
// (release), the others poll it (relaxed) and take one acquire fence,
// which invalidates the CU's stale lines for the whole block.  The words
// are laid out as kBarWords in mfe_internal.h.  The wait is bounded: after `spin` polls a
// block raises ERR_SYNC and leaves.  A block goes on to the next phase
// only when every block has arrived (so the data of the finished phase is
// complete) and no block has given up; otherwise it returns false, the
// kernel ends in every block, and the host reports the error, clears the
// barrier and the cell counts, and rebuilds the list from scratch.
constexpr int kGridSpin = 1 << 22;

__device__ __forceinline__ bool grid_sync(unsigned *bar, int *flags, int spin) {
  __shared__ int ok_s;
  // every wave waits for its own stores to be acknowledged (in L2) before
  // the block barrier (a workgroup-scope barrier does not wait for them)
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    int ok = 1;
    const unsigned nblk = gridDim.x;
    const unsigned ng = nblk < (unsigned)kBarGroups ? nblk : (unsigned)kBarGroups;
    const unsigned grp = blockIdx.x % ng;
    const unsigned ingrp = (nblk - 1u - grp) / ng + 1u;  // blocks of this group
    unsigned *gc = bar + grp * kBarStride;
    unsigned *gen_p = bar + kBarGen, *top = bar + kBarTop;
    const unsigned gen = __hip_atomic_load(gen_p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bool final_block = false;
    if (__hip_atomic_fetch_add(gc, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1u == ingrp) {
      __hip_atomic_store(gc, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (__hip_atomic_fetch_add(top, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1u == ng) {
        __hip_atomic_store(top, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_add(gen_p, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        final_block = true;
      }
    }
    if (!final_block) {
      int spins = 0;
      while (__hip_atomic_load(gen_p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gen) {
        if (++spins > spin) {
          atomicOr(&flags[0], ERR_SYNC);
          ok = 0;
          break;
        }
        __builtin_amdgcn_s_sleep(8);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    if (ok && (__hip_atomic_load(&flags[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) &
               ERR_SYNC))
      ok = 0;
    ok_s = ok;
  }
  __syncthreads();
  return ok_s != 0;
}

// The list rebuild's phases in order, separated by grid barriers, run by
// every block of a launch whose blocks are all resident (one 1024-thread
// block per CU).  A block leaves as soon as a barrier gives up.
__device__ __forceinline__ void rebuild_phases(const SysDev &V, unsigned *bar, int spin) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
  __shared__ int base[kScanBlocks];
  ph_cell_count(V, t0, nt);
  if (!grid_sync(bar, V.flags, spin)) return;
  ph_scan_local(V, blockIdx.x, gridDim.x);
  if (!grid_sync(bar, V.flags, spin)) return;
  scan_bases(V, base);
  ph_cell_scatter(V, t0, nt, base);
  if (!grid_sync(bar, V.flags, spin)) return;
  ph_cell_rank(V, t0, nt);
  if (!grid_sync(bar, V.flags, spin)) return;
  ph_nlist_build(V, t0, nt, V.list_lsh);
  if (t0 == 0) V.flags[2] += 1;
}

// The gated list rebuild of one engine as one kernel: it returns at once
// when the skin test did not fire (one launch per step instead of five),
// or after a failed rebuild earlier in the same call (the list is void
// until the host rebuilds it); otherwise the phases run.  Launched with
// one 1024-thread block per CU, so all blocks are resident.
// gate: the engine's flags (V.flags), passed directly so that the skin
// decision is one load away rather than behind the view's.
__global__ void __launch_bounds__(1024) k_rebuild(const SysDev *__restrict__ sys,
                                                  const int *__restrict__ gate, unsigned *bar,
                                                  int spin) {
  // one thread's reading decides for the block (see k_finalize_rebuild)
  __shared__ int go_s;
  if (threadIdx.x == 0)
    go_s = gate[1] != 0 &&
           !(__hip_atomic_load(&gate[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ERR_SYNC);
  __syncthreads();
  if (!go_s) return;
  rebuild_phases(sys[0], bar, spin);
}

// positions and types in cell order for the pair kernel (every UTotal)
__global__ void k_sort_pos(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  ph_sort_pos(V, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// ------------------------------------------------------------ pair forces
// First interval (in storage order) with r2 >= zlow -- the interval the
// reference's linear walk stops at (Src/energy.F90:482-486).  zlow
// decreases along the table; the walk starts at the interval kb of r2's
// bin and moves to lower r2 while r2 < zlow, then to higher r2 while the
// next bound is still <= r2.  Both moves together reach the first k with
// r2 >= zl(k) from any start, so the bin only sets the walk's length
// (0-2 steps for bins about as wide as the intervals).
template <typename Z>
__device__ __forceinline__ int find_interval(const Z &zl, int n, double r2, int kb) {
  int k = kb;
  while (k < n - 1 && !(r2 >= zl(k))) ++k;
  while (k > 0 && r2 >= zl(k - 1)) --k;
  return k;
}

// list entries a lane loads together (indices, then positions)
constexpr int kPairBatch = 4;

// The first `bytes` (a multiple of 16) of the tables' image copied into LDS,
// 16 bytes per load and eight loads in flight per thread: one memory round
// trip for what element-wise copies of the bins, bounds and coefficients
// took a dozen for (about 12 us of a small system's pair launch).
__device__ __forceinline__ void stage_image(unsigned char *lds, const TableDev &t,
                                            size_t bytes) {
  uint4 *dst = reinterpret_cast<uint4 *>(lds);
  batched_copy(
      (int)(bytes / 16), [&](int e) -> uint4 { return t.img[e]; },
      [&](int e, uint4 v) { dst[e] = v; });
}

// The sum of a particle's lanes' values (lanes a power of two, the same for
// the whole block), in a fixed order.
__device__ __forceinline__ double lane_sum(double x, int lanes) {
  if (lanes >= 2) x += quad_swap<kXor1>(x);
  if (lanes >= 4) x += quad_swap<kXor2>(x);
  if (lanes >= 8) x += quad_swap<kHalfMirror>(x);
  if (lanes >= 16) x += quad_swap<kMirror>(x);
  if (lanes >= 32) x += __shfl_xor(x, 16, 64);
  if (lanes >= 64) x += __shfl_xor(x, 32, 64);
  return x;
}

// k_skin_blocks' computation for skin blocks sb0 and sb0 + 1 (256
// particles each, the k_move partition), one per half of a 512-thread
// block: the same maxima in the same order, so the same candidates.
__device__ __forceinline__ void skin_two_blocks(const SysDev &V, int sb0) {
  __shared__ double wred[kPairBlock / 64];
  const int sub = threadIdx.x >> 8, t = threadIdx.x & 255;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, w0 = 4 * sub;
  const int sb = sb0 + sub;
  const bool valid = sb < V.nblk_np;
  const double *part_max = V.part + V.off_move;
  // running maximum entering the block: the maxima of the earlier blocks
  double pm = 0.0;
  if (valid)
    for (int b2 = t; b2 < sb; b2 += 256) pm = fmax(pm, part_max[b2]);
  for (int w = 32; w > 0; w >>= 1) pm = fmax(pm, __shfl_down(pm, w, 64));
  if (lane == 0) wred[wv] = pm;
  __syncthreads();
  const double P = fmax(fmax(wred[w0], wred[w0 + 1]), fmax(wred[w0 + 2], wred[w0 + 3]));
  __syncthreads();
  const int i = sb * 256 + t;
  const double v = (valid && i < V.np) ? V.r2disp[i] : 0.0;
  // inclusive max-scan inside the wavefront, then the earlier wavefronts
  double inc = v;
  for (int off = 1; off < 64; off <<= 1) {
    const double y = __shfl_up(inc, off, 64);
    if (lane >= off) inc = fmax(inc, y);
  }
  double excl = __shfl_up(inc, 1, 64);
  if (lane == 0) excl = 0.0;
  if (lane == 63) wred[wv] = inc;
  __syncthreads();
  double pw = 0.0;
  for (int k = w0; k < wv; ++k) pw = fmax(pw, wred[k]);
  const double before = fmax(P, fmax(pw, excl));
  double cand = (valid && i < V.np && !(v > before)) ? v : 0.0;
  __syncthreads();
  for (int w = 32; w > 0; w >>= 1) cand = fmax(cand, __shfl_down(cand, w, 64));
  if (lane == 0) wred[wv] = cand;
  __syncthreads();
  if (t == 0 && valid)
    V.part[V.off_skin + sb] =
        fmax(fmax(wred[w0], wred[w0 + 1]), fmax(wred[w0 + 2], wred[w0 + 3]));
}

// Pair forces over the Verlet list.  V.pair_lanes lanes share one particle
// (cell order i) and split its list k = lane, lane + lanes, ...; their
// partial forces are combined by lane exchanges in FP64 in a fixed order, so
// forces need no atomics and stay deterministic.  Every pair is seen from
// both ends, so its energy and virial carry weight 1/2.  semantics: 0 =
// vlist (r2 <= rcut2 kept), 1 = cell list (r2 < rcut2 kept).
//
// The grid is persistent: nblk_pair (<= kPairGridMax) blocks each stage
// the tables in LDS once -- r2 bins, interval bounds and, with CF, the
// polynomial coefficients -- and then walk one contiguous range of chunks
// of kPairBlock / lanes particles.  A lane loads the indices of
// kPairBatch of its entries together, then their positions, then
// evaluates them.  NT bounds the number of types: up to 4 the energies
// accumulate per pair type in registers over all chunks, else per partner
// type, converted per chunk into a per-wavefront LDS row; either way in a
// fixed order, and per block into the partials.
// With skin (MD/BD steps) blocks from pgrid on take the skin test's block
// candidates (two k_move blocks each) instead of a separate launch.
template <int NT, bool CF>
__global__ void __launch_bounds__(kPairBlock) __attribute__((amdgpu_waves_per_eu(4)))
k_pair(const SysDev *__restrict__ sys, int energy, int pgrid, int skin) {
  using CT = double;
  const SysDev &V = sys[blockIdx.z];
  if (skin && (int)blockIdx.x >= pgrid) {
    skin_two_blocks(V, 2 * ((int)blockIdx.x - pgrid));
    return;
  }
  const int blk = xcd_block(blockIdx.x, pgrid);
  const int nb = V.nblk_pair;
  if (blk >= nb) return;
  const double *__restrict__ ro = V.ro_s;
  const int *__restrict__ type = V.type_s;
  const int np = V.np;
  const int *__restrict__ nn = V.nn;
  const int *__restrict__ nbr = V.nbr;
  const Box b = V.box;
  const TableDev t = V.tab;
  const int semantics = V.nlsem;
  int *flags = V.flags;
  extern __shared__ __align__(16) unsigned char pair_lds[];
  __shared__ PairRec rec_s[MFE_MAX_PAIRS];
  __shared__ int pidx_s[MFE_MAX_TYPES * MFE_MAX_TYPES];
  __shared__ double wacc[kPairBlock / 64][MFE_MAX_PAIRS + 1];
  const int P = t.nptpt, nbin = t.nbin, nzl = t.nzl, npt = t.npt;
  const bool lds_zl = CF || t.lds_mode >= 1;
  const size_t bb = pair_bin_bytes(P, nbin);
  unsigned short *bin_s = reinterpret_cast<unsigned short *>(pair_lds);
  double *zl_s = reinterpret_cast<double *>(pair_lds + bb);
  CT *cf_s = reinterpret_cast<CT *>(pair_lds + bb + pair_zl_bytes(nzl));
  stage_image(pair_lds, t,
              bb + (lds_zl ? pair_zl_bytes(nzl) : 0) +
                  (CF ? (size_t)nzl * kCoefStride * sizeof(CT) : 0));
  for (int k = threadIdx.x; k < P; k += blockDim.x) rec_s[k] = t.rec[k];
  for (int k = threadIdx.x; k < npt * npt; k += blockDim.x) pidx_s[k] = t.pairidx[k];
  const int l64 = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int k = l64; k <= P; k += 64) wacc[wv][k] = 0.0;
  __syncthreads();
  // the 12 stored coefficients of interval iv (16-byte loads)
  auto coefs = [&](int iv, CT *c) {
    const double2 *q = CF ? reinterpret_cast<const double2 *>(cf_s) + 6 * iv
                          : reinterpret_cast<const double2 *>(t.coef) + 6 * iv;
#pragma unroll
    for (int h = 0; h < 6; ++h) {
      const double2 v = q[h];
      c[2 * h] = v.x;
      c[2 * h + 1] = v.y;
    }
  };
  auto zlow = [&](int idx) -> double {
    if constexpr (CF) return zl_s[idx];
    else return lds_zl ? zl_s[idx] : t.zlow[idx];
  };
  // lanes per particle (lsh their log2)
  const int LANES = V.pair_lanes, lsh = __builtin_ctz(LANES);
  const int lane = threadIdx.x & (LANES - 1);
  // energy accumulators: per pair type for up to 4 types (kept over all
  // chunks), else per partner type (converted to pair types per chunk)
  constexpr bool kRegE = NT <= 4;
  constexpr int NA = kRegE ? NT * (NT + 1) / 2 : NT;
  double ej[NA];
#pragma unroll
  for (int k = 0; k < NA; ++k) ej[k] = 0.0;
  double vir = 0.0;
  double fx, fy, fz;
  int ti = 0;
  // pair index of this particle with partner type u in bits 8u..8u+7
  unsigned long long ptp = 0;
  int err = 0;    // error bits, flagged once at the end
  // one list entry: partner of type tj at (dx, dy, dz) = r_i - r_j.  The
  // LDS reads come before any branch, so the entries of a batch overlap.
  auto eval = [&](double dx, double dy, double dz, int tj) {
    const double r2 = pbcr2(dx, dy, dz, b);
    const bool in = semantics == 0 ? !(r2 > t.rcut2) : (r2 < t.rcut2);
    const int p = (int)((ptp >> (8 * tj)) & 0xffu);
    const PairRec R = rec_s[p];
    // interval of r2 (of lo below the table: such an entry is an error
    // or a hard core, and only its flags count)
    const double r2c = fmax(r2, R.lo);
    const float sf = __builtin_amdgcn_rcpf((float)r2c);
    const float xb = fminf(fmaxf((sf - R.s_lo) * R.s_inv, 0.0f), (float)(nbin - 1));
    const int bk = bin_s[p * nbin + (int)xb];
    const int o = R.off, n = R.nint, kb = bk & (kSlowBin - 1);
    const double z0 = zlow(o + kb), z1 = zlow(o + min(kb + 1, n - 1));
    int iv;
    double zv;
    if (bk & kSlowBin) {
      auto zl = [&](int k) -> double { return zlow(o + k); };
      iv = find_interval(zl, n, r2c, kb);
      zv = zlow(o + iv);
    } else {
      const bool at = r2c >= z0;
      iv = at ? kb : min(kb + 1, n - 1);
      zv = at ? z0 : z1;
    }
    CT c[kCoefStride];
    coefs(o + iv, c);
    const bool hc = r2 < R.r2at;
    const bool ov = !hc && r2 < R.r2um;
    const bool te = !hc && !ov && !(r2 >= R.lo);
    if (in) err |= (ov ? ERR_OVERLAP : 0) | (te ? ERR_TABLE : 0);
    if (!in || ov || te) return;
    const double d = r2 - zv;
    double fsum = c[6] + d * (c[7] + d * (c[8] + d * (c[9] + d * c[10])));
    double usum = c[0] + d * (c[1] + d * (c[2] + d * (c[3] + d * (c[4] + d * c[5]))));
    if (hc) {
      usum = 1e10;
      fsum = 1e10;
    } else if (V.nknot) {
      // additive spline term: u += sum c w, fsum -= u'/r
      const double r = sqrt(r2);
      int ki;
      double w[4], dw[4];
      if (knot_weights(r, V.knot_r0, V.knot_dinv, V.nknot, ki, w, dw)) {
        const double *kc = V.knot_c + (size_t)p * V.nknot + ki;
        const double du = kc[0] * w[0] + kc[1] * w[1] + kc[2] * w[2] + kc[3] * w[3];
        const double dup = (kc[0] * dw[0] + kc[1] * dw[1] + kc[2] * dw[2] + kc[3] * dw[3]) *
                           V.knot_dinv;
        usum += du;
        fsum -= dup / r;
      }
    }
    fx += fsum * dx;
    fy += fsum * dy;
    fz += fsum * dz;
    if (energy) {
#pragma unroll
      for (int k2 = 0; k2 < NA; ++k2) ej[k2] += (k2 == (kRegE ? p : tj)) ? 0.5 * usum : 0.0;
      vir -= 0.5 * fsum * r2;
    }
  };
  // this block's chunks: an even share of the contiguous chunk range
  const int kChunk = kPairBlock >> lsh;
  const int nch = (np + kChunk - 1) / kChunk;
  const int ch0 = (int)((long long)blk * nch / nb), ch1 = (int)((long long)(blk + 1) * nch / nb);
  for (int ch = ch0; ch < ch1; ++ch) {
    const int i = ch * kChunk + (threadIdx.x >> lsh);
    if (!kRegE) {
#pragma unroll
      for (int k = 0; k < NA; ++k) ej[k] = 0.0;
    }
    fx = fy = fz = 0.0;
    ti = 0;
    if (i < np) {
      const double xi = ro[3 * i], yi = ro[3 * i + 1], zi = ro[3 * i + 2];
      ti = type[i];
      ptp = 0;
      for (int u = 0; u < npt; ++u)
        ptp |= (unsigned long long)pidx_s[ti * npt + u] << (8 * u);
      const int n = nn[i];
      // the loads are unconditional (rows clamped into the list; past its
      // end the particle itself) so no branch makes the compiler wait for
      // them one by one
      const int last = n - 1;
      for (int k0 = lane; k0 < n; k0 += kPairBatch * LANES) {
        int js[kPairBatch];
#pragma unroll
        for (int g = 0; g < kPairBatch; ++g) {
          const int kk = k0 + g * LANES;
          const int jr = (int)((unsigned)nbr[(size_t)max(0, min(kk, last)) * np + i] & kNbrIdxMask);
          js[g] = kk < n ? jr : i;
        }
        double xs[kPairBatch], ys[kPairBatch], zs[kPairBatch];
        int ts[kPairBatch];
#pragma unroll
        for (int g = 0; g < kPairBatch; ++g) {
          xs[g] = ro[3 * js[g]];
          ys[g] = ro[3 * js[g] + 1];
          zs[g] = ro[3 * js[g] + 2];
          ts[g] = type[js[g]];
        }
#pragma unroll
        for (int g = 0; g < kPairBatch; ++g)
          if (k0 + g * LANES < n) eval(xi - xs[g], yi - ys[g], zi - zs[g], ts[g]);
      }
    }
    fx = lane_sum(fx, LANES);
    fy = lane_sum(fy, LANES);
    fz = lane_sum(fz, LANES);
    if (i < np && lane == 0) {
      const int io = V.c_sorted[i];
      V.force[3 * io] = fx;
      V.force[3 * io + 1] = fy;
      V.force[3 * io + 2] = fz;
    }
    if (energy && !kRegE) {
      // pair-type energies of this chunk: wave_sum in each
      // wavefront, added to the wavefront's own LDS row
      for (int k = 0; k < P; ++k) {
        double v = 0.0;
        if (i < np) {
#pragma unroll
          for (int u = 0; u < NA; ++u)
            if (u < npt && pidx_s[ti * npt + u] == k) v += ej[u];
        }
        v = wave_sum(v);
        if (l64 == 0) wacc[wv][k] += v;
      }
    }
  }
  if (err) atomicOr(&flags[0], err);
  if (energy) {
    if (kRegE) {
      // the pair-type energies of all chunks: wave_sum in each
      // wavefront
#pragma unroll
      for (int k = 0; k < NA; ++k) {
        const double v = wave_sum(ej[k]);
        if (l64 == 0 && k < P) wacc[wv][k] = v;
      }
    }
    // the virial, then per-block partials, component-major (component k
    // of block b at k * nblk_pair + b), the wavefronts summed in order
    const double v = wave_sum(vir);
    if (l64 == 0) wacc[wv][P] = v;
    __syncthreads();
    double *out = V.part + V.off_pair + blk;
    for (int k = threadIdx.x; k <= P; k += blockDim.x) {
      double s2 = wacc[0][k];
      for (int w = 1; w < (int)(blockDim.x >> 6); ++w) s2 += wacc[w][k];
      out[(size_t)k * nb] = s2;
    }
  }
}

// The mixed path's tables as a pair evaluation sees them (in LDS, or the
// coefficients in global memory when they do not fit): bins, FP32 interval
// bounds, coefficient records, per-pair records, and the list semantics.
struct PairTabF {
  const unsigned short *bin;
  const float *zl;
  const float *cf;
  const PairRecF *rec;
  int nbin, semantics;
  float rc2;
};

// One FP32 pair term at separation (dx, dy, dz), pair type p: false when
// the pair is outside the cut-off or an error (overlap below r2umin, r2
// below the table: bits added to err); else the force factor fs (force =
// fs * d), the energy usum (FP64; with energy) and r2.  The interval is
// chosen on FP32 bounds and the polynomials are evaluated in d = r2 -
// (float)zlow; the FP32 coefficients were re-expanded about the rounded
// bound, so that rounding shifts no interval's argument.  The interval
// constant w0 enters in FP64 (its FP32 value plus the rounding kept in
// slot 11).  KN: the additive spline term (when the replica carries one).
template <bool KN>
__device__ __forceinline__ bool pair_eval_f(const SysDev &V, const PairTabF &T, float dx, float dy,
                                            float dz, int p, int energy, float &fs,
                                            double &usum, float &r2, int &err) {
  r2 = dx * dx + dy * dy + dz * dz;
  const bool in = T.semantics == 0 ? !(r2 > T.rc2) : (r2 < T.rc2);
  const PairRecF R = T.rec[p];
  const float r2c = fmaxf(r2, R.lo);
  const float sf = __builtin_amdgcn_rcpf(r2c);
  const float xb = fminf(fmaxf((sf - R.s_lo) * R.s_inv, 0.0f), (float)(T.nbin - 1));
  const int bk = T.bin[p * T.nbin + (int)xb];
  const int o = R.off, n = R.nint, kb = bk & (kSlowBin - 1);
  const float z0 = T.zl[o + kb], z1 = T.zl[o + min(kb + 1, n - 1)];
  int iv;
  float zv;
  if (bk & kSlowBin) {
    auto zl = [&](int k) -> float { return T.zl[o + k]; };
    iv = find_interval(zl, n, r2c, kb);
    zv = T.zl[o + iv];
  } else {
    const bool at = r2c >= z0;
    iv = at ? kb : min(kb + 1, n - 1);
    zv = at ? z0 : z1;
  }
  const float4 *q = reinterpret_cast<const float4 *>(T.cf) + 3 * (o + iv);
  const float4 c0 = q[0], c1 = q[1], c2 = q[2];
  const bool hc = r2 < R.r2at;
  const bool ov = !hc && r2 < R.r2um;
  const bool te = !hc && !ov && !(r2 >= R.lo);
  if (in) err |= (ov ? ERR_OVERLAP : 0) | (te ? ERR_TABLE : 0);
  if (!in || ov || te) return false;
  const float df = r2 - zv;
  // c0 = (w0, w1, w2, w3), c1 = (w4, w5, f0, f1), c2 = (f2, f3, f4, w0 rounding)
  fs = c1.z + df * (c1.w + df * (c2.x + df * (c2.y + df * c2.z)));
  usum = 0.0;
  if (energy) {
    const float up = df * (c0.y + df * (c0.z + df * (c0.w + df * (c1.x + df * c1.y))));
    usum = ((double)c0.x + (double)c2.w) + (double)up;
  }
  if (hc) {
    usum = 1e10;
    fs = 1e10f;
  } else if (KN && V.nknot) {
    const double r = sqrt((double)r2);
    int ki;
    double w[4], dw[4];
    if (knot_weights(r, V.knot_r0, V.knot_dinv, V.nknot, ki, w, dw)) {
      const double *kc = V.knot_c + (size_t)p * V.nknot + ki;
      usum += kc[0] * w[0] + kc[1] * w[1] + kc[2] * w[2] + kc[3] * w[3];
      fs -= (float)((kc[0] * dw[0] + kc[1] * dw[1] + kc[2] * dw[2] + kc[3] * dw[3]) *
                    V.knot_dinv / r);
    }
  }
  return true;
}

// The mixed path's pair forces: the list walk, partition and reductions of
// k_pair, in FP32 (pair_eval_f).  Positions come from pos_f (relative to
// the particle's cell reference point, 16 bytes with the type); a list
// entry's code names the pair's cell offset, kept in LDS per code, so
// dx = x_i - x_j + offset is formed in FP32 from values of at most a cell
// edge or so.  Forces are Kahan-compensated FP32 sums, energies FP64 per
// partner type, flushed into the wavefront's LDS row per chunk.  KN:
// some replica carries the additive spline term.  V.pair_lanes lanes share
// a particle's list (pair_lanes_for); a replica's choice is its own, so it
// computes the same alone and in a batch.  POS64: the replicas whose box has an
// axis of fewer than three list cells, where cell-relative coordinates
// would span half the box -- the pair's separation is formed in FP64 from
// the cell-ordered positions and rounded once; the other replicas' blocks
// return (a group launches both variants when it holds both kinds).
// The body takes its block index bxi (the launch's own, or its place in a
// launch that also carries other work).
template <int NT, bool CF, bool KN, bool POS64>
__device__ __forceinline__ void pair_f_body(const SysDev *__restrict__ sys, int energy, int pgrid,
                                            int skin, int bxi) {
  const SysDev &V = sys[blockIdx.z];
  if (skin && bxi >= pgrid) {
    skin_two_blocks(V, 2 * (bxi - pgrid));
    return;
  }
  const int blk = xcd_block(bxi, pgrid);
  const int nb = V.nblk_pair;
  if (blk >= nb || V.pair_pos64 != (POS64 ? 1 : 0)) return;
  const float4 *__restrict__ pos = V.pos_f;
  const int np = V.np;
  const int *__restrict__ nn = V.nn;
  const unsigned *__restrict__ nbr = reinterpret_cast<const unsigned *>((const int *)V.nbr);
  const TableDev t = V.tab;
  const int semantics = V.nlsem;
  extern __shared__ __align__(16) unsigned char pair_lds[];
  __shared__ PairRecF rec_s[MFE_MAX_PAIRS];
  __shared__ int pidx_s[MFE_MAX_TYPES * MFE_MAX_TYPES];
  __shared__ float4 off_s[125];
  __shared__ double wacc[kPairBlock / 64][MFE_MAX_PAIRS + 1];
  const int P = t.nptpt, nbin = t.nbin, nzl = t.nzl, npt = t.npt;
  const size_t bb = pair_bin_bytes(P, nbin);
  unsigned short *bin_s = reinterpret_cast<unsigned short *>(pair_lds);
  float *zl_s = reinterpret_cast<float *>(pair_lds + bb);
  float *cf_s = reinterpret_cast<float *>(pair_lds + bb + pair_zl_bytes(nzl));
  const bool lds_zl = CF || t.lds_mode >= 1;
  stage_image(pair_lds, t,
              bb + (lds_zl ? pair_zl_bytes(nzl) : 0) +
                  (CF ? (size_t)nzl * kCoefStride * sizeof(float) : 0));
  for (int k = threadIdx.x; k < P; k += blockDim.x) rec_s[k] = t.rec_f[k];
  for (int k = threadIdx.x; k < npt * npt; k += blockDim.x) pidx_s[k] = t.pairidx[k];
  for (int k = threadIdx.x; k < 125; k += blockDim.x)
    off_s[k] = make_float4(V.cg.off[0][k % 5], V.cg.off[1][(k / 5) % 5], V.cg.off[2][k / 25], 0.f);
  const int l64 = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int k = l64; k <= P; k += 64) wacc[wv][k] = 0.0;
  __syncthreads();
  const float rc2 = (float)t.rcut2;
  const float L0 = V.cg.L[0], L1 = V.cg.L[1], L2 = V.cg.L[2];
  const float H0 = V.cg.L2[0], H1 = V.cg.L2[1], H2 = V.cg.L2[2];
  // lanes per particle (lsh their log2)
  const int LANES = V.pair_lanes, lsh = __builtin_ctz(LANES);
  const int lane = threadIdx.x & (LANES - 1);
  double ej[NT];
  double vir = 0.0;
  KahanF fxf, fyf, fzf;
  int ti = 0;
  unsigned long long ptp = 0;
  int err = 0;
  // the separation of a partner at relative position pj with code e
  auto sep = [&](float xi, float yi, float zi, float4 pj, unsigned e, float &dx, float &dy,
                 float &dz) {
    const float4 o4 = off_s[e >> kNbrCodeShift];
    dx = (xi - pj.x) + o4.x;
    dy = (yi - pj.y) + o4.y;
    dz = (zi - pj.z) + o4.z;
    // axes of one cell: the minimum image
    if (fabsf(dx) > H0) dx -= copysignf(L0, dx);
    if (fabsf(dy) > H1) dy -= copysignf(L1, dy);
    if (fabsf(dz) > H2) dz -= copysignf(L2, dz);
  };
  const PairTabF T{bin_s, lds_zl ? zl_s : (const float *)t.zlow_f,
                   CF ? cf_s : (const float *)t.coef_f, rec_s, nbin, semantics, rc2};
  // one list entry: a partner of type tj at separation (dx, dy, dz)
  auto eval = [&](float dx, float dy, float dz, int tj) {
    const int p = (int)((ptp >> (8 * tj)) & 0xffu);
    float fs, r2;
    double usum;
    if (!pair_eval_f<KN>(V, T, dx, dy, dz, p, energy, fs, usum, r2, err)) return;
    fxf.add(fs * dx);
    fyf.add(fs * dy);
    fzf.add(fs * dz);
    if (energy) {
#pragma unroll
      for (int k2 = 0; k2 < NT; ++k2) ej[k2] += (k2 == tj) ? 0.5 * usum : 0.0;
      vir -= 0.5 * (double)(fs * r2);
    }
  };
  const int kChunk = kPairBlock >> lsh;
  const int nch = (np + kChunk - 1) / kChunk;
  const int ch0 = (int)((long long)blk * nch / nb), ch1 = (int)((long long)(blk + 1) * nch / nb);
  const int maxrow = V.maxnn - 1;
  for (int ch = ch0; ch < ch1; ++ch) {
    const int i = ch * kChunk + (threadIdx.x >> lsh);
#pragma unroll
    for (int k = 0; k < NT; ++k) ej[k] = 0.0;
    fxf = KahanF();
    fyf = KahanF();
    fzf = KahanF();
    ti = 0;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    if (i < np) {
      // the particle, its list length and its first entries issued together
      const float4 pi = POS64 ? make_float4(0.f, 0.f, 0.f, __int_as_float(V.type_s[i])) : pos[i];
      const double xi = POS64 ? V.ro_s[3 * i] : 0.0, yi = POS64 ? V.ro_s[3 * i + 1] : 0.0,
                   zi = POS64 ? V.ro_s[3 * i + 2] : 0.0;
      const int n = nn[i];
      unsigned es[kPairBatch];
#pragma unroll
      for (int g = 0; g < kPairBatch; ++g)
        es[g] = nbr[(size_t)min(lane + g * LANES, maxrow) * np + i];
      ti = __float_as_int(pi.w);
      ptp = 0;
      for (int u = 0; u < npt; ++u)
        ptp |= (unsigned long long)pidx_s[ti * npt + u] << (8 * u);
      for (int k0 = lane; k0 < n; k0 += kPairBatch * LANES) {
        if (k0 != lane) {
#pragma unroll
          for (int g = 0; g < kPairBatch; ++g)
            es[g] = nbr[(size_t)min(k0 + g * LANES, maxrow) * np + i];
        }
        if constexpr (POS64) {
          double xs[kPairBatch], ys[kPairBatch], zs[kPairBatch];
          int ts[kPairBatch];
#pragma unroll
          for (int g = 0; g < kPairBatch; ++g) {
            const int j = k0 + g * LANES < n ? (int)(es[g] & kNbrIdxMask) : i;
            xs[g] = V.ro_s[3 * j];
            ys[g] = V.ro_s[3 * j + 1];
            zs[g] = V.ro_s[3 * j + 2];
            ts[g] = V.type_s[j];
          }
#pragma unroll
          for (int g = 0; g < kPairBatch; ++g) {
            if (k0 + g * LANES < n) {
              double ddx = xi - xs[g], ddy = yi - ys[g], ddz = zi - zs[g];
              pbcr2(ddx, ddy, ddz, V.box);
              eval((float)ddx, (float)ddy, (float)ddz, ts[g]);
            }
          }
        } else {
          float4 ps[kPairBatch];
#pragma unroll
          for (int g = 0; g < kPairBatch; ++g) {
            // entries past the list end read the particle itself
            const int j = k0 + g * LANES < n ? (int)(es[g] & kNbrIdxMask) : i;
            ps[g] = pos[j];
          }
#pragma unroll
          for (int g = 0; g < kPairBatch; ++g) {
            if (k0 + g * LANES < n) {
              float dx, dy, dz;
              sep(pi.x, pi.y, pi.z, ps[g], es[g], dx, dy, dz);
              eval(dx, dy, dz, __float_as_int(ps[g].w));
            }
          }
        }
      }
      fx = fxf.value();
      fy = fyf.value();
      fz = fzf.value();
    }
    fx = lane_sum(fx, LANES);
    fy = lane_sum(fy, LANES);
    fz = lane_sum(fz, LANES);
    if (i < np && lane == 0) {
      const int io = V.c_sorted[i];
      V.force[3 * io] = fx;
      V.force[3 * io + 1] = fy;
      V.force[3 * io + 2] = fz;
    }
    if (energy) {
      // pair-type energies of this chunk: wave_sum in each
      // wavefront, added to the wavefront's own LDS row
      for (int k = 0; k < P; ++k) {
        double v = 0.0;
        if (i < np) {
#pragma unroll
          for (int u = 0; u < NT; ++u)
            if (u < npt && (int)((ptp >> (8 * u)) & 0xffu) == k) v += ej[u];
        }
        v = wave_sum(v);
        if (l64 == 0) wacc[wv][k] += v;
      }
    }
  }
  if (err) atomicOr(&V.flags[0], err);
  if (energy) {
    const double v = wave_sum(vir);
    if (l64 == 0) wacc[wv][P] = v;
    __syncthreads();
    double *out = V.part + V.off_pair + blk;
    for (int k = threadIdx.x; k <= P; k += blockDim.x) {
      double s2 = wacc[0][k];
      for (int w = 1; w < (int)(blockDim.x >> 6); ++w) s2 += wacc[w][k];
      out[(size_t)k * nb] = s2;
    }
  }
}

template <int NT, bool CF, bool KN, bool POS64>
__global__ void __launch_bounds__(kPairBlock) __attribute__((amdgpu_waves_per_eu(KN || POS64 ? 4 : 5)))
k_pair_f(const SysDev *__restrict__ sys, int energy, int pgrid, int skin) {
  pair_f_body<NT, CF, KN, POS64>(sys, energy, pgrid, skin, (int)blockIdx.x);
}

// ------------------------------------------------------------------ SPME
// Brick of every particle and its slot within the brick, both indexed by
// the particle's place t in the cell order, from the cell-ordered positions
// (current whenever SPME runs: k_move or the pair launch refreshes them).
// A block takes 1024 consecutive particles of the cell order -- a compact
// piece of the box, spanning a few dozen bricks -- counts them in an LDS
// histogram and
// then adds each non-empty bin to the global count with one atomic, so
// global atomics scale with the bricks a block touches, not with its
// particles.  Meshes with more bricks than the histogram holds fall back to
// one global atomic per particle.
constexpr int kCountThreads = 1024;
constexpr int kCountBins = 8192;
// Up to this many bricks every k_spme_scatter block scans the counts itself
// (no done counter and no last-block scan in k_spme_count), k_spread clears
// each brick's count after the scatter has used it, and a binning that is
// not followed by spreading clears them with k_spme_clear.
constexpr int kScatterScan = 2048;
static_assert(kScatterScan % kBlock == 0, "the scatter's scan gives each thread whole runs");

__global__ void __launch_bounds__(kCountThreads) k_spme_count(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  const int np = V.np;
  const int nblk = (np + kCountThreads - 1) / kCountThreads;
  if ((int)blockIdx.x >= nblk) return;
  const double *__restrict__ ro_s = V.ro_s;
  const SpmeGeom g = V.sg;
  int *bcount = V.b_count, *bid = V.b_id, *bslot = V.b_slot;
  __shared__ int hist[kCountBins];
  const int t = blockIdx.x * kCountThreads + threadIdx.x;
  const bool act = t < np;
  int id = 0;
  if (act) {
    int mm[3];
    double fr[3];
    mesh_coords(ro_s + 3 * t, g, mm, fr);
    id = fdiv(mm[0], g.fB[0]) + g.nb[0] * (fdiv(mm[1], g.fB[1]) + g.nb[1] * fdiv(mm[2], g.fB[2]));
  }
  if (V.nbricks > kCountBins) {
    if (act) {
      bid[t] = id;
      bslot[t] = atomicAdd(&bcount[id], 1);
    }
  } else {
    for (int k = threadIdx.x; k < V.nbricks; k += kCountThreads) hist[k] = 0;
    __syncthreads();
    const int rank = act ? atomicAdd(&hist[id], 1) : 0;
    __syncthreads();
    // one global atomic per non-empty bin; its old value is the bin's base
    for (int k = threadIdx.x; k < V.nbricks; k += kCountThreads) {
      const int c = hist[k];
      if (c) hist[k] = atomicAdd(&bcount[k], c);
    }
    __syncthreads();
    if (act) {
      bid[t] = id;
      bslot[t] = hist[id] + rank;
    }
  }
  if (V.nbricks <= kScatterScan) return;
  // The last block to finish scans the counts into b_start and clears them
  // (no separate scan launch).  Every count atomic of this block has
  // returned -- its value was used -- before the block barrier, so the
  // done counter is incremented after them; the last block takes an
  // acquire fence before reading the counts.  Nothing waits.
  __shared__ int last;
  __syncthreads();
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(V.b_done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           nblk - 1;
  __syncthreads();
  if (!last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  ph_scan(bcount, V.b_start, V.nbricks);
  if (threadIdx.x == 0) __hip_atomic_store(V.b_done, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// particle records in brick order: fraction (x, y, z) and charge, plus the
// packed meshmax (10 bits per axis) and the particle index; one thread per
// place t of the cell order
// Exclusive scan of the brick counts into LDS (st[k], st[n] = the total),
// by one block of kBlock threads, each taking a contiguous run of bricks.
__device__ __forceinline__ void block_scan_counts(const int *__restrict__ count, int *st,
                                                  int n) {
  constexpr int kPer = kScatterScan / kBlock;
  __shared__ int wsum[kBlock / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lo = threadIdx.x * kPer;
  int v[kPer];
  int x = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    v[u] = lo + u < n ? count[lo + u] : 0;
    x += v[u];
  }
  int inc = x;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(inc, o, 64);
    if (lane >= o) inc += y;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  int run = inc - x, tot = 0;
  for (int w = 0; w < kBlock / 64; ++w) {
    run += w < wave ? wsum[w] : 0;
    tot += wsum[w];
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    if (lo + u < n) st[lo + u] = run;
    run += v[u];
  }
  if (threadIdx.x == 0) st[n] = tot;
  __syncthreads();
}

template <typename R>
__global__ void __launch_bounds__(kBlock) k_spme_scatter(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  const double *__restrict__ ro_s = V.ro_s;
  const double *__restrict__ q = V.q;
  const SpmeGeom g = V.sg;
  const int *bid = V.b_id, *bslot = V.b_slot, *bstart = V.b_start;
  R *frac = (R *)V.rec_frac;
  int2 *meta = V.rec_meta;
  const int nbk = V.nbricks;
  // the particle's own loads first, so that they are in flight during the
  // scan of the counts
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const bool act = t < V.np;
  int i = 0, b = 0, slot = 0, mm[3] = {0, 0, 0};
  double fr[3] = {0.0, 0.0, 0.0}, qi = 0.0;
  if (act) {
    i = V.c_sorted[t];
    b = bid[t];
    slot = bslot[t];
    mesh_coords(ro_s + 3 * t, g, mm, fr);
    qi = q[i];
  }
  __shared__ int st[kScatterScan + 1];
  if (nbk <= kScatterScan) {
    // the brick starts from the counts k_spme_count left (every block the
    // same scan); block 0 stores them for the spreading and the gather
    block_scan_counts(V.b_count, st, nbk);
    if (st[nbk] != V.np) {
      if (threadIdx.x == 0) atomicOr(&V.flags[0], ERR_BIN);
      return;
    }
    if (blockIdx.x == 0)
      for (int k = threadIdx.x; k <= nbk; k += blockDim.x) V.b_start[k] = st[k];
  }
  if (!act) return;
  const int pos = (nbk <= kScatterScan ? st[b] : bstart[b]) + slot;
  frac[4 * pos] = (R)fr[0];
  frac[4 * pos + 1] = (R)fr[1];
  frac[4 * pos + 2] = (R)fr[2];
  frac[4 * pos + 3] = (R)qi;
  meta[pos] = make_int2(mm[0] | (mm[1] << 10) | (mm[2] << 20), i);
}

// the brick counts cleared after a binning that no spreading follows
__global__ void k_spme_clear(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (V.nbricks <= kScatterScan && k < V.nbricks) V.b_count[k] = 0;
}

// Spreading, each particle once and no global atomics: one block per brick
// takes the brick's own particles and adds their whole stencil -- points
// m, m-1, ..., m-order+1 along each axis from meshmax m
// (Src/energy.F90:1232-1244) -- into an LDS tile of the brick extended by
// order-1 points on the low side of each axis, then writes the tile to a
// scratch array.  The forward x FFT reads each mesh point as its own
// brick's tile value plus the low-side halos of the next bricks (at most 8
// tiles) in a fixed order (spread_point in mfe_fft_rows.hip).  Work is handed
// out as (particle, stencil plane) items, order planes per particle; each
// item computes the particle's B-splines in registers (no staging, no
// barrier between particles) and loads the record of its next item before
// its own adds, so the load latency hides behind them.
// 1024 threads share one brick's tile; without other LDS two blocks fit a
// CU at 16-point bricks of order <= 6 (at order 7 a tile is 83 KB).
constexpr int kSpreadThreads = 1024;

template <typename R, int ORDER>
__global__ void __launch_bounds__(kSpreadThreads) k_spread(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  if ((int)blockIdx.x >= V.nbricks) return;
  // the scatter has used this brick's count: cleared for the next binning
  if (V.nbricks <= kScatterScan && threadIdx.x == 0) V.b_count[blockIdx.x] = 0;
  const R *__restrict__ frac = (const R *)V.rec_frac;
  const int2 *__restrict__ meta = V.rec_meta;
  const int *__restrict__ bstart = V.b_start;
  const SpmeGeom g = V.sg;
  typedef typename SpreadAcc<R>::T Acc;
  extern __shared__ char smem[];
  Acc *tile = reinterpret_cast<Acc *>(smem);
  const int bx = blockIdx.x % g.nb[0];
  const int by = (blockIdx.x / g.nb[0]) % g.nb[1];
  const int bz = blockIdx.x / (g.nb[0] * g.nb[1]);
  // meshmax - brick origin + order-1: extended-tile coordinates
  const int o0 = bx * g.B[0] - (ORDER - 1), o1 = by * g.B[1] - (ORDER - 1),
            o2 = bz * g.B[2] - (ORDER - 1);
  const int E0 = g.B[0] + ORDER - 1, E1 = g.B[1] + ORDER - 1, E2 = g.B[2] + ORDER - 1;
  const int ntile = E0 * E1 * E2, plane = g.plane;
  const int first = bstart[blockIdx.x], items = (bstart[blockIdx.x + 1] - first) * ORDER;
  int r = threadIdx.x;
  Rec4<R> f{};
  int code = 0;
  if (r < items) {
    const int rec = first + r / ORDER;
    f = load_rec(frac + 4 * rec);
    code = meta[rec].x;
  }
  for (int k = threadIdx.x; k < plane * E2; k += kSpreadThreads) tile[k] = Acc(0);
  __syncthreads();
  for (; r < items; r += kSpreadThreads) {
    const int rn = r + kSpreadThreads;
    Rec4<R> fn = f;
    int cn = code;
    if (rn < items) {
      const int rec = first + rn / ORDER;
      fn = load_rec(frac + 4 * rec);
      cn = meta[rec].x;
    }
    const int iz = r % ORDER;
    R wx[ORDER], wy[ORDER], wz[ORDER];
    bspline<R, ORDER>(f.x, wx, nullptr);
    bspline<R, ORDER>(f.y, wy, nullptr);
    bspline<R, ORDER>(f.z, wz, nullptr);
    R wzi = wz[0];
#pragma unroll
    for (int k = 1; k < ORDER; ++k)
      if (iz == k) wzi = wz[k];
    const int lx = (code & 1023) - o0;
    const int ly = ((code >> 10) & 1023) - o1;
    const int lz = ((code >> 20) & 1023) - o2;
    constexpr double kScale = kSplineScale<ORDER, 0>;
    const R qz = SpreadAcc<R>::pre(f.q, kScale) * wzi;
    Acc *zp = tile + (lz - iz) * plane;
#pragma unroll
    for (int jy = 0; jy < ORDER; ++jy) {
      const R qyz = qz * wy[jy];
      Acc *row = zp + (ly - jy) * E0 + lx;
#pragma unroll
      for (int j = 0; j < ORDER; ++j) SpreadAcc<R>::add(&row[-j], qyz * wx[j], kScale);
    }
    f = fn;
    code = cn;
  }
  __syncthreads();
  R *__restrict__ out = (R *)V.spread_tiles + (size_t)blockIdx.x * ntile;
  store_tile<R>(g, E0, E1, E2, tile, out);
}

// per-lane stencil sums: compensated FP32 on the mixed path, plain FP64
template <typename R>
struct Acc3;
template <>
struct Acc3<float> {
  KahanF a[3];
  __device__ __forceinline__ void add(int m, float v) { a[m].add(v); }
  __device__ __forceinline__ double get(int m) const { return a[m].value(); }
};
template <>
struct Acc3<double> {
  double a[3] = {0.0, 0.0, 0.0};
  __device__ __forceinline__ void add(int m, double v) { a[m] += v; }
  __device__ __forceinline__ double get(int m) const { return a[m]; }
};

// CalcProp (Src/energy.F90:1259-1285): esum over the order^3 stencil of the
// convolved mesh; force -= q * esum * dkdr * EpsiFourPi.  One block per
// brick stages the mesh the brick's particles touch -- points
// [o - (order-1), o + B) per axis -- in LDS; each particle is taken by a
// few lanes, each computing the particle's B-splines and derivatives in
// registers and summing some of its stencil planes (FP32 with compensated
// row sums on the mixed path); the lanes are combined by lane exchanges in
// FP64 in a fixed order.  No barrier between particles: each lane loads
// its next particle's record while it sums the current one.
constexpr int kGatherLanes = 512;

// the finalize phase split in its loads and its arithmetic and stores, so
// a kernel can issue the loads early; and the reductions (defined below)
struct FinState {
  double aold[3], v[3], q, mi;
};
__device__ __forceinline__ void fin_load(const SysDev &V, int i, int mode, FinState &st);
__device__ __forceinline__ void fin_apply(const SysDev &V, int i, const double f[3],
                                         const FinState &st, int mode, double dt,
                                         const double es[3]);
__device__ __forceinline__ void ph_reduce(const SysDev &V, int energy, int skin, int bd);

// MODE: GM_FORCE adds the force; GM_POT also writes efp * phi_i (the
// reciprocal potential, dE_rec/dq_i); GM_FIELD also writes the reciprocal
// field -efp grad phi_i (the force per unit charge); GM_POTONLY writes
// efp * phi_i of the mesh and leaves the forces alone (the backward pass
// of the force-matching loss interpolates its own convolved mesh).
// FIN: also the finalize phase of each particle (its owner lane, after the
// force) and, in block nbricks, the reductions, whose inputs come from
// earlier launches.
// GM_FORCE_REC writes the reciprocal force alone into force_rec (the
// finalize adds it to the pair force).  The body takes its block index bxi.
template <typename R, int ORDER, int MODE, bool FIN>
__device__ __forceinline__ void gather_body(const SysDev *__restrict__ sys, FinArgs fa, int bxi) {
  const SysDev &V = sys[blockIdx.z];
  if (FIN && bxi == V.nbricks) {
    ph_reduce(V, fa.energy, fa.skin, fa.bd);
    return;
  }
  if (bxi >= V.nbricks) return;
  const R *__restrict__ frac = (const R *)V.rec_frac;
  const int2 *__restrict__ meta = V.rec_meta;
  const int *__restrict__ bstart = V.b_start;
  const SpmeGeom g = V.sg;
  const R *__restrict__ mesh = (const R *)V.mesh_r;
  const double efp = V.efp;
  double *__restrict__ force = V.force;
  extern __shared__ char smem[];
  R *tile = reinterpret_cast<R *>(smem);
  const int bx = bxi % g.nb[0];
  const int by = (bxi / g.nb[0]) % g.nb[1];
  const int bz = bxi / (g.nb[0] * g.nb[1]);
  const int o0 = bx * g.B[0], o1 = by * g.B[1], o2 = bz * g.B[2];
  const int E0 = g.B[0] + ORDER - 1, E1 = g.B[1] + ORDER - 1, E2 = g.B[2] + ORDER - 1;
  const int nstage = E0 * E1 * E2;
  // two lanes share a particle, lane l summing stencil planes l, l + 2, ...
  // (none idle at even orders), each with the particle's splines: FP64, 200k
  // ions, order 6, 28.3 us with two lanes, 30.1 with four, 34.9 with eight
  constexpr int GL = 2;
  constexpr int kGStep = kGatherLanes / GL;
  constexpr int kPlanes = (ORDER + GL - 1) / GL;
  const int first = bstart[bxi], n = bstart[bxi + 1] - first;
  const int l = threadIdx.x % GL;
  int p = threadIdx.x / GL;
  // the first particle's record is in flight during the staging
  Rec4<R> f{};
  int2 md = make_int2(0, 0);
  if (p < n) {
    f = load_rec(frac + 4 * (first + p));
    md = meta[first + p];
  }
  // staged in batches of kU loads per lane, so the loads of a batch are in
  // flight together (one batch for bricks of 16 and order <= 8)
  constexpr int kU = 24;
  for (int k0 = threadIdx.x; k0 < nstage; k0 += kU * blockDim.x) {
    R val[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int k = k0 + u * blockDim.x;
      val[u] = R(0);
      if (k < nstage) {
        // exact: the tile fits LDS (k < 40960) and its edges are short
        const int k01 = fdiv(k, g.fE[0]);
        const int ze = fdiv(k01, g.fE[1]);
        const int xe = k - k01 * E0, ye = k01 - ze * E1;
        // region coordinates lie in [o - (order-1), o + B) with o + B <= s
        // and s >= order: one wrap, below zero only
        int x = o0 - (ORDER - 1) + xe, y = o1 - (ORDER - 1) + ye, z = o2 - (ORDER - 1) + ze;
        x += x < 0 ? g.s[0] : 0;
        y += y < 0 ? g.s[1] : 0;
        z += z < 0 ? g.s[2] : 0;
        // meshes up to 1024 per axis: the offset fits 32 bits
        val[u] = mesh[(unsigned)((z * g.s[1] + y) * g.s[0] + x)];
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int k = k0 + u * blockDim.x;
      if (k < nstage) tile[k] = val[u];
    }
  }
  __syncthreads();
  for (; p < n; p += kGStep) {
    // the force this particle's owner lane updates and the next particle's
    // record, loaded now so the loads overlap the stencil sums
    const bool owner = l == 0;
    const int idx = md.y;
    double f0 = 0.0, f1 = 0.0, f2 = 0.0;
    FinState st;
    if (owner && MODE != GM_POTONLY && MODE != GM_FORCE_REC) {
      f0 = force[3 * idx];
      f1 = force[3 * idx + 1];
      f2 = force[3 * idx + 2];
      if (FIN) fin_load(V, idx, fa.mode, st);
    }
    const int pn = p + kGStep;
    Rec4<R> fn = f;
    int2 mn = md;
    if (pn < n) {
      fn = load_rec(frac + 4 * (first + pn));
      mn = meta[first + pn];
    }
    R v[3][ORDER], d[3][ORDER];
    bspline<R, ORDER>(f.x, v[0], d[0]);
    bspline<R, ORDER>(f.y, v[1], d[1]);
    bspline<R, ORDER>(f.z, v[2], d[2]);
    // brick-local coordinates inside the staged region
    const int lx = (md.x & 1023) - o0 + ORDER - 1;
    const int ly = ((md.x >> 10) & 1023) - o1 + ORDER - 1;
    const int lz = ((md.x >> 20) & 1023) - o2 + ORDER - 1;
    Acc3<R> acc;
    double pacc = 0.0;
#pragma unroll
    for (int kz = 0; kz < kPlanes; ++kz) {
      const int iz = l + GL * kz;
      if (iz >= ORDER) break;
      // weights of plane iz, selected without indexing registers
      R vz = v[2][0], dz = d[2][0];
#pragma unroll
      for (int k = 1; k < ORDER; ++k)
        if (iz == k) {
          vz = v[2][k];
          dz = d[2][k];
        }
      const R *plane = tile + (size_t)(lz - iz) * E1 * E0;
#pragma unroll
      for (int iy = 0; iy < ORDER; ++iy) {
        const R *row = plane + (ly - iy) * E0;
        R sx = R(0), sdx = R(0);
#pragma unroll
        for (int ix = 0; ix < ORDER; ++ix) {
          const R qv = row[lx - ix];
          sx += v[0][ix] * qv;
          sdx += d[0][ix] * qv;
        }
        if (MODE != GM_POTONLY) {
          acc.add(0, sdx * (v[1][iy] * vz));
          acc.add(1, sx * (d[1][iy] * vz));
          acc.add(2, sx * (v[1][iy] * dz));
        }
        if (MODE == GM_POT || MODE == GM_POTONLY) pacc += (double)sx * (double)(v[1][iy] * vz);
      }
    }
    double ex = acc.get(0) * kSplineScale<ORDER, 1>;
    double ey = acc.get(1) * kSplineScale<ORDER, 1>;
    double ez = acc.get(2) * kSplineScale<ORDER, 1>;
    double ep = pacc * kSplineScale<ORDER, 0>;
    // both lanes of a particle are in or out of the loop: the lane pair within
    // a quad, by DPP
    ex += quad_swap<kXor1>(ex);
    ey += quad_swap<kXor1>(ey);
    ez += quad_swap<kXor1>(ez);
    if (MODE == GM_POT || MODE == GM_POTONLY) ep += quad_swap<kXor1>(ep);
    if (owner) {
      // q fld rounded before the pair force is added (no contraction): the
      // same sum as the finalize forms from force and force_rec
#pragma clang fp contract(off)
      const double qd = (double)f.q;
      const double fld[3] = {-ex * g.dkdr[0] * efp, -ey * g.dkdr[1] * efp,
                             -ez * g.dkdr[2] * efp};
      const double fr[3] = {qd * fld[0], qd * fld[1], qd * fld[2]};
      const double ft[3] = {f0 + fr[0], f1 + fr[1], f2 + fr[2]};
      if (MODE == GM_FORCE_REC) {
        V.force_rec[3 * idx] = fr[0];
        V.force_rec[3 * idx + 1] = fr[1];
        V.force_rec[3 * idx + 2] = fr[2];
      } else if (MODE != GM_POTONLY) {
        force[3 * idx] = ft[0];
        force[3 * idx + 1] = ft[1];
        force[3 * idx + 2] = ft[2];
      }
      // dE_rec/dq = efp * sum_stencil theta * (G * Q) (the convolved mesh)
      if (MODE == GM_POT || MODE == GM_POTONLY) V.phi_rec[idx] = efp * ep;
      if (MODE == GM_FIELD) {
        V.fm_fld[3 * idx] = fld[0];
        V.fm_fld[3 * idx + 1] = fld[1];
        V.fm_fld[3 * idx + 2] = fld[2];
      }
      if (FIN) {
        const double es[3] = {0.0, 0.0, 0.0};
        fin_apply(V, idx, ft, st, fa.mode, fa.dt, es);
      }
    }
    f = fn;
    md = mn;
  }
}

// two blocks per CU on the FP64 path up to the order whose tile and
// registers allow it
template <typename R, int ORDER, int MODE, bool FIN>
__global__ void __launch_bounds__(kGatherLanes, sizeof(R) == 8 && ORDER <= 6 ? 4 : 1) k_gather(const SysDev *__restrict__ sys,
                                                         FinArgs fa) {
  gather_body<R, ORDER, MODE, FIN>(sys, fa, (int)blockIdx.x);
}

// The mixed path's pair forces and the reciprocal forces in one launch:
// blocks [0, npb) run k_pair_f's blocks (pair partition, then the skin
// blocks; npb a multiple of eight, so the gather blocks keep their
// placement on the XCDs), block npb + b the gather of brick b, which
// writes force_rec.  The two share no data; the pair waves, a lane per
// particle at low density, fill what the gather leaves idle.
static_assert(kPairBlock == kGatherLanes, "the fused launch runs both bodies in one block size");

template <int NT, int ORDER>
__global__ void __launch_bounds__(kPairBlock) __attribute__((amdgpu_waves_per_eu(5)))
k_pair_gather(const SysDev *__restrict__ sys, int energy, int pgrid, int skin, int npb) {
  const int b = (int)blockIdx.x;
  if (b < npb) {
    pair_f_body<NT, true, false, false>(sys, energy, pgrid, skin, b);
    return;
  }
  gather_body<float, ORDER, GM_FORCE_REC, false>(sys, FinArgs{0, 0, 0, 0, 0.0}, b - npb);
}

// an accepted trial move written into a copy of the positions
__global__ void __launch_bounds__(256) k_mc_place(int natm, const int *__restrict__ ia,
                                                  const double *__restrict__ rtm,
                                                  double *__restrict__ ro_stage) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= natm) return;
  const int i = ia[a];
  for (int m = 0; m < 3; ++m) ro_stage[3 * i + m] = rtm[3 * a + m];
}

// ------------------------------------------------------- MC trial move
// DUTwoBodyEwaldRecSPM (Src/denergy.F90:1413-1495) takes the reciprocal
// energy of the trial mesh -- the current one less the moved particles' old
// stencils plus their new ones (DUMakeGQMesh, :1432-1460) -- minus the
// current energy.  The transform is linear, so the trial spectrum is the
// current one, F, plus D(k), the transform of the stencil difference: per
// moved particle q (prod_m c'_m(k_m) - prod_m c_m(k_m)), each factor a
// one-dimensional sum over the particle's stencil along axis m, c(k) =
// sum_j w_j exp(-2 pi i k (p - j) / s) (weight w_j at mesh point p - j from
// meshmax p), the forward transform's sign.  The energy change is then
// sum_k wt(k) G(k) (2 Re(conj(F) D) + |D|^2) with the convolution pass's
// weights wt and Green function G: one pass over the kept spectrum, no
// transform per trial, and no difference of two large energies.  Weights
// and charge are rounded as the spreading rounds them (the fraction and q
// to R, the B-spline in R), so D takes out the stencil the mesh holds up
// to the rounding of the spreading's products.  One replica, fewer than
// 2^31 points, kx fastest.
//
// A block takes tiles of 256 P consecutive spectrum points (P per thread,
// their D in registers) and holds the factors that the tile needs in LDS, of
// up to `chunk` moved particles at a time: x factors c(kx) with the charge
// folded in, and per mesh row (ky, kz) the product of its y and z factors,
// each for the current (n = 0) and the trial (1) position (McLds).  apply ==
// false writes the block's part of the energy change to part[block] (the
// host adds the parts in block order); apply == true adds D to F.
constexpr int kMcPoints = 4;
// mesh rows that a tile can touch
__host__ __device__ inline int mc_rows(int hx, int P) { return (256 * P - 1) / hx + 2; }

__device__ __forceinline__ int mc_ia(const McMove &mv, int a) {
  return mv.natm <= kMcArg ? mv.ia_v[a] : mv.ia[a];
}
__device__ __forceinline__ double mc_rtm(const McMove &mv, int k) {
  return mv.natm <= kMcArg ? mv.rtm_v[k] : mv.rtm[k];
}

// fill(a, trial, x, row): the factor of moved particle a at wavenumber x >= 0
// of the x axis, or (x < 0) the product of its factors along mesh row `row`
template <int P, typename Fill>
__device__ __forceinline__ void mc_pass(const SysDev &V, int natm, int chunk, double2 *lds,
                                        double2 *__restrict__ F, bool apply,
                                        double *__restrict__ part, int blk, int nblk,
                                        Fill fill) {
  const SpmeAxes &ax = V.ax;
  const int s0 = V.sg.s[0], s1 = V.sg.s[1], s2 = V.sg.s[2], hx = V.hx;
  const unsigned n = (unsigned)hx * s1 * s2;
  const int rows = mc_rows(hx, P);
  double2 *fx = lds;                     // [2 chunk][hx]
  double2 *fr = fx + 2 * chunk * hx;     // [2 chunk][rows]
  double acc = 0.0;
  for (unsigned e0 = (unsigned)blk * (256 * P); e0 < n; e0 += (unsigned)nblk * (256 * P)) {
    const unsigned r0 = e0 / (unsigned)hx;
    const unsigned r1 = (min(e0 + 256 * P, n) - 1) / (unsigned)hx;
    const int nr = (int)(r1 - r0) + 1, ne = hx + nr;
    double2 v[P];
    double dr[P], di[P];
#pragma unroll
    for (int u = 0; u < P; ++u) {
      v[u] = F[min(e0 + u * 256 + threadIdx.x, n - 1)];
      dr[u] = 0.0;
      di[u] = 0.0;
    }
    for (int a0 = 0; a0 < natm; a0 += chunk) {
      const int na = min(chunk, natm - a0);
      // the roots are written, the last chunk's factors read
      __syncthreads();
      for (int t = threadIdx.x; t < 2 * na * ne; t += blockDim.x) {
        const int row = t / ne, k = t - row * ne;
        const double2 c = fill(a0 + (row >> 1), row & 1, k < hx ? k : -1,
                               r0 + (unsigned)max(k - hx, 0));
        (k < hx ? fx[row * hx + k] : fr[row * rows + k - hx]) = c;
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < P; ++u) {
        const unsigned e = min(e0 + u * 256 + threadIdx.x, n - 1), r = e / (unsigned)hx;
        const int kx = (int)(e - r * (unsigned)hx), kr = (int)(r - r0);
        for (int a = 0; a < 2 * na; a += 2) {
          const double2 x0 = fx[a * hx + kx], y0 = fr[a * rows + kr];
          const double2 x1 = fx[(a + 1) * hx + kx], y1 = fr[(a + 1) * rows + kr];
          dr[u] += (x1.x * y1.x - x1.y * y1.y) - (x0.x * y0.x - x0.y * y0.y);
          di[u] += (x1.x * y1.y + x1.y * y1.x) - (x0.x * y0.y + x0.y * y0.x);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < P; ++u) {
      const unsigned e = e0 + u * 256 + threadIdx.x;
      if (e >= n) continue;
      if (apply) {
        F[e] = make_double2(v[u].x + dr[u], v[u].y + di[u]);
        continue;
      }
      const unsigned r = e / (unsigned)hx, kzu = r / (unsigned)s1;
      const int kx = (int)(e - r * (unsigned)hx), ky = (int)(r - kzu * (unsigned)s1);
      const int ny = min(ky, s1 - ky), nz = min((int)kzu, s2 - (int)kzu);
      const double m2 = ax.kk[0][kx] + ax.kk[1][ny] + ax.kk[2][nz];
      if (m2 > 0.0) {
        const double mf = ax.fac0 * ax.g[0][kx] * ax.g[1][ny] * ax.g[2][nz] / m2;
        const double wt = (kx == 0 || 2 * kx == s0) ? 0.5 : 1.0;
        acc += wt * mf * (2.0 * (v[u].x * dr[u] + v[u].y * di[u]) +
                          (dr[u] * dr[u] + di[u] * di[u]));
      }
    }
  }
  if (apply) return;
  __shared__ double sh[256 / 64];
  const double t = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blk] = t;
}

// the roots exp(-2 pi i p / s) of the three axes, by the whole block
__device__ __forceinline__ void mc_roots(const SpmeGeom &g, double2 *root) {
  const int s0 = g.s[0], s1 = g.s[1], s2 = g.s[2];
  for (int k = threadIdx.x; k < s0 + s1 + s2; k += blockDim.x) {
    const int m = k < s0 ? 0 : (k < s0 + s1 ? 1 : 2);
    const int ph = k - (m == 0 ? 0 : (m == 1 ? s0 : s0 + s1));
    double sn, cs;
    sincospi(-2.0 * (double)ph / (double)(m == 0 ? s0 : (m == 1 ? s1 : s2)), &sn, &cs);
    root[k] = make_double2(cs, sn);
  }
}

// the factor of an axis of sm points (its roots at rt) at wavenumber k:
// ORDER products with roots at exactly reduced phases
template <typename R, int ORDER>
__device__ __forceinline__ double2 mc_factor(double x, double dk, int sm, const double2 *rt,
                                             int k) {
  const double u = dk * x;
  const double f = floor(u);
  int pt = (int)f % sm;
  pt += pt < 0 ? sm : 0;
  R w[ORDER];
  bspline<R, ORDER>((R)(u - f), w, nullptr);
  // the phase k (pt - j) reduced to [0, s): pt, k < s < 2^15
  int ph = (int)(((unsigned)k * (unsigned)pt) % (unsigned)sm);
  double re = 0.0, im = 0.0;
#pragma unroll
  for (int j = 0; j < ORDER; ++j) {
    const double2 c = rt[ph];
    re += (double)w[j] * c.x;
    im += (double)w[j] * c.y;
    ph -= k;
    ph += ph < 0 ? sm : 0;
  }
  return make_double2(re, im);
}
__device__ __forceinline__ double2 mc_mul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a moved particle's charge with the splines' divisors
template <typename R, int ORDER>
__device__ __forceinline__ double mc_charge(const SysDev &V, int i) {
  return (double)(R)V.q[i] * kSplineScale<ORDER, 0>;
}

// Moves of fewer than kMcTable particles: each block forms the factors of its
// tile from the roots, so a trial costs one launch, bound by the latencies
// of roots, factors and spectrum: 8.6 us for one particle in an 80^3 mesh
// (the factors, the pass and the sum as kernels of their own took 7.5, 4.6
// and 3.8 us).  Two points per thread and twice the blocks measured 8.8 us.
// Block 0 of a trial keeps the current positions in `old`; the accept takes
// the change of the move just tried from those.
template <typename R, int ORDER>
__device__ __forceinline__ void mc_rec_body(const SysDev &V, const McMove &mv, int chunk,
                                            double2 *__restrict__ F, double *__restrict__ old,
                                            bool apply, double *__restrict__ part, int blk,
                                            int nblk) {
  extern __shared__ __align__(16) unsigned char mc_lds[];
  const SpmeGeom &g = V.sg;
  const int s0 = g.s[0], s1 = g.s[1], s2 = g.s[2];
  double2 *root = reinterpret_cast<double2 *>(mc_lds);        // [s0 + s1 + s2]
  mc_roots(g, root);
  if (!apply && blk == 0)
    for (int k = threadIdx.x; k < 3 * mv.natm; k += blockDim.x)
      old[k] = V.ro[3 * mc_ia(mv, k / 3) + k % 3];
  mc_pass<kMcPoints>(
      V, mv.natm, chunk, root + s0 + s1 + s2, F, apply, part, blk, nblk,
      [&](int a, int trial, int x, unsigned row) -> double2 {
        const int i = mc_ia(mv, a);
        double r[3];
#pragma unroll
        for (int m = 0; m < 3; ++m)
          r[m] = trial ? mc_rtm(mv, 3 * a + m) : (apply ? old[3 * a + m] : V.ro[3 * i + m]);
        if (x >= 0) {
          const double2 c = mc_factor<R, ORDER>(r[0], g.dkdr[0], s0, root, x);
          const double q = mc_charge<R, ORDER>(V, i);
          return make_double2(c.x * q, c.y * q);
        }
        const unsigned kz = row / (unsigned)s1;
        return mc_mul(mc_factor<R, ORDER>(r[1], g.dkdr[1], s1, root + s0,
                                          (int)(row - kz * (unsigned)s1)),
                      mc_factor<R, ORDER>(r[2], g.dkdr[2], s2, root + s0 + s1, (int)kz));
      });
}

template <typename R, int ORDER>
__global__ void __launch_bounds__(256) k_mc_rec(const SysDev *__restrict__ sys, const McMove mv,
                                                int chunk, double2 *spec, double *old,
                                                double *part) {
  mc_rec_body<R, ORDER>(sys[0], mv, chunk, spec, old, false, part, (int)blockIdx.x,
                        (int)gridDim.x);
}

// Moves of kMcTable particles and more: a launch of its own forms the factors
// of all moved particles, fac[(2 a + n) (s1 + s2 + s3) + axis offset + k], the
// charge in those of the x axis; the trial's pass and the accept's take them
// from there.  Formed in every block they are the time of a larger move: 64
// particles, order 6, meshes of 80^3 97 us (66 from the table), of 48^3 96
// (42); 500 particles 613 (352) and 612 (175).  The table costs a launch, so
// for one or two particles the trial is up to 0.7 us faster without it
// (128^3).  Small meshes take one point per thread, so that their tiles
// occupy the chip: 24^3, 64 particles 68 us with four, 39 with one.
constexpr int kMcTable = 3;
template <typename R, int ORDER>
__global__ void __launch_bounds__(256) k_mc_fac(const SysDev *__restrict__ sys, const McMove mv,
                                                double2 *__restrict__ fac) {
  extern __shared__ __align__(16) unsigned char mc_lds[];
  const SysDev &V = sys[0];
  const SpmeGeom &g = V.sg;
  const int s0 = g.s[0], s1 = g.s[1], s2 = g.s[2], ns = s0 + s1 + s2;
  double2 *root = reinterpret_cast<double2 *>(mc_lds);
  mc_roots(g, root);
  __syncthreads();
  const long long total = 2ll * mv.natm * ns;
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < total;
       t += (long long)gridDim.x * blockDim.x) {
    const int row = (int)(t / ns), k0 = (int)(t - (long long)row * ns);
    const int a = row >> 1, i = mc_ia(mv, a);
    const int m = k0 < s0 ? 0 : (k0 < s0 + s1 ? 1 : 2);
    const int off = m == 0 ? 0 : (m == 1 ? s0 : s0 + s1);
    const double x = (row & 1) ? mc_rtm(mv, 3 * a + m) : V.ro[3 * i + m];
    const double2 c = mc_factor<R, ORDER>(x, g.dkdr[m], g.s[m], root + off, k0 - off);
    const double q = m == 0 ? mc_charge<R, ORDER>(V, i) : 1.0;
    fac[t] = make_double2(c.x * q, c.y * q);
  }
}

template <int P>
__device__ __forceinline__ void mc_tab_body(const SysDev &V, int natm, int chunk,
                                            double2 *__restrict__ F,
                                            const double2 *__restrict__ fac, bool apply,
                                            double *__restrict__ part, int blk, int nblk) {
  extern __shared__ __align__(16) unsigned char mc_lds[];
  const int s0 = V.sg.s[0], s1 = V.sg.s[1], ns = s0 + s1 + V.sg.s[2];
  mc_pass<P>(V, natm, chunk, reinterpret_cast<double2 *>(mc_lds), F, apply, part, blk, nblk,
             [&](int a, int trial, int x, unsigned row) -> double2 {
               const double2 *f = fac + (size_t)(2 * a + trial) * ns;
               if (x >= 0) return f[x];
               const unsigned kz = row / (unsigned)s1;
               return mc_mul(f[s0 + (int)(row - kz * (unsigned)s1)], f[s0 + s1 + (int)kz]);
             });
}

template <int P>
__global__ void __launch_bounds__(256) k_mc_tab(const SysDev *__restrict__ sys, int natm,
                                                int chunk, double2 *spec,
                                                const double2 *__restrict__ fac, double *part) {
  mc_tab_body<P>(sys[0], natm, chunk, spec, fac, false, part, (int)blockIdx.x, (int)gridDim.x);
}

// UTwoBodyANew/UTwoBodyAOld (Src/denergy.F90:289-495) for a trial move of
// natm particles: each moved particle against its list partners that stay
// (u at the trial position minus u at the current one), plus the pairs of
// moved particles among themselves, each once (both trial minus both
// current, as its lptmdutwob branch), in FP64 on both precision paths.  A
// trial pair inside the hard core or below r2umin is an overlap (its goto
// 400).  One block and a list of tens of partners: the time is the chain
// of dependent loads, so the pair records are staged in LDS while the
// particle's own data arrive, a lane's first list entry is loaded with the
// list's length, and both positions of a pair are looked up together, by
// the bin of r2 (the interval the reference's walk from the pair's first
// interval to the first with r2 >= zlow stops at): 6.8 us with 9 partners,
// 9.3 with that walk, the two positions in turn and the move in host memory.
// One pair: u(d[0]) - u(d[1]), trial less current; skip() says that the pair
// is not to be counted, and is asked only within the cut-off: with the cell
// list's semantics the partners are all particles, nearly all of them
// beyond it (moves of 8 particles in 500000: 46.8 us, 82.7 with every pair
// looked up; of 64 in 50000: 93 us, 375 so and skip() asked for all).
template <typename Skip>
__device__ __forceinline__ double mc_pair_du(const SysDev &V, const PairRec *rec_s,
                                             const int *pidx_s, int ti, int tj,
                                             double (&d)[2][3], int &ovl, Skip skip) {
  const TableDev &t = V.tab;
  const int p = pidx_s[ti * t.npt + tj], nbin = t.nbin;
  const PairRec R = rec_s[p];
  const unsigned short *bins = reinterpret_cast<const unsigned short *>((const uint4 *)t.img) +
                               (size_t)p * nbin;
  const double *zl = (const double *)t.zlow + R.off;
  double r2[2], r2c[2], z0[2], z1[2], zv[2], u[2];
  bool in[2];
  int bk[2], iv[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    r2[s] = pbcr2(d[s][0], d[s][1], d[s][2], V.box);
    in[s] = V.nlsem == 0 ? !(r2[s] > t.rcut2) : (r2[s] < t.rcut2);
  }
  if ((!in[0] && !in[1]) || skip()) return 0.0;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    r2c[s] = fmax(r2[s], R.lo);
    const float sf = __builtin_amdgcn_rcpf((float)r2c[s]);
    bk[s] = bins[(int)fminf(fmaxf((sf - R.s_lo) * R.s_inv, 0.0f), (float)(nbin - 1))];
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int kb = bk[s] & (kSlowBin - 1);
    z0[s] = zl[kb];
    z1[s] = zl[min(kb + 1, R.nint - 1)];
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int kb = bk[s] & (kSlowBin - 1);
    if (bk[s] & kSlowBin) {
      iv[s] = find_interval([&](int k) -> double { return zl[k]; }, R.nint, r2c[s], kb);
      zv[s] = zl[iv[s]];
    } else {
      const bool at = r2c[s] >= z0[s];
      iv[s] = at ? kb : min(kb + 1, R.nint - 1);
      zv[s] = at ? z0[s] : z1[s];
    }
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const double2 *q = reinterpret_cast<const double2 *>((const double *)t.coef) +
                       (size_t)(kCoefStride / 2) * (R.off + iv[s]);
    const double2 a = q[0], b = q[1], c = q[2];
    const double x = r2[s] - zv[s];
    u[s] = a.x + x * (a.y + x * (b.x + x * (b.y + x * (c.x + x * c.y))));
    const bool ov = in[s] && (r2[s] < R.r2at || r2[s] < R.r2um);
    if (s == 0) ovl |= ov ? 1 : 0;
    if (!in[s] || ov) u[s] = 0.0;
  }
  return u[0] - u[1];
}

__global__ void __launch_bounds__(256) k_mc_pair(const SysDev *__restrict__ sys, const McMove mv,
                                                double *__restrict__ out,
                                                double *__restrict__ part) {
  const SysDev &V = sys[blockIdx.z];
  // up to kMcArg moved particles are in the arguments and copied into LDS
  // once per block, more are read from device memory
  __shared__ int ia_s[kMcArg];
  __shared__ double rtm_s[3 * kMcArg];
  __shared__ PairRec rec_s[MFE_MAX_PAIRS];
  __shared__ int pidx_s[MFE_MAX_TYPES * MFE_MAX_TYPES];
  const TableDev &tab = V.tab;
  const int natm = mv.natm;
  const bool staged = natm <= kMcArg;
  for (int k = threadIdx.x; k < tab.nptpt; k += blockDim.x) rec_s[k] = tab.rec[k];
  for (int k = threadIdx.x; k < tab.npt * tab.npt; k += blockDim.x) pidx_s[k] = tab.pairidx[k];
  if (staged) {
    for (int k = threadIdx.x; k < natm; k += blockDim.x) ia_s[k] = mv.ia_v[k];
    for (int k = threadIdx.x; k < 3 * natm; k += blockDim.x) rtm_s[k] = mv.rtm_v[k];
  }
  __syncthreads();
  const int *ia = staged ? ia_s : mv.ia;
  const double *rtm = staged ? rtm_s : mv.rtm;
  const int np = V.np;
  // cell-list semantics (UTwoBodyANew/OldCellList, Src/denergy.F90:728-928):
  // every particle within rcut of the old or new position, as the cells
  // around each position hold them; Verlet list (UTwoBodyANew/Old): the
  // moved particle's list partners, on all of the block's lanes for one
  // moved particle, else a wavefront per moved particle
  const bool all = V.nlsem == 1, whole = all || natm == 1;
  const int l0 = all ? (int)(blockIdx.x * blockDim.x + threadIdx.x)
                     : (whole ? (int)threadIdx.x : (int)(threadIdx.x & 63));
  const int nl = all ? (int)(gridDim.x * blockDim.x) : (whole ? (int)blockDim.x : 64);
  const int a1 = whole ? 1 : (int)(blockDim.x >> 6);
  double acc = 0.0;
  int ovl = 0;
  for (int a = whole ? 0 : (int)(threadIdx.x >> 6); a < natm; a += a1) {
    const int i = ia[a], t = V.c_pos[i], ti = V.type[i];
    const double xo = V.ro[3 * i], yo = V.ro[3 * i + 1], zo = V.ro[3 * i + 2];
    const double xn = rtm[3 * a], yn = rtm[3 * a + 1], zn = rtm[3 * a + 2];
    const int n = all ? np : V.nn[t];
    const int first = all ? 0 : V.nbr[(size_t)min(l0, V.maxnn - 1) * np + t];
    for (int k = l0; k < n; k += nl) {
      int jp, tj;
      double xj, yj, zj;
      if (all) {
        jp = k;
        tj = V.type[k];
        xj = V.ro[3 * k];
        yj = V.ro[3 * k + 1];
        zj = V.ro[3 * k + 2];
      } else {
        const int e = k == l0 ? first : V.nbr[(size_t)k * np + t];
        const int j = (int)((unsigned)e & kNbrIdxMask);  // cell-ordered slot
        jp = V.c_sorted[j];
        tj = V.type_s[j];
        xj = V.ro_s[3 * j];
        yj = V.ro_s[3 * j + 1];
        zj = V.ro_s[3 * j + 2];
      }
      // pairs of moved particles are counted below
      auto moved = [&]() {
        bool m = false;
        for (int b = 0; b < natm; ++b) m |= ia[b] == jp;
        return m;
      };
      double d[2][3] = {{xn - xj, yn - yj, zn - zj}, {xo - xj, yo - yj, zo - zj}};
      acc += mc_pair_du(V, rec_s, pidx_s, ti, tj, d, ovl, moved);
    }
  }
  for (int q = blockIdx.x == 0 ? (int)threadIdx.x : natm * natm; q < natm * natm;
       q += blockDim.x) {
    const int a = q / natm, b = q - a * natm;
    if (b <= a) continue;
    const int i = ia[a], j = ia[b];
    double d[2][3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      d[0][m] = rtm[3 * a + m] - rtm[3 * b + m];
      d[1][m] = V.ro[3 * i + m] - V.ro[3 * j + m];
    }
    acc += mc_pair_du(V, rec_s, pidx_s, V.type[i], V.type[j], d, ovl, [] { return false; });
  }
  __shared__ double red[256 / 64];
  for (int w = 32; w > 0; w >>= 1) acc += __shfl_down(acc, w, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  const int any = __syncthreads_or(ovl);
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
    if (gridDim.x == 1) {
      out[2 * blockIdx.z] = s;
      out[2 * blockIdx.z + 1] = any ? 1.0 : 0.0;
    } else {
      part[2 * blockIdx.x] = s;
      part[2 * blockIdx.x + 1] = any ? 1.0 : 0.0;
    }
  }
}

// the block partials of a many-block k_mc_pair in a fixed order
__global__ void __launch_bounds__(64) k_mc_pair_sum(const double *__restrict__ part, int nblk,
                                                    double *__restrict__ out) {
  double s = 0.0, o = 0.0;
  for (int b = threadIdx.x; b < nblk; b += 64) {
    s += part[2 * b];
    o = fmax(o, part[2 * b + 1]);
  }
  for (int w = 32; w > 0; w >>= 1) {
    s += __shfl_down(s, w, 64);
    o = fmax(o, __shfl_down(o, w, 64));
  }
  if (threadIdx.x == 0) {
    out[0] = s;
    out[1] = o;
  }
}

// --------------------------------------------------------- standard Ewald
// UEwaldRecStd (Src/energy.F90:1050-1096) over the k-vectors of its kfac
// table: one block per k-vector sums the four sign combinations of the
// structure factor; a second kernel gives each particle its force.
//
// The phases of a k-vector's four combinations (-x,-y,+z), (-x,+y,+z),
// (+x,-y,+z), (+x,+y,+z) are products of the three axes' phases, so a
// particle takes three sincos (or none, from a table per axis) in place of
// four, and at smaller arguments.
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ void four_phases(double2 ex, double2 ey, double2 ez, double2 e[4]) {
  const double2 exc = make_double2(ex.x, -ex.y);
  const double2 A = cmul(ey, ez), B = cmul(make_double2(ey.x, -ey.y), ez);
  e[0] = cmul(exc, B);
  e[1] = cmul(exc, A);
  e[2] = cmul(ex, B);
  e[3] = cmul(ex, A);
}
__device__ __forceinline__ double2 phase(double x) {
  double2 e;
  sincos(x, &e.y, &e.x);
  return e;
}

// 512 threads per k-vector (a thousand particles are two rounds), the eight
// sums combined through one LDS exchange: 1000 ions, 8 wave numbers per
// axis: 9.4 us (11.5 with 256 threads, four sincos, eight block sums); bound
// by the FP64 sincos chain of each thread.
constexpr int kSkThreads = 512;
__device__ __forceinline__ void ewald_sk_body(const SysDev &V, int energy, int kn) {
  if (kn >= V.nkvec) return;
  const double *__restrict__ ro = V.ro;
  const double *__restrict__ q = V.q;
  const int np = V.np;
  const double *__restrict__ kv = V.k_vec;
  const double alpha2 = V.alpha * V.alpha;
  __shared__ double red[8][kSkThreads / 64];
  const double kx = kv[4 * kn], ky = kv[4 * kn + 1], kz = kv[4 * kn + 2];
  double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int i = threadIdx.x; i < np; i += kSkThreads) {
    const double qi = q[i];
    double2 e[4];
    four_phases(phase(kx * ro[3 * i]), phase(ky * ro[3 * i + 1]), phase(kz * ro[3 * i + 2]), e);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      s[2 * c] += qi * e[c].x;
      s[2 * c + 1] += qi * e[c].y;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    for (int w = 32; w > 0; w >>= 1) s[c] += __shfl_down(s[c], w, 64);
    if (lane == 0) red[c][wave] = s[c];
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  // lane c of the first wavefront: component c, the wavefronts in order
  double t = 0.0;
  if (lane < 8) {
    for (int w = 0; w < kSkThreads / 64; ++w) t += red[lane][w];
    V.k_sum[8 * kn + lane] = t;
  }
  if (energy) {
    double t2 = t * t;
    for (int w = 4; w > 0; w >>= 1) t2 += __shfl_down(t2, w, 64);
    if (lane == 0) {
      double *part = V.part + V.off_std;
      const double term = kv[4 * kn + 3] * t2;
      const double k2 = kx * kx + ky * ky + kz * kz;
      part[kn] = term;
      part[V.nkvec + kn] = -(1.0 - k2 / (2.0 * alpha2)) * term;
    }
  }
}

__global__ void __launch_bounds__(kSkThreads) k_ewald_sk(const SysDev *__restrict__ sys,
                                                         int energy) {
  ewald_sk_body(sys[blockIdx.z], energy, (int)blockIdx.x);
}

// The mixed path's pair forces and the structure factors in one launch, the
// pair and skin blocks [0, npb) first: both leave most of the chip idle and
// share no data (1000 ions, 8 wave numbers per axis: 12 + 9 us in two).
static_assert(kSkThreads == kPairBlock, "the fused launch runs both bodies in one block size");
template <int NT, bool POS64>
__global__ void __launch_bounds__(kPairBlock) __attribute__((amdgpu_waves_per_eu(4)))
k_pair_sk(const SysDev *__restrict__ sys, int energy, int pgrid, int skin, int npb) {
  const int b = (int)blockIdx.x;
  if (b < npb) pair_f_body<NT, true, false, POS64>(sys, energy, pgrid, skin, b);
  else ewald_sk_body(sys[blockIdx.z], energy, b - npb);
}

// One wavefront per particle, its lanes over the k-vectors: a thread per
// particle ran every k-vector's four sincos one after another, on a few
// wavefronts (1000 ions, 8 wave numbers per axis: 259 us, now 5.8, bound by
// the reads of the structure factors and the launch).  TAB: the axes'
// phases e^{i n 2 pi x / L}, n = 0..ncut, are computed once per particle
// into LDS; without it (tables beyond the launch's LDS) per k-vector.
constexpr int kEwParticles = 4;
template <bool TAB>
__global__ void __launch_bounds__(64 * kEwParticles) k_ewald_force(
    const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  extern __shared__ __align__(16) double2 ew_tab[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = blockIdx.x * kEwParticles + wave;
  if (blockIdx.x * kEwParticles >= V.np) return;
  const bool act = i < V.np;
  const double *__restrict__ kv = V.k_vec;
  const double *__restrict__ ksum = V.k_sum;
  const int nk = V.nkvec, nt = V.ncut + 1;
  double2 *tab = ew_tab + (size_t)wave * 3 * nt;
  double r[3] = {0.0, 0.0, 0.0}, qi = 0.0;
  if (act) {
#pragma unroll
    for (int m = 0; m < 3; ++m) r[m] = V.ro[3 * i + m];
    qi = V.q[i];
  }
  if (TAB) {
    for (int e = lane; e < 3 * nt; e += 64) {
      const int m = e / nt, n = e - m * nt;
      tab[e] = phase((n * V.tpb[m]) * (m == 0 ? r[0] : (m == 1 ? r[1] : r[2])));
    }
    __syncthreads();
  }
  double fx = 0.0, fy = 0.0, fz = 0.0;
  for (int kn = lane; kn < nk; kn += 64) {
    const double kx = kv[4 * kn], ky = kv[4 * kn + 1], kz = kv[4 * kn + 2];
    const double kfac2 = V.efp * 2.0 * kv[4 * kn + 3];
    const double *S = ksum + 8 * kn;
    double2 ex, ey, ez, e[4];
    if (TAB) {
      const ushort4 n = V.k_n[kn];
      ex = tab[n.x];
      ey = tab[nt + n.y];
      ez = tab[2 * nt + n.z];
    } else {
      ex = phase(kx * r[0]);
      ey = phase(ky * r[1]);
      ez = phase(kz * r[2]);
    }
    four_phases(ex, ey, ez, e);
    double f[4];
    // -Re(q e) Im(S) + Im(q e) Re(S)
#pragma unroll
    for (int c = 0; c < 4; ++c) f[c] = qi * (-e[c].x * S[2 * c + 1] + e[c].y * S[2 * c]);
    fx += kfac2 * kx * (-f[0] - f[1] + f[2] + f[3]);
    fy += kfac2 * ky * (-f[0] + f[1] - f[2] + f[3]);
    fz += kfac2 * kz * (f[0] + f[1] + f[2] + f[3]);
  }
  for (int w = 32; w > 0; w >>= 1) {
    fx += __shfl_down(fx, w, 64);
    fy += __shfl_down(fy, w, 64);
    fz += __shfl_down(fz, w, 64);
  }
  if (act && lane == 0) {
    V.force[3 * i] += fx;
    V.force[3 * i + 1] += fy;
    V.force[3 * i + 2] += fz;
  }
}

// ------------------------------------------------------------------ bonds
// One bond angle of UAngle (Src/energy.F90:5409-5481), centred on bead c
// with neighbours jm (earlier) and jp (later): unit vectors from jm and jp
// to c, theta = acos(clamped cosine), u = k (theta - eq)^p with k already
// divided by p.  fm and fp are the forces on jm and jp; c receives
// -(fm + fp).  sin(theta) = 0 divides by zero, as in the reference.
__device__ __forceinline__ double angle_at(const double *__restrict__ ro, int c, int jm, int jp,
                                           const Box &b, double k, double eq, int p,
                                           double fm[3], double fp[3]) {
  double dxm = ro[3 * c] - ro[3 * jm], dym = ro[3 * c + 1] - ro[3 * jm + 1],
         dzm = ro[3 * c + 2] - ro[3 * jm + 2];
  const double dmi = 1.0 / sqrt(pbcr2(dxm, dym, dzm, b));
  dxm *= dmi;
  dym *= dmi;
  dzm *= dmi;
  double dxp = ro[3 * c] - ro[3 * jp], dyp = ro[3 * c + 1] - ro[3 * jp + 1],
         dzp = ro[3 * c + 2] - ro[3 * jp + 2];
  const double dpi = 1.0 / sqrt(pbcr2(dxp, dyp, dzp, b));
  dxp *= dpi;
  dyp *= dpi;
  dzp *= dpi;
  const double cosine = dxm * dxp + dym * dyp + dzm * dzp;
  const double theta = acos(fmax(-1.0, fmin(cosine, 1.0)));
  const double term = theta - eq;
  double pw = 1.0;
  for (int e = 1; e < p; ++e) pw *= term;
  double fac = k * pw;
  const double u = fac * term;
  fac = -p * fac / sin(theta);
  fm[0] = (fac * dmi) * (dxp - cosine * dxm);
  fm[1] = (fac * dmi) * (dyp - cosine * dym);
  fm[2] = (fac * dmi) * (dzp - cosine * dzm);
  fp[0] = (fac * dpi) * (dxm - cosine * dxp);
  fp[1] = (fac * dpi) * (dym - cosine * dyp);
  fp[2] = (fac * dpi) * (dzm - cosine * dzp);
  return u;
}

// UBond (Src/energy.F90:5335-5372): u = k (r - eq)^p with k already
// divided by p; each particle gathers the forces of its (at most two)
// bonds, and the bond to the next bead carries the energy.  With an angle
// force constant, also UAngle (Src/energy.F90:5409-5481): each particle
// gathers the forces of the (at most three) angles it takes part in, each
// angle evaluated by angle_at, and the centre bead carries the energy.
__global__ void __launch_bounds__(kBlock) k_bonds(const SysDev *__restrict__ sys,
                                                  int energy) {
  const SysDev &V = sys[blockIdx.z];
  if (V.nchain == 0 || (int)blockIdx.x >= V.nblk_np) return;
  const double *__restrict__ ro = V.ro;
  const int np = V.np;
  const int *__restrict__ prev = V.ch_prev;
  const int *__restrict__ next = V.ch_next;
  const Box b = V.box;
  const double k = V.bond_k, eq = V.bond_eq;
  const int p = V.bond_p;
  double *__restrict__ force = V.force;
  double *part = V.part + V.off_bond;
  __shared__ double sh[kBlock];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double ub = 0.0, vir = 0.0, ua = 0.0;
  if (i < np) {
    double f[3] = {0.0, 0.0, 0.0};
    const int nb2[2] = {next[i], prev[i]};
    for (int s = 0; s < 2; ++s) {
      const int j = nb2[s];
      if (j < 0) continue;
      // bond (a, c) with a the earlier bead: dx = ro(a) - ro(c)
      const int a = s == 0 ? i : j, c = s == 0 ? j : i;
      double dx = ro[3 * a] - ro[3 * c], dy = ro[3 * a + 1] - ro[3 * c + 1],
             dz = ro[3 * a + 2] - ro[3 * c + 2];
      const double r2 = pbcr2(dx, dy, dz, b);
      const double r1 = sqrt(r2);
      const double term = r1 - eq;
      double pw = 1.0;
      for (int e = 1; e < p; ++e) pw *= term;
      double fac = k * pw;
      if (s == 0) {
        ub += fac * term;
      }
      fac = -p * fac / r1;
      const double sg = s == 0 ? 1.0 : -1.0;
      f[0] += sg * fac * dx;
      f[1] += sg * fac * dy;
      f[2] += sg * fac * dz;
      if (s == 0) vir -= fac * r2;
    }
    if (V.ang_k != 0.0) {
      const double ka = V.ang_k, eqa = V.ang_eq;
      const int pa = V.ang_p;
      double fm[3], fp[3];
      const int jm = prev[i], jp = next[i];
      // i as the later bead of the angle centred on jm
      if (jm >= 0 && prev[jm] >= 0) {
        (void)angle_at(ro, jm, prev[jm], i, b, ka, eqa, pa, fm, fp);
        f[0] += fp[0];
        f[1] += fp[1];
        f[2] += fp[2];
      }
      // i as the centre
      if (jm >= 0 && jp >= 0) {
        ua += angle_at(ro, i, jm, jp, b, ka, eqa, pa, fm, fp);
        f[0] -= fm[0] + fp[0];
        f[1] -= fm[1] + fp[1];
        f[2] -= fm[2] + fp[2];
      }
      // i as the earlier bead of the angle centred on jp
      if (jp >= 0 && next[jp] >= 0) {
        (void)angle_at(ro, jp, i, next[jp], b, ka, eqa, pa, fm, fp);
        f[0] += fm[0];
        f[1] += fm[1];
        f[2] += fm[2];
      }
    }
    force[3 * i] += f[0];
    force[3 * i + 1] += f[1];
    force[3 * i + 2] += f[2];
  }
  if (energy) {
    double s1 = block_sum(ub, sh);
    double s2 = block_sum(vir, sh);
    double s3 = block_sum(ua, sh);
    if (threadIdx.x == 0) {
      part[blockIdx.x] = s1;
      part[V.nblk_np + blockIdx.x] = s2;
      part[2 * V.nblk_np + blockIdx.x] = s3;
    }
  }
}

// ------------------------------------------------------- surface + sums
__global__ void __launch_bounds__(kBlock) k_surf_sum(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  if (!V.lsurf || (int)blockIdx.x >= V.nblk_np) return;
  const double *__restrict__ ro = V.ro;
  const double *__restrict__ q = V.q;
  const int np = V.np;
  double *part = V.part + V.off_surf;
  __shared__ double sh[kBlock];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double s[3] = {0, 0, 0};
  if (i < np)
    for (int m = 0; m < 3; ++m) s[m] = q[i] * ro[3 * i + m];
  for (int m = 0; m < 3; ++m) {
    double t = block_sum(s[m], sh);
    if (threadIdx.x == 0) part[m * V.nblk_np + blockIdx.x] = t;
  }
}

constexpr int kRedComp = MFE_MAX_PAIRS + 12;

// Final sums in a fixed order (one block, one pass over the partials):
// writes en = [tot, twob0, rec, bond, virial, Sx, Sy, Sz, twob(1..nptpt)]
// and, in MD, the skin-test flag of NList (Src/nlist.F90:612-615).
// bd: also advance the replica's Brownian-dynamics step counter.
// Each wavefront sums whole components (partials are component-major),
// four independent accumulators per lane, then a shuffle tree; the fixed
// order keeps the result deterministic.
constexpr int kReduceThreads = 1024;

__device__ __forceinline__ void ph_reduce(const SysDev &V, int energy, int skin, int bd) {
  double *en = V.en;
  int *flags = V.flags;
  const int P = V.nptpt;
  const int nc = P + 11;
  const int nb = V.nblk_np;
  const int nrec = V.ewald == MFE_EWALD_SPME ? V.nblk_conv
                                             : (V.ewald == MFE_EWALD_STD ? V.nkvec : 0);
  const int offrec = V.ewald == MFE_EWALD_SPME ? V.off_conv : V.off_std;
  __shared__ double red[kRedComp];
  if (bd && threadIdx.x == 0) flags[3] += 1;
  // component layout: [0,P) pair energies, P pair virial, P+1..P+2 rec
  // (u, vir), P+3..P+4 bond (u, vir), P+5..P+7 S, P+8 max r2, P+9 cand,
  // P+10 angle u
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int c = wave; c < nc; c += (int)(blockDim.x >> 6)) {
    const double *src;
    int n;
    bool mx = false;
    if (c <= P) {
      src = V.part + V.off_pair + (size_t)c * V.nblk_pair;
      n = energy ? V.nblk_pair : 0;
    } else if (c <= P + 2) {
      src = V.part + offrec + (size_t)(c - P - 1) * nrec;
      n = energy ? nrec : 0;
    } else if (c <= P + 4) {
      src = V.part + V.off_bond + (size_t)(c - P - 3) * nb;
      n = (energy && V.nchain > 0) ? nb : 0;
    } else if (c <= P + 7) {
      src = V.part + V.off_surf + (size_t)(c - P - 5) * nb;
      n = V.lsurf ? nb : 0;
    } else if (c == P + 10) {
      src = V.part + V.off_bond + (size_t)2 * nb;
      n = (energy && V.nchain > 0 && V.ang_k != 0.0) ? nb : 0;
    } else {
      src = V.part + (c == P + 8 ? V.off_move : V.off_skin);
      n = skin ? nb : 0;
      mx = true;
    }
    // eight accumulators, eight loads in flight per lane
    double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int b2 = lane;
    for (; b2 + 7 * 64 < n; b2 += 8 * 64) {
      double a[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] = src[b2 + u * 64];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc[u] = mx ? fmax(acc[u], a[u]) : acc[u] + a[u];
    }
    for (; b2 < n; b2 += 64) acc[0] = mx ? fmax(acc[0], src[b2]) : acc[0] + src[b2];
    double sv;
    if (mx) {
      sv = fmax(fmax(fmax(acc[0], acc[1]), fmax(acc[2], acc[3])),
                fmax(fmax(acc[4], acc[5]), fmax(acc[6], acc[7])));
    } else {
      sv = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
    }
    for (int w = 32; w > 0; w >>= 1) {
      const double o = __shfl_down(sv, w, 64);
      sv = mx ? fmax(sv, o) : sv + o;
    }
    if (lane == 0) red[c] = sv;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  const double *v = red;
  const double S[3] = {v[P + 5], v[P + 6], v[P + 7]};
  for (int m = 0; m < 3; ++m) en[5 + m] = S[m];
  if (skin) flags[1] = (sqrt(v[P + 8]) + sqrt(v[P + 9]) > V.drnlist) ? 1 : 0;
  if (!energy) return;
  double twob0 = 0.0;
  for (int k = 0; k < P; ++k) {
    en[8 + k] = v[k];
    twob0 += v[k];
  }
  double vir = v[P];
  double urec = v[P + 1], virrec = v[P + 2];
  const double ubond = v[P + 3];
  vir += v[P + 4];
  double rec = 0.0;
  if (V.ewald != MFE_EWALD_NONE) {
    // self term; the neutralising background of a net charge scales as
    // 1/V, so its virial (dE/dlambda under r -> lambda r) is -3 times it
    urec += V.self_energy + V.net_energy;
    virrec -= 3.0 * V.net_energy;
    if (V.lsurf) {
      const double fac = 2.0 * 3.1415926535897932 / (3.0 * V.vol);
      const double term = fac * (S[0] * S[0] + S[1] * S[1] + S[2] * S[2]);
      urec += term;
      virrec -= term;
    }
    rec = V.efp * urec;
    vir += V.efp * virrec;
  }
  const double uangle = v[P + 10];
  en[0] = twob0 + rec + ubond + uangle;
  en[1] = twob0;
  en[2] = rec;
  en[3] = ubond;
  en[4] = vir;
  en[kEnAngle] = uangle;
}

__global__ void __launch_bounds__(kReduceThreads) k_reduce(const SysDev *__restrict__ sys,
                                                           int energy, int skin, int bd) {
  ph_reduce(sys[blockIdx.z], energy, skin, bd);
}

// --------------------------------------------------------------- adjoint
// Gradient of the pair model (Pot_1_6_12, Src/potential.F90:1349-1425,
// with exact erfc, plus the spline term) with respect to its parameters,
// summed over the same pair set as the pair kernel.  Each pair is seen from
// both ends: the visit (i, j) adds
//   dE/dq_i        q_j efp erfc(alpha r)/r                       (full)
//   dE/dsig[t_i]   1/2 dLJ/dsig_ij            (sig_ij = (sig_i+sig_j)/2)
//   dE/deps[t_i]   dLJ/deps_ij eps_j/(2 eps_ij)   (eps_ij = sqrt(eps_i eps_j))
//   dE/dc[p][k]    1/2 spline weight of coefficient k
// and 1/2 of the pair's model energy.  Per-block column partials:
// [E, dsig(npt), deps(npt), dc(nptpt*nknot)].
//
// Four lanes share a particle's list, each with the indices and then the
// positions of four entries in flight: a thread per particle, one entry at
// a time, left the FP64 units to a wavefront per SIMD (66000 particles, 117
// partners: 322 -> 130 us, now bound by FP64 issue: erfc, roots, divisions).
constexpr int kAdjLanes = 4;
constexpr int kAdjPer = kBlock / kAdjLanes;  // particles per block
__global__ void __launch_bounds__(kBlock) k_adjoint(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  const int np = V.np;
  if ((int)blockIdx.x * kAdjPer >= np) return;
  extern __shared__ double sk[];
  __shared__ double sh[kBlock / 64];
  const int nk = V.nptpt * V.nknot;
  // the types' parameters in LDS (read per entry by the partner's type); the
  // sums of the spline coefficients may take nearly all of it (adjoint_lds)
  __shared__ double zat_s[MFE_MAX_TYPES], sig_s[MFE_MAX_TYPES], eps_s[MFE_MAX_TYPES];
  const PairParams &pp = V.pp;
  const TableDev &t = V.tab;
  for (int k = threadIdx.x; k < V.npt; k += blockDim.x) {
    zat_s[k] = pp.zat[k];
    sig_s[k] = pp.sigat[k];
    eps_s[k] = pp.epsat[k];
  }
  for (int k = threadIdx.x; k < nk; k += blockDim.x) sk[k] = 0.0;
  __syncthreads();
  const Box b = V.box;
  const int lane = threadIdx.x % kAdjLanes;
  const int tt = blockIdx.x * kAdjPer + threadIdx.x / kAdjLanes;
  const bool act = tt < np;
  double eu = 0.0, gs = 0.0, ge = 0.0, phi = 0.0;
  int ti = -1;
  if (act) {
    const double xi = V.ro_s[3 * tt], yi = V.ro_s[3 * tt + 1], zi = V.ro_s[3 * tt + 2];
    ti = V.type_s[tt];
    const double qi = zat_s[ti];
    const int n = V.nn[tt];
    for (int k0 = lane; k0 < n; k0 += kPairBatch * kAdjLanes) {
      int pjs[kPairBatch], tjs[kPairBatch];
      double xs[kPairBatch], ys[kPairBatch], zs[kPairBatch];
#pragma unroll
      for (int u = 0; u < kPairBatch; ++u) {
        // rows clamped into the list; past its end the particle itself
        const int k = k0 + u * kAdjLanes;
        const int e = (int)((unsigned)V.nbr[(size_t)min(k, n - 1) * np + tt] & kNbrIdxMask);
        pjs[u] = k < n ? e : tt;
      }
#pragma unroll
      for (int u = 0; u < kPairBatch; ++u) {
        xs[u] = V.ro_s[3 * pjs[u]];
        ys[u] = V.ro_s[3 * pjs[u] + 1];
        zs[u] = V.ro_s[3 * pjs[u] + 2];
        tjs[u] = V.type_s[pjs[u]];
      }
#pragma unroll
      for (int u = 0; u < kPairBatch; ++u) {
        if (k0 + u * kAdjLanes >= n) break;
        double dx = xi - xs[u], dy = yi - ys[u], dz = zi - zs[u];
        const double r2 = pbcr2(dx, dy, dz, b);
        if (V.nlsem == 0 ? (r2 > t.rcut2) : !(r2 < t.rcut2)) continue;
        const int tj = tjs[u];
        const double r = sqrt(r2);
        const double qj = zat_s[tj];
        const double c0 = pp.lewald ? erfc(pp.alpha * r) : 1.0;
        phi += qj * pp.efp * c0 / r;
        eu += 0.5 * qi * qj * pp.efp * c0 / r;
        const double sig = 0.5 * (sig_s[ti] + sig_s[tj]);
        const double eps = sqrt(eps_s[ti] * eps_s[tj]);
        if (!pp.lljcut || r < pp.ljrcut * sig) {
          const double x = sig / r, x2 = x * x, s6 = x2 * x2 * x2, s12 = s6 * s6;
          const double sh_ = pp.lljcut ? pp.ljushift : 0.0;
          eu += 0.5 * (4.0 * eps * (s12 - s6) + sh_ * eps);
          gs += 0.5 * 4.0 * eps * (12.0 * s12 - 6.0 * s6) / sig;
          if (eps > 0.0) ge += (4.0 * (s12 - s6) + sh_) * eps_s[tj] / (2.0 * eps);
        }
        if (V.nknot) {
          int ki;
          double w[4], dw[4];
          if (knot_weights(r, V.knot_r0, V.knot_dinv, V.nknot, ki, w, dw)) {
            const int pidx = pair_index(ti, tj, t.npt);
            const double *c = V.knot_c + (size_t)pidx * V.nknot + ki;
            eu += 0.5 * (c[0] * w[0] + c[1] * w[1] + c[2] * w[2] + c[3] * w[3]);
            for (int m = 0; m < 4; ++m) atomicAdd(&sk[pidx * V.nknot + ki + m], 0.5 * w[m]);
          }
        }
      }
    }
  }
  phi = lane_sum(phi, kAdjLanes);
  if (act && lane == 0) V.adj_phi[V.c_sorted[tt]] = phi;
  double *out = V.adj_part + (size_t)blockIdx.x * V.adj_ncol;
  const double se = block_sum(eu, sh);
  if (threadIdx.x == 0) out[0] = se;
  for (int u = 0; u < V.npt; ++u) {
    const double a = block_sum(ti == u ? gs : 0.0, sh);
    const double c = block_sum(ti == u ? ge : 0.0, sh);
    if (threadIdx.x == 0) {
      out[1 + u] = a;
      out[1 + V.npt + u] = c;
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < nk; k += blockDim.x) out[1 + 2 * V.npt + k] = sk[k];
}

// dE/dq_i = real-space potential + efp * reciprocal potential
//           - 2 efp alpha/sqrt(pi) q_i (UEwaldSelf) + surface term
// and what the caller gets of it and of the forces: the block's sums per
// type (dE/dzat) into zpart[block][npt], and dE/dr = -force (UTotal's
// force before the unit scaling) into dro, both formed here because the
// host took 0.25 ms for the sum and the 3 np divisions of 66000 particles.
__global__ void __launch_bounds__(kBlock) k_adjoint_q(const SysDev *__restrict__ sys,
                                                      double *__restrict__ zpart,
                                                      double *__restrict__ dro) {
  const SysDev &V = sys[blockIdx.z];
  __shared__ double sh[kBlock / 64];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double d = 0.0;
  int t = -1;
  if (i < V.np) {
    d = V.adj_phi[i];
    t = V.type[i];
    if (V.ewald == MFE_EWALD_SPME) {
      d += V.phi_rec[i];
      d -= 2.0 * V.efp * (V.alpha / 1.7724538509055160273) * V.q[i];
      d += V.efp * V.net_dq;
    }
    if (V.lsurf) {
      // efp (2 pi/3V) |sum q r|^2 -> efp (4 pi/3V) (sum q r) . r_i
      const double f = V.efp * 4.0 * 3.1415926535897932 / (3.0 * V.vol);
      d += f * (V.en[5] * V.ro[3 * i] + V.en[6] * V.ro[3 * i + 1] + V.en[7] * V.ro[3 * i + 2]);
    }
    V.adj_dq[i] = d;
#pragma unroll
    for (int m = 0; m < 3; ++m) dro[3 * i + m] = -V.forceo[3 * i + m] / V.ffac;
  }
  for (int k = 0; k < V.npt; ++k) {
    const double z = block_sum(t == k ? d : 0.0, sh);
    if (threadIdx.x == 0) zpart[(size_t)blockIdx.x * V.npt + k] = z;
  }
}

// column sums of the adjoint's block partials in a fixed order
__global__ void __launch_bounds__(kSumThreads) k_adjoint_sum(const double *__restrict__ part,
                                                             int rows, int ncol, double *out) {
  column_sums(part, rows, ncol, ncol, out, false);
}

// ------------------------------------------------- counter-based noise
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as
// easy as 1, 2, 3", SC'11): ten rounds of two 32x32->64 multiplies with
// the round keys bumped by the Weyl constants.
__host__ __device__ __forceinline__ void philox_round(uint32_t c[4], const uint32_t k[2]) {
  const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
  const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
  const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
  const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
  const uint32_t n0 = hi1 ^ c[1] ^ k[0], n2 = hi0 ^ c[3] ^ k[1];
  c[0] = n0;
  c[1] = lo1;
  c[2] = n2;
  c[3] = lo0;
}

__host__ __device__ __forceinline__ void philox10(uint32_t c[4], uint32_t k0, uint32_t k1) {
  uint32_t k[2] = {k0, k1};
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    philox_round(c, k);
    k[0] += 0x9E3779B9u;
    k[1] += 0xBB67AE85u;
  }
}

// three standard normal deviates for particle i at step n: Box-Muller on
// the uniforms (x + 1/2) 2^-32 of the first two pairs of Philox words
__device__ __forceinline__ void gauss3(unsigned long long seed, unsigned i, unsigned n,
                                       double g[3]) {
  uint32_t c[4] = {i, n, 0u, 0u};
  philox10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
  const double s = 2.3283064365386963e-10;  // 2^-32
  const double u0 = ((double)c[0] + 0.5) * s, u1 = ((double)c[1] + 0.5) * s;
  const double u2 = ((double)c[2] + 0.5) * s, u3 = ((double)c[3] + 0.5) * s;
  const double r0 = sqrt(-2.0 * log(u0)), r1 = sqrt(-2.0 * log(u2));
  double sn, cs;
  sincospi(2.0 * u1, &sn, &cs);
  g[0] = r0 * cs;
  g[1] = r0 * sn;
  g[2] = r1 * cospi(2.0 * u3);
}

// ------------------------------------------------------------ integrators
// VelVer positions (Src/md.F90:287-298): drostep = dt v + dt^2/2 a,
// ro += drostep, PBC with ANINT; the skin bookkeeping of NList
// (Src/nlist.F90:601-603) is folded in: drosum += drostep, r2 = |drosum|^2
// and the block maximum of r2 for the second-largest rule.
// For BD (Src/bd.F90:141-151): drostep = fac1 forceo + fac2 noise, with
// the noise supplied by the host (bd = 1) or drawn from the replica's
// counter-based stream (bd = 2): particle i at BD step n takes
// Philox4x32-10(counter (i, n, 0, 0), key seed) and three Box-Muller
// deviates of it.
__global__ void __launch_bounds__(kBlock) k_move(const SysDev *__restrict__ sys,
                                                 double dt, int bd) {
#pragma clang fp contract(off)
  const SysDev &V = sys[blockIdx.z];
  if ((int)blockIdx.x >= V.nblk_np) return;
  // after a failed list rebuild (a grid barrier gave up) the state stays
  // where it was for the rest of the call, which then reports the error:
  // the flag is read alongside the particle's loads and holds back only
  // the stores (the block maximum it still writes feeds a skin decision
  // that no rebuild acts on after the failure)
  const bool halt = (V.flags[0] & ERR_SYNC) != 0;
  double *__restrict__ ro = V.ro;
  const double *__restrict__ rod = V.rod;
  const double *__restrict__ rodd = V.rodd;
  const double *__restrict__ forceo = V.forceo;
  const int *__restrict__ type = V.type;
  const double *__restrict__ fac1 = V.bd_fac1;
  const double *__restrict__ fac2 = V.bd_fac2;
  const int np = V.np;
  const Box b = V.box;
  double *__restrict__ drosum = V.drosum;
  double *r2disp = V.r2disp;
  double *part_max = V.part + V.off_move;
  __shared__ double sh[kBlock];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double r2 = 0.0;
  if (i < np) {
    // every load before the first store (the arrays may alias as far as
    // the compiler knows, which would serialise the loads behind stores)
    const double fac = 0.5 * (dt * dt);
    double x[3], d[3], s[3];
    const int cp = V.c_pos[i];
    const int cell = V.pos_f ? V.c_of[i] : 0, ty = V.pos_f ? type[i] : 0;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      x[m] = ro[3 * i + m];
      s[m] = drosum[3 * i + m];
    }
    if (bd) {
      double gn[3] = {0.0, 0.0, 0.0};
      if (bd == 1) {
#pragma unroll
        for (int m = 0; m < 3; ++m) gn[m] = V.noise[3 * i + m];
      } else {
        gauss3(V.seed, (unsigned)i, (unsigned)V.flags[3], gn);
      }
      const int t = type[i];
      const double f1 = fac1[t], f2 = fac2[t];
#pragma unroll
      for (int m = 0; m < 3; ++m) d[m] = f1 * forceo[3 * i + m] + f2 * gn[m];
    } else {
      double v[3], a[3];
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        v[m] = rod[3 * i + m];
        a[m] = rodd[3 * i + m];
      }
#pragma unroll
      for (int m = 0; m < 3; ++m) d[m] = dt * v[m] + fac * a[m];
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      double xm = x[m] + d[m];
      if (fabs(xm) > b.L2[m]) xm = xm - b.L[m] * round(xm * b.Li[m]);
      x[m] = xm;
      s[m] = s[m] + d[m];
    }
    r2 = s[0] * s[0];
    r2 = r2 + s[1] * s[1];
    r2 = r2 + s[2] * s[2];
    if (!halt) {
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        ro[3 * i + m] = x[m];
        V.ro_s[3 * cp + m] = x[m];
        drosum[3 * i + m] = s[m];
      }
      if (V.pos_f) V.pos_f[cp] = rel_pos(V, x, cell, ty);
      r2disp[i] = r2;
    }
  }
  const double m = block_max(r2, sh);
  if (threadIdx.x == 0) part_max[blockIdx.x] = m;
}

// New positions with a valid list: NList's displacement bookkeeping
// (Src/nlist.F90:601-603) on the step since the last upload, taken as the
// minimum image of new - old (one shift per axis, as PBCr2), so the skin
// test that follows decides whether the list is rebuilt.  The new
// positions are ro_new (a host upload), or, with ro_new null, the current
// ones with the move's particles (at most kMcArg) at their new places.
__device__ __forceinline__ void set_positions_body(const SysDev &V,
                                                   const double *__restrict__ ro_new,
                                                   const McMove *mv) {
#pragma clang fp contract(off)
  __shared__ double sh[kBlock];
  const Box b = V.box;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double r2 = 0.0;
  if (i < V.np) {
    // every load before the first store
    double xn[3], xo[3], s[3];
    const int cp = V.c_pos[i];
    const int cell = V.pos_f ? V.c_of[i] : 0, ty = V.pos_f ? V.type[i] : 0;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      xo[m] = V.ro[3 * i + m];
      s[m] = V.drosum[3 * i + m];
    }
    if (ro_new) {
#pragma unroll
      for (int m = 0; m < 3; ++m) xn[m] = ro_new[3 * i + m];
    } else {
#pragma unroll
      for (int m = 0; m < 3; ++m) xn[m] = xo[m];
      for (int a = 0; a < mv->natm; ++a)
        if (mv->ia_v[a] == i) {
#pragma unroll
          for (int m = 0; m < 3; ++m) xn[m] = mv->rtm_v[3 * a + m];
        }
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      double d = xn[m] - xo[m];
      if (fabs(d) > b.L2[m]) d = d - copysign(b.L[m], d);
      s[m] = s[m] + d;
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      V.ro[3 * i + m] = xn[m];
      V.ro_s[3 * cp + m] = xn[m];
      V.drosum[3 * i + m] = s[m];
    }
    if (V.pos_f) V.pos_f[cp] = rel_pos(V, xn, cell, ty);
    const double *ds = s;
    r2 = ds[0] * ds[0];
    r2 = r2 + ds[1] * ds[1];
    r2 = r2 + ds[2] * ds[2];
    V.r2disp[i] = r2;
  }
  const double mx = block_max(r2, sh);
  if (threadIdx.x == 0) V.part[V.off_move + blockIdx.x] = mx;
}

__global__ void __launch_bounds__(kBlock) k_set_positions(const SysDev *__restrict__ sys,
                                                          const double *__restrict__ ro_new) {
  const SysDev &V = sys[blockIdx.z];
  if ((int)blockIdx.x < V.nblk_np) set_positions_body(V, ro_new, nullptr);
}

// An accepted move: the first nset blocks (V.nblk_np, or none where the
// positions are set apart) place a move of up to kMcArg particles and update
// the displacements, the others add the trial's change to the kept spectrum
// (none where no spectrum is kept).  That change is taken from `old`, the
// positions before the move, or from the trial's factor table, so the two
// parts are independent: 9.3 us in one launch (one of 50000 particles, 80^3
// mesh), 4.6 and 5.9 us in two.
template <typename R, int ORDER>
__global__ void __launch_bounds__(kBlock) k_mc_accept(const SysDev *__restrict__ sys,
                                                      const McMove mv, int nset, int chunk,
                                                      double2 *spec, double *old) {
  if ((int)blockIdx.x < nset)
    set_positions_body(sys[0], nullptr, &mv);
  else
    mc_rec_body<R, ORDER>(sys[0], mv, chunk, spec, old, true, nullptr, (int)blockIdx.x - nset,
                          (int)gridDim.x - nset);
}
// the same with the change from the trial's factor table
template <int P>
__global__ void __launch_bounds__(kBlock) k_mc_accept_tab(const SysDev *__restrict__ sys,
                                                          const McMove mv, int nset, int chunk,
                                                          double2 *spec,
                                                          const double2 *__restrict__ fac) {
  if ((int)blockIdx.x < nset)
    set_positions_body(sys[0], nullptr, &mv);
  else
    mc_tab_body<P>(sys[0], mv.natm, chunk, spec, fac, true, nullptr, (int)blockIdx.x - nset,
                   (int)gridDim.x - nset);
}

// NList's r2max2 (Src/nlist.F90:602-608) is the largest r2 that is not a
// new running maximum at the moment it is visited in particle order.  Each
// block owns the same particle range as in k_move; the running maximum
// entering it is the max of the earlier blocks' maxima.
__global__ void __launch_bounds__(kBlock) k_skin_blocks(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  if ((int)blockIdx.x >= V.nblk_np) return;
  const double *__restrict__ r2disp = V.r2disp;
  const int np = V.np;
  const double *part_max = V.part + V.off_move;
  double *part_cand = V.part + V.off_skin;
  __shared__ double sh[kBlock];
  double pm = 0.0;
  for (int b2 = threadIdx.x; b2 < (int)blockIdx.x; b2 += blockDim.x) pm = fmax(pm, part_max[b2]);
  const double P = block_max(pm, sh);
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const double v = i < np ? r2disp[i] : 0.0;
  // running max in particle order: inclusive max-scan inside each
  // wavefront by shuffles, then the maxima of the earlier wavefronts
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double inc = v;
  for (int off = 1; off < 64; off <<= 1) {
    const double y = __shfl_up(inc, off, 64);
    if (lane >= off) inc = fmax(inc, y);
  }
  double excl = __shfl_up(inc, 1, 64);
  if (lane == 0) excl = 0.0;
  __shared__ double wmax[kBlock / 64];
  if (lane == 63) wmax[wave] = inc;
  __syncthreads();
  double pw = 0.0;
  for (int k = 0; k < wave; ++k) pw = fmax(pw, wmax[k]);
  const double before = fmax(P, fmax(pw, excl));
  const double cand = (i < np && !(v > before)) ? v : 0.0;
  const double c = block_max(cand, sh);
  if (threadIdx.x == 0) part_cand[blockIdx.x] = c;
}

// UTotal's tail (Src/energy.F90:405-418) plus, for MD, GetLinAcc and the
// velocity half of VelVer (Src/md.F90:348-358):
//   mode 0: forceo = force*fac        mode 1: + VelVer kick
// one particle of k_finalize; es = the reduced surface field en[5..7]
__device__ __forceinline__ void fin_load(const SysDev &V, int i, int mode, FinState &st) {
  if (mode == 1) {
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      st.aold[m] = V.rodd[3 * i + m];
      st.v[m] = V.rod[3 * i + m];
    }
  }
  st.q = V.lsurf ? V.q[i] : 0.0;
  st.mi = mode == 1 ? V.massip[i] : 0.0;
}

__device__ __forceinline__ void fin_apply(const SysDev &V, int i, const double f[3],
                                         const FinState &st, int mode, double dt,
                                         const double es[3]) {
#pragma clang fp contract(off)
  double *__restrict__ forceo = V.forceo;
  const double ffac = V.ffac, surf_fac = V.surf_fac;
  const int surf = V.lsurf;
  double *__restrict__ rod = V.rod;
  double *__restrict__ rodd = V.rodd;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    double fm = f[m];
    if (surf) fm = fm - surf_fac * st.q * es[m];
    const double fo = fm * ffac;
    forceo[3 * i + m] = fo;
    if (mode == 1) {
      const double anew = st.mi * fo;
      rodd[3 * i + m] = anew;
      rod[3 * i + m] = st.v[m] + 0.5 * dt * (anew + st.aold[m]);
    }
  }
}

// every load before the first store; split: the reciprocal forces are in
// force_rec (the fused pair + gather launch), added here
__device__ __forceinline__ void ph_finalize(const SysDev &V, int i, int mode, double dt,
                                            const double es[3], bool split = false) {
  double f[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) f[m] = V.force[3 * i + m];
  if (split) {
    double r[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) r[m] = V.force_rec[3 * i + m];
#pragma unroll
    for (int m = 0; m < 3; ++m) f[m] = f[m] + r[m];
  }
  FinState st;
  fin_load(V, i, mode, st);
  fin_apply(V, i, f, st, mode, dt, es);
}

__global__ void __launch_bounds__(kBlock) k_finalize(const SysDev *__restrict__ sys,
                                                     int mode, double dt) {
  const SysDev &V = sys[blockIdx.z];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V.np) return;
  double es[3] = {0.0, 0.0, 0.0};
  if (V.lsurf) {
#pragma unroll
    for (int m = 0; m < 3; ++m) es[m] = V.en[5 + m];
  }
  ph_finalize(V, i, mode, dt, es);
}

// Without the surface term the reduction and k_finalize are independent:
// one launch in which block 0 reduces the partials (dispatched first, so
// its chain of loads overlaps the rest) and blocks [1, F] finalize
// kReduceThreads particles each (F of the replica).
__global__ void __launch_bounds__(kReduceThreads) k_reduce_finalize(const SysDev *__restrict__ sys,
                                                                    int energy, int skin, int bd,
                                                                    int mode, double dt,
                                                                    int split) {
  const SysDev &V = sys[blockIdx.z];
  const int F = (V.np + kReduceThreads - 1) / kReduceThreads;
  if (blockIdx.x == 0) {
    ph_reduce(V, energy, skin, bd);
    return;
  }
  if ((int)blockIdx.x <= F) {
    const int i = ((int)blockIdx.x - 1) * kReduceThreads + threadIdx.x;
    const double es[3] = {0.0, 0.0, 0.0};
    if (i < V.np) ph_finalize(V, i, mode, dt, es, split != 0);
  }
}

// The last launch of an MD or BD step on one engine: k_reduce_finalize's
// work (block 0 reduces, the other blocks finalize the particles, grid-
// stride) and then, in the same launch, the gated list rebuild.  Every
// block takes the skin decision itself, ph_reduce's test on the same block
// maxima (Src/nlist.F90:601-608), so no block waits for another to learn
// it, and the launch ends there when the test did not fire.  The rebuild
// reads the positions and writes the cell, list and cell-ordered arrays;
// the finalize reads and writes forces, velocities and accelerations only,
// so the rebuild's first phase needs no barrier after it.  One
// 1024-thread block per CU, all resident, as the rebuild's grid barriers
// require.
// mode < 0: no finalize (new positions from the host or an accepted MC
// move).  hflags, if given, is pinned host memory for the flags as they
// stand when the test did not fire, which spares the host a copy; where
// hflags[1] says that it fired, the host reads them after the rebuild.
__global__ void __launch_bounds__(kReduceThreads) k_finalize_rebuild(
    const SysDev *__restrict__ sys, int energy, int bd, int mode, double dt, int split,
    unsigned *bar, int spin, int *hflags) {
  const SysDev &V = sys[0];
  const int nb = V.nblk_np;
  const double *pmove = V.part + V.off_move, *pcand = V.part + V.off_skin;
  // this thread's share of the two maxima, loaded before the finalize so
  // that the loads overlap it
  double m1 = 0.0, m2 = 0.0;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) {
    m1 = fmax(m1, pmove[b]);
    m2 = fmax(m2, pcand[b]);
  }
  if (blockIdx.x == 0) {
    ph_reduce(V, energy, 1, bd);
  } else if (mode >= 0) {
    const double es[3] = {0.0, 0.0, 0.0};
    const int stride = ((int)gridDim.x - 1) * kReduceThreads;
    for (int i = ((int)blockIdx.x - 1) * kReduceThreads + (int)threadIdx.x; i < V.np;
         i += stride)
      ph_finalize(V, i, mode, dt, es, split != 0);
  }
  __shared__ double mx_s[2][kReduceThreads / 64];
  __shared__ int void_s;
  // one thread's reading decides for the block: a block of this launch may
  // raise the error meanwhile, and waves that read different values would
  // part, some into the rebuild without the others
  if (threadIdx.x == 0)
    void_s = __hip_atomic_load(&V.flags[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ERR_SYNC;
  for (int w = 32; w > 0; w >>= 1) {
    m1 = fmax(m1, __shfl_xor(m1, w, 64));
    m2 = fmax(m2, __shfl_xor(m2, w, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    mx_s[0][threadIdx.x >> 6] = m1;
    mx_s[1][threadIdx.x >> 6] = m2;
  }
  __syncthreads();
  double M1 = 0.0, M2 = 0.0;
  for (int w = 0; w < kReduceThreads / 64; ++w) {
    M1 = fmax(M1, mx_s[0][w]);
    M2 = fmax(M2, mx_s[1][w]);
  }
  const bool fired = sqrt(M1) + sqrt(M2) > V.drnlist;
  if (hflags && blockIdx.x == 0 && threadIdx.x == 0) {
    hflags[0] = V.flags[0];
    hflags[1] = fired ? 1 : 0;
    hflags[2] = V.flags[2];
  }
  if (!fired) return;
  // after a failed rebuild earlier in the call the list stays void
  if (void_s) return;
  rebuild_phases(V, bar, spin);
}

// ------------------------------------------------- persistent batched BD
// Many small replicas advanced by BDStep in one launch: a workgroup takes
// a replica from a queue (the costliest first), runs all nsteps steps of
// it -- move with the counter-based noise, NList's skin test, FP32 pair
// forces, SPME (fixed-point spreading into the replica's own mesh, the five
// FFT passes tile by tile, Green function, gather), the finalize and the
// reductions, the gated list rebuild -- with workgroup barriers only, then
// takes the next replica.  The arithmetic is the mixed path's: the same
// pair evaluation (pair_eval_f), B-splines, FFT passes and reductions in
// FP64.  Each replica's result depends on that replica alone (integer
// spreading sums, fixed summation orders), so a batch computes exactly
// what the same kernel computes for each replica on its own.
// Eligible replicas: mixed precision, SPME, no chains, surface term or
// spline knots.

struct PersistArgs {
  const SysDev *sys;
  const int *order;                   // replica indices, costliest first
  int nrep, nsteps, energy;
  int *queue;                         // dequeue counter, zero at the launch
  int lds;                            // dynamic LDS bytes (tables, slabs, FFT tiles)
};

// inclusive prefix maximum over the block of one value per thread (wave
// shuffles, then the earlier waves' maxima from LDS); tot gets the block's
// maximum.  wm: one slot per wave.
__device__ __forceinline__ double block_prefix_max(double v, double *wm, double &excl,
                                                   double &tot) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  double inc = v;
  for (int off = 1; off < 64; off <<= 1) {
    const double y = __shfl_up(inc, off, 64);
    if (lane >= off) inc = fmax(inc, y);
  }
  double e = __shfl_up(inc, 1, 64);
  if (lane == 0) e = 0.0;
  if (lane == 63) wm[wave] = inc;
  __syncthreads();
  double pw = 0.0, t = 0.0;
  for (int k = 0; k < nw; ++k) {
    if (k < wave) pw = fmax(pw, wm[k]);
    t = fmax(t, wm[k]);
  }
  __syncthreads();
  excl = fmax(pw, e);
  tot = t;
  return inc;
}

// exclusive prefix sum of cnt[0..n) into start[0..n], start[n] = total;
// the counts are left zero, as every rebuild expects them (ph_cell_rank)
__device__ __forceinline__ void block_scan_counts(int *cnt, int *start, int n, int *wsum) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int carry = 0;
  for (int base = 0; base < n; base += blockDim.x) {
    const int k = base + threadIdx.x;
    const int v = k < n ? cnt[k] : 0;
    int inc = v;
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(inc, off, 64);
      if (lane >= off) inc += y;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    int pw = 0, t = 0;
    for (int w = 0; w < nw; ++w) {
      if (w < wave) pw += wsum[w];
      t += wsum[w];
    }
    if (k < n) {
      start[k] = carry + pw + inc - v;
      cnt[k] = 0;
    }
    carry += t;
    __syncthreads();
  }
  if (threadIdx.x == 0) start[n] = carry;
}

// BDStep for particle i at step n (k_move's arithmetic, device noise):
// position, its cell-ordered copies, NList's displacement sum; returns
// |sum|^2 (also stored in r2disp)
__device__ __forceinline__ double bd_move_particle(const SysDev &V, int i, unsigned n) {
#pragma clang fp contract(off)
  const Box b = V.box;
  double x[3], d[3], sd[3], gn[3];
  const int cp = V.c_pos[i];
  const int cell = V.c_of[i], ty = V.type[i];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    x[m] = V.ro[3 * i + m];
    sd[m] = V.drosum[3 * i + m];
  }
  gauss3(V.seed, (unsigned)i, n, gn);
  const double f1 = V.bd_fac1[ty], f2 = V.bd_fac2[ty];
#pragma unroll
  for (int m = 0; m < 3; ++m) d[m] = f1 * V.forceo[3 * i + m] + f2 * gn[m];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    double xm = x[m] + d[m];
    if (fabs(xm) > b.L2[m]) xm = xm - b.L[m] * round(xm * b.Li[m]);
    x[m] = xm;
    sd[m] = sd[m] + d[m];
  }
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    V.ro[3 * i + m] = x[m];
    V.ro_s[3 * cp + m] = x[m];
    V.drosum[3 * i + m] = sd[m];
  }
  V.pos_f[cp] = rel_pos(V, x, cell, ty);
  double r2 = sd[0] * sd[0];
  r2 = r2 + sd[1] * sd[1];
  r2 = r2 + sd[2] * sd[2];
  V.r2disp[i] = r2;
  return r2;
}

// The stages of the persistent step, each a function of its own (not
// inlined) so that register allocation works stage by stage.
#define MFE_STAGE __device__ __attribute__((noinline))

// BDStep for the replica's particles, then NList's skin test
// (Src/nlist.F90:597-621): the largest displacement and the largest one
// that was not a running maximum, in particle order.  Returns the rebuild
// decision (every thread).
MFE_STAGE int p_move_skin(const SysDev &V, unsigned stepctr, double *wm, int *flag_s) {
  const int tid = threadIdx.x, NT = blockDim.x, np = V.np;
  double run = 0.0, cand = 0.0;
  for (int base = 0; base < np; base += NT) {
    const int i = base + tid;
    const double v = i < np ? bd_move_particle(V, i, stepctr) : 0.0;
    double excl, tot;
    block_prefix_max(v, wm, excl, tot);
    const double before = fmax(run, excl);
    if (i < np && !(v > before)) cand = fmax(cand, v);
    run = fmax(run, tot);
  }
  const double c = block_max(cand, wm);
  if (tid == 0) *flag_s = (sqrt(run) + sqrt(c) > V.drnlist) ? 1 : 0;
  __syncthreads();
  return *flag_s;
}

// Where the persistent pair stage keeps the replica's cell-relative
// positions: after the tables in LDS (offset po) when they fit the launch's
// dynamic LDS, and the separations are formed in FP32; else (false) they
// are read from global memory.
__device__ __forceinline__ bool pair_pos_in_lds(const SysDev &V, int lds, size_t &po) {
  const TableDev &t = V.tab;
  size_t tb = pair_bin_bytes(t.nptpt, t.nbin) + pair_zl_bytes(t.nzl);
  if (t.lds_mode >= 2) tb += (size_t)t.nzl * kCoefStride * sizeof(float);
  po = (tb + 15) / 16 * 16;
  return V.pair_pos64 == 0 && po + (size_t)V.np * sizeof(float4) <= (size_t)lds;
}

// FP32 pair forces in cell order, one lane per particle (pair_eval_f);
// per-wavefront pair-type energies in wred[wave][0..P), virial in [P].
// NTY bounds the number of particle types (energies per partner type).
// POSL: the partners' positions are read from an LDS copy (pair_pos_in_lds),
// a few hundred cycles instead of an L2 round trip per batch of partners.
template <int NTY, bool POSL>
MFE_STAGE void p_pair(const SysDev &V, int energy, char *smem, int lds, double (*wred)[40],
                      PairRecF *rec_s, int *pidx_s, float4 *off_s) {
  const int tid = threadIdx.x, NT = blockDim.x, np = V.np;
  const int lane = tid & 63, wave = tid >> 6;
  const TableDev t = V.tab;
  const int P = t.nptpt, npt = t.npt, nbin = t.nbin, nzl = t.nzl;
  const size_t bb = pair_bin_bytes(P, nbin);
  unsigned short *bin_s = reinterpret_cast<unsigned short *>(smem);
  float *zl_s = reinterpret_cast<float *>(smem + bb);
  float *cf_s = reinterpret_cast<float *>(smem + bb + pair_zl_bytes(nzl));
  const bool cf_lds = t.lds_mode >= 2;
  stage_image(reinterpret_cast<unsigned char *>(smem), t,
              bb + pair_zl_bytes(nzl) + (cf_lds ? (size_t)nzl * kCoefStride * sizeof(float) : 0));
  for (int k = tid; k < P; k += NT) rec_s[k] = t.rec_f[k];
  for (int k = tid; k < npt * npt; k += NT) pidx_s[k] = t.pairidx[k];
  for (int k = tid; k < 125; k += NT)
    off_s[k] = make_float4(V.cg.off[0][k % 5], V.cg.off[1][(k / 5) % 5], V.cg.off[2][k / 25], 0.f);
  for (int k = lane; k <= P; k += 64) wred[wave][k] = 0.0;
  const float4 *__restrict__ pos = V.pos_f;
  if constexpr (POSL) {
    size_t po = 0;
    (void)pair_pos_in_lds(V, lds, po);
    float4 *pos_s = reinterpret_cast<float4 *>(smem + po);
    for (int k = tid; k < np; k += NT) pos_s[k] = V.pos_f[k];
    pos = pos_s;
  }
  __syncthreads();
  const PairTabF T{bin_s, zl_s, cf_lds ? cf_s : (const float *)t.coef_f, rec_s, nbin, V.nlsem,
                   (float)t.rcut2};
  const float L0 = V.cg.L[0], L1 = V.cg.L[1], L2 = V.cg.L[2];
  const float H0 = V.cg.L2[0], H1 = V.cg.L2[1], H2 = V.cg.L2[2];
  const unsigned *__restrict__ nbr = reinterpret_cast<const unsigned *>((const int *)V.nbr);
  const int maxrow = V.maxnn - 1;
  const bool pos64 = V.pair_pos64 != 0;
  double vir = 0.0;
  int err = 0;
  for (int base = 0; base < np; base += NT) {
    const int tt = base + tid;
    double ej[NTY];
#pragma unroll
    for (int k = 0; k < NTY; ++k) ej[k] = 0.0;
    int ti = 0;
    if (tt < np) {
      // boxes with an axis of fewer than three list cells: separations in
      // FP64 from the cell-ordered positions (as k_pair_f's POS64 variant)
      const float4 pi = pos64 ? make_float4(0.f, 0.f, 0.f, __int_as_float(V.type_s[tt]))
                              : pos[tt];
      const double xi = pos64 ? V.ro_s[3 * tt] : 0.0, yi = pos64 ? V.ro_s[3 * tt + 1] : 0.0,
                   zi = pos64 ? V.ro_s[3 * tt + 2] : 0.0;
      const int n = V.nn[tt];
      ti = __float_as_int(pi.w);
      unsigned long long ptp = 0;
      for (int u = 0; u < npt; ++u) ptp |= (unsigned long long)pidx_s[ti * npt + u] << (8 * u);
      KahanF fxf, fyf, fzf;
      // the indices of the next two batches are in flight while this one
      // is evaluated (lists of tens of partners: the list loads, not the
      // arithmetic, would otherwise set the pace)
      unsigned en[kPairBatch], en2[kPairBatch];
#pragma unroll
      for (int q = 0; q < kPairBatch; ++q) en[q] = nbr[(size_t)min(q, maxrow) * np + tt];
#pragma unroll
      for (int q = 0; q < kPairBatch; ++q)
        en2[q] = nbr[(size_t)min(kPairBatch + q, maxrow) * np + tt];
      for (int k0 = 0; k0 < n; k0 += kPairBatch) {
        unsigned es[kPairBatch];
        float4 ps[kPairBatch];
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q) {
          es[q] = en[q];
          en[q] = en2[q];
        }
        if (pos64) {
#pragma unroll
          for (int q = 0; q < kPairBatch; ++q) {
            const int j = k0 + q < n ? (int)(es[q] & kNbrIdxMask) : tt;
            double ddx = xi - V.ro_s[3 * j], ddy = yi - V.ro_s[3 * j + 1],
                   ddz = zi - V.ro_s[3 * j + 2];
            pbcr2(ddx, ddy, ddz, V.box);
            ps[q] = make_float4((float)ddx, (float)ddy, (float)ddz, __int_as_float(V.type_s[j]));
          }
        } else {
#pragma unroll
          for (int q = 0; q < kPairBatch; ++q)
            ps[q] = pos[k0 + q < n ? (int)(es[q] & kNbrIdxMask) : tt];
        }
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q)
          en2[q] = nbr[(size_t)min(k0 + 2 * kPairBatch + q, maxrow) * np + tt];
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q) {
          if (k0 + q >= n) break;
          float dx, dy, dz;
          if (pos64) {
            dx = ps[q].x;
            dy = ps[q].y;
            dz = ps[q].z;
          } else {
            const float4 o4 = off_s[es[q] >> kNbrCodeShift];
            dx = (pi.x - ps[q].x) + o4.x;
            dy = (pi.y - ps[q].y) + o4.y;
            dz = (pi.z - ps[q].z) + o4.z;
            if (fabsf(dx) > H0) dx -= copysignf(L0, dx);
            if (fabsf(dy) > H1) dy -= copysignf(L1, dy);
            if (fabsf(dz) > H2) dz -= copysignf(L2, dz);
          }
          const int tj = __float_as_int(ps[q].w);
          const int p = (int)((ptp >> (8 * tj)) & 0xffu);
          float fs, r2;
          double usum;
          if (!pair_eval_f<false>(V, T, dx, dy, dz, p, energy, fs, usum, r2, err)) continue;
          fxf.add(fs * dx);
          fyf.add(fs * dy);
          fzf.add(fs * dz);
          if (energy) {
#pragma unroll
            for (int k2 = 0; k2 < NTY; ++k2) ej[k2] += (k2 == tj) ? 0.5 * usum : 0.0;
            vir -= 0.5 * (double)(fs * r2);
          }
        }
      }
      const int io = V.c_sorted[tt];
      V.force[3 * io] = fxf.value();
      V.force[3 * io + 1] = fyf.value();
      V.force[3 * io + 2] = fzf.value();
    }
    if (energy) {
      for (int k = 0; k < P; ++k) {
        double v = 0.0;
        if (tt < np) {
#pragma unroll
          for (int u = 0; u < NTY; ++u)
            if (u < npt && pidx_s[ti * npt + u] == k) v += ej[u];
        }
        for (int w = 32; w > 0; w >>= 1) v += __shfl_down(v, w, 64);
        if (lane == 0) wred[wave][k] += v;
      }
    }
  }
  if (err) atomicOr(&V.flags[0], err);
  for (int w = 32; w > 0; w >>= 1) vir += __shfl_down(vir, w, 64);
  if (lane == 0) wred[wave][P] = vir;
  __syncthreads();
}

// spreading, slab by slab of z planes in LDS: each slab's points are
// accumulated in exact fixed point (LDS 64-bit adds) from every particle
// whose stencil reaches it -- the points m, m-1, ..., m-order+1 from
// meshmax m per axis (Src/energy.F90:1223-1246), each product q wz wy wx
// in FP32 as k_spread forms it -- and then stored, rounded to FP32, into
// the real mesh (the x pass reads it there)
template <int ORDER>
MFE_STAGE void p_spread(const SysDev &V, char *smem, int lds) {
  typedef SpreadAcc<float>::T Acc;
  const int tid = threadIdx.x, NT = blockDim.x, np = V.np;
  const SpmeGeom g = V.sg;
  const int s1 = g.s[0], s2 = g.s[1], s3 = g.s[2];
  const int plane = s1 * s2;
  const int nzs = max(1, min(s3, lds / (plane * (int)sizeof(Acc))));
  Acc *slab = reinterpret_cast<Acc *>(smem);
  float *__restrict__ mesh = (float *)V.mesh_r;
  for (int z0 = 0; z0 < s3; z0 += nzs) {
    const int nz = min(nzs, s3 - z0);
    for (int k = tid; k < nz * plane; k += NT) slab[k] = Acc(0);
    __syncthreads();
    for (int i = tid; i < np; i += NT) {
      int mm[3];
      double fr[3];
      mesh_coords(V.ro + 3 * i, g, mm, fr);
      // stencil planes mm2, mm2-1, ... (mod s3) inside the slab
      bool any = false;
#pragma unroll
      for (int iz = 0; iz < ORDER; ++iz) {
        const int z = mm[2] - iz < 0 ? mm[2] - iz + s3 : mm[2] - iz;
        any |= (unsigned)(z - z0) < (unsigned)nz;
      }
      if (!any) continue;
      float wx[ORDER], wy[ORDER], wz[ORDER];
      bspline<float, ORDER>((float)fr[0], wx, nullptr);
      bspline<float, ORDER>((float)fr[1], wy, nullptr);
      bspline<float, ORDER>((float)fr[2], wz, nullptr);
      const float q = (float)V.q[i];
#pragma unroll
      for (int iz = 0; iz < ORDER; ++iz) {
        const int z = mm[2] - iz < 0 ? mm[2] - iz + s3 : mm[2] - iz;
        if ((unsigned)(z - z0) >= (unsigned)nz) continue;
        const float qz = q * wz[iz];
#pragma unroll
        for (int iy = 0; iy < ORDER; ++iy) {
          const int y = mm[1] - iy < 0 ? mm[1] - iy + s2 : mm[1] - iy;
          const float qyz = qz * wy[iy];
          Acc *row = slab + ((z - z0) * s2 + y) * s1;
#pragma unroll
          for (int ix = 0; ix < ORDER; ++ix) {
            const int x = mm[0] - ix < 0 ? mm[0] - ix + s1 : mm[0] - ix;
            SpreadAcc<float>::add(&row[x], qyz * wx[ix], kSplineScale<ORDER, 0>);
          }
        }
      }
    }
    __syncthreads();
    float *out = mesh + (size_t)z0 * plane;
    for (int k = tid; k < nz * plane; k += NT) out[k] = SpreadAcc<float>::get(slab[k]);
    __syncthreads();
  }
}

// the five FFT passes of the replica's mesh (one function per pass), each
// over as many rows, planes or lines as the lds bytes of LDS hold; the
// convolution's energy and virial terms of this thread into esum, vsum
constexpr int kCplxF = (int)sizeof(cplx<float>), kTwF = (int)sizeof(Twiddle<float>);
__device__ __forceinline__ int persist_rows(const SysDev &V, int lds) {
  const int m = V.sg.s[0] / 2;
  return max(1, (lds - (m + V.sg.s[0]) * kTwF) / (2 * (m + 1) * kCplxF));
}
__device__ __forceinline__ int persist_planes(const SysDev &V, int lds) {
  return max(1, (lds - V.sg.s[1] * kTwF) / (2 * V.hx * (V.sg.s[1] + 1) * kCplxF));
}
__device__ __forceinline__ int persist_lines(const SysDev &V, int lds) {
  return max(1, (lds - V.sg.s[2] * kTwF) / (2 * V.hx * (V.sg.s[2] + 1) * kCplxF));
}
MFE_STAGE void p_fftx_fwd(const SysDev &V, char *smem, int lds) {
  const int s1 = V.sg.s[0], s2 = V.sg.s[1], nrows = V.sg.s[1] * V.sg.s[2];
  const int cap = persist_rows(V, lds);
  const float *__restrict__ mesh = (const float *)V.mesh_r;
  for (int row0 = 0; row0 < nrows; row0 += cap) {
    fftx_fwd_rows<float>(V, row0, min(cap, nrows - row0), cap, smem, [&](int x, int y, int z) {
      return mesh[((size_t)z * s2 + y) * s1 + x];
    });
    __syncthreads();
  }
}
MFE_STAGE void p_ffty(const SysDev &V, int inv, char *smem, int lds) {
  const int s3 = V.sg.s[2], cap = persist_planes(V, lds);
  for (int z0 = 0; z0 < s3; z0 += cap) {
    ffty_planes<float>(V, z0, min(cap, s3 - z0), inv, smem);
    __syncthreads();
  }
}
MFE_STAGE void p_fftconv(const SysDev &V, int energy, char *smem, int lds, double *esum,
                         double *vsum) {
  const int s2 = V.sg.s[1], cap = persist_lines(V, lds);
  double e = 0.0, v = 0.0;
  for (int y0 = 0; y0 < s2; y0 += cap) {
    fftconv_lines<float>(V, y0, min(cap, s2 - y0), energy, smem, e, v);
    __syncthreads();
  }
  *esum = e;
  *vsum = v;
}
MFE_STAGE void p_fftx_inv(const SysDev &V, char *smem, int lds) {
  const int nrows = V.sg.s[1] * V.sg.s[2], cap = persist_rows(V, lds);
  for (int row0 = 0; row0 < nrows; row0 += cap) {
    fftx_inv_rows<float>(V, row0, min(cap, nrows - row0), cap, smem);
    __syncthreads();
  }
}

// gather (CalcProp, Src/energy.F90:1259-1285) in particle order, then
// BDStep's forceo (fin_apply, UTotal's scaling)
template <int ORDER>
MFE_STAGE void p_gather(const SysDev &V, char *smem, int lds) {
  const int tid = threadIdx.x, NT = blockDim.x, np = V.np;
  const SpmeGeom g = V.sg;
  const int s1 = g.s[0], s2 = g.s[1], s3 = g.s[2];
  // particle i's field from the convolved mesh read through rd
  auto one = [&](int i, auto rd) {
    int mm[3];
    double fr[3];
    mesh_coords(V.ro + 3 * i, g, mm, fr);
    float v[3][ORDER], dv[3][ORDER];
    bspline<float, ORDER>((float)fr[0], v[0], dv[0]);
    bspline<float, ORDER>((float)fr[1], v[1], dv[1]);
    bspline<float, ORDER>((float)fr[2], v[2], dv[2]);
    Acc3<float> ac;
#pragma unroll
    for (int iz = 0; iz < ORDER; ++iz) {
      const int z = mm[2] - iz < 0 ? mm[2] - iz + s3 : mm[2] - iz;
      const float vz = v[2][iz], dz = dv[2][iz];
#pragma unroll
      for (int iy = 0; iy < ORDER; ++iy) {
        const int y = mm[1] - iy < 0 ? mm[1] - iy + s2 : mm[1] - iy;
        const int row = (z * s2 + y) * s1;
        float sx = 0.f, sdx = 0.f;
#pragma unroll
        for (int ix = 0; ix < ORDER; ++ix) {
          const int x = mm[0] - ix < 0 ? mm[0] - ix + s1 : mm[0] - ix;
          const float qv = rd(row + x);
          sx += v[0][ix] * qv;
          sdx += dv[0][ix] * qv;
        }
        ac.add(0, sdx * (v[1][iy] * vz));
        ac.add(1, sx * (dv[1][iy] * vz));
        ac.add(2, sx * (v[1][iy] * dz));
      }
    }
    const double qd = (double)(float)V.q[i];
    constexpr double kScale = kSplineScale<ORDER, 1>;
    const double fld[3] = {-(ac.get(0) * kScale) * g.dkdr[0] * V.efp,
                           -(ac.get(1) * kScale) * g.dkdr[1] * V.efp,
                           -(ac.get(2) * kScale) * g.dkdr[2] * V.efp};
    double ft[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) ft[m] = V.force[3 * i + m] + qd * fld[m];
#pragma unroll
    for (int m = 0; m < 3; ++m) V.force[3 * i + m] = ft[m];
    FinState st;
    fin_load(V, i, 0, st);
    const double es[3] = {0.0, 0.0, 0.0};
    fin_apply(V, i, ft, st, 0, 0.0, es);
  };
  const int M = s1 * s2 * s3;
  const float *__restrict__ mesh = (const float *)V.mesh_r;
  if ((size_t)M * sizeof(float) <= (size_t)lds) {
    // the convolved mesh staged in LDS (one pass over it), every stencil
    // read from there
    float *m_s = reinterpret_cast<float *>(smem);
    for (int k = tid; k < M; k += NT) m_s[k] = mesh[k];
    __syncthreads();
    for (int i = tid; i < np; i += NT) one(i, [&](int k) { return m_s[k]; });
    __syncthreads();
  } else {
    for (int i = tid; i < np; i += NT) one(i, [&](int k) { return mesh[k]; });
  }
}

// the gated list rebuild (the phases of k_rebuild with workgroup barriers)
MFE_STAGE void p_rebuild(const SysDev &V, int *wi) {
  const int tid = threadIdx.x, NT = blockDim.x;
  const int nc = V.cg.ncells;
  for (int k = tid; k < nc; k += NT) V.c_count[k] = 0;
  __syncthreads();
  ph_cell_count(V, tid, NT);
  __syncthreads();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  block_scan_counts(V.c_count, V.c_start, nc, wi);
  __syncthreads();
  ph_cell_scatter(V, tid, NT, nullptr);
  __syncthreads();
  ph_cell_rank(V, tid, NT);
  __syncthreads();
  ph_nlist_build(V, tid, NT, 0);
  if (tid == 0) V.flags[2] += 1;
  __syncthreads();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}
#undef MFE_STAGE

template <int ORDER>
__device__ void persist_replica(const SysDev &V, int nsteps, int energy, char *smem, int lds,
                                double (*wred)[40], double *wm, int *wi) {
  const int tid = threadIdx.x, nw = blockDim.x >> 6;
  const int lane = tid & 63, wave = tid >> 6;
  const int P = V.tab.nptpt;
  __shared__ PairRecF rec_s[MFE_MAX_PAIRS];
  __shared__ int pidx_s[MFE_MAX_TYPES * MFE_MAX_TYPES];
  __shared__ float4 off_s[125];
  __shared__ int flag_s;
  unsigned stepctr = (unsigned)V.flags[3];
  for (int step = 0; step < nsteps; ++step) {
    const int rebuild = p_move_skin(V, stepctr, wm, &flag_s);
    const int npt = V.tab.npt;
    size_t po = 0;
    if (pair_pos_in_lds(V, lds, po)) {
      if (npt <= 2) p_pair<2, true>(V, energy, smem, lds, wred, rec_s, pidx_s, off_s);
      else if (npt <= 4) p_pair<4, true>(V, energy, smem, lds, wred, rec_s, pidx_s, off_s);
      else p_pair<MFE_MAX_TYPES, true>(V, energy, smem, lds, wred, rec_s, pidx_s, off_s);
    } else {
      if (npt <= 2) p_pair<2, false>(V, energy, smem, lds, wred, rec_s, pidx_s, off_s);
      else if (npt <= 4) p_pair<4, false>(V, energy, smem, lds, wred, rec_s, pidx_s, off_s);
      else p_pair<MFE_MAX_TYPES, false>(V, energy, smem, lds, wred, rec_s, pidx_s, off_s);
    }
    p_spread<ORDER>(V, smem, lds);
    double esum = 0.0, vsum = 0.0;
    p_fftx_fwd(V, smem, lds);
    p_ffty(V, 0, smem, lds);
    p_fftconv(V, energy, smem, lds, &esum, &vsum);
    p_ffty(V, 1, smem, lds);
    p_fftx_inv(V, smem, lds);
    p_gather<ORDER>(V, smem, lds);
    // ---- reductions (ph_reduce's energy terms)
    for (int w = 32; w > 0; w >>= 1) {
      esum += __shfl_down(esum, w, 64);
      vsum += __shfl_down(vsum, w, 64);
    }
    if (lane == 0) {
      wred[wave][P + 1] = esum;
      wred[wave][P + 2] = vsum;
    }
    __syncthreads();
    if (tid == 0) {
      int *flags = V.flags;
      double *en = V.en;
      flags[3] = (int)(stepctr + 1u);
      for (int m = 0; m < 3; ++m) en[5 + m] = 0.0;
      if (energy) {
        // each component's wavefront partials in wavefront order
        auto total = [&](int k) {
          double sacc = wred[0][k];
          for (int w = 1; w < nw; ++w) sacc += wred[w][k];
          return sacc;
        };
        double twob0 = 0.0;
        for (int k = 0; k < P; ++k) {
          const double u = total(k);
          en[8 + k] = u;
          twob0 += u;
        }
        const double urec = total(P + 1) + V.self_energy + V.net_energy;
        const double virrec = total(P + 2) - 3.0 * V.net_energy;
        const double rec = V.efp * urec;
        en[0] = twob0 + rec;
        en[1] = twob0;
        en[2] = rec;
        en[3] = 0.0;
        en[4] = total(P) + V.efp * virrec;
        en[kEnAngle] = 0.0;
      }
      flags[1] = 0;
    }
    ++stepctr;
    __syncthreads();
    // ---- the gated list rebuild (SetVListMD after NList's test)
    if (rebuild) p_rebuild(V, wi);
  }
}

template <int ORDER>
__global__ void __launch_bounds__(kPersistThreads) __attribute__((amdgpu_waves_per_eu(4)))
k_bd_persistent(PersistArgs a) {
  extern __shared__ __align__(16) char smem[];
  __shared__ int r_s;
  __shared__ double wred[kPersistThreads / 64][40];
  __shared__ double wm[kPersistThreads / 64];
  __shared__ int wi[kPersistThreads / 64];
  for (;;) {
    if (threadIdx.x == 0) r_s = atomicAdd(a.queue, 1);
    __syncthreads();
    const int rr = r_s;
    __syncthreads();
    if (rr >= a.nrep) return;
    const int r = a.order[rr];
    persist_replica<ORDER>(a.sys[r], a.nsteps, a.energy, smem, a.lds, wred, wm, wi);
  }
}

inline int nblocks(int n) { return (n + kBlock - 1) / kBlock; }

inline dim3 grid(int x, const Group &g, int y = 1) { return dim3(x > 0 ? x : 1, y, g.R); }

}  // namespace

template <typename R, int O>
const void *k_spread_ptr() {
  return (const void *)&k_spread<R, O>;
}
template <typename R, int O>
const void *k_gather_ptr(int mode, bool fin) {
  if (fin) return (const void *)&k_gather<R, O, GM_FORCE, true>;
  switch (mode) {
    case GM_POT: return (const void *)&k_gather<R, O, GM_POT, false>;
    case GM_FIELD: return (const void *)&k_gather<R, O, GM_FIELD, false>;
    case GM_POTONLY: return (const void *)&k_gather<R, O, GM_POTONLY, false>;
    default: return (const void *)&k_gather<R, O, GM_FORCE, false>;
  }
}

void philox4x32(const uint32_t ctr[4], const uint32_t key[2], uint32_t out[4]) {
  for (int k = 0; k < 4; ++k) out[k] = ctr[k];
  philox10(out, key[0], key[1]);
}

void launch_fill_int(int *p, int n, int v, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_fill_int, dim3(nblocks(n)), dim3(kBlock), 0, s, p, n, v);
}
void launch_fill_double(double *p, int n, double v, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(k_fill_double, dim3(nblocks(n)), dim3(kBlock), 0, s, p, n, v);
}

void launch_nlist_rebuild(const Group &g, bool gated) {
  if (gated && g.R == 1 && g.rebuild_bar && g.flags && g.ncu > 0) {
    hipLaunchKernelGGL(k_rebuild, dim3(g.ncu), dim3(1024), 0, g.stream, g.d, g.flags,
                       g.rebuild_bar, g.sync_spin >= 0 ? g.sync_spin : kGridSpin);
    return;
  }
  // gated kernels run on small grids (grid-stride loops): when the skin
  // test does not fire they cost one dispatch of a few hundred wavefronts
  const int gb = gated ? std::min(g.np_blocks, 256) : g.np_blocks;
  const int gl = gated ? std::min(g.list_blocks, 1024) : g.list_blocks;
  const int gs = gated && g.R > 1 ? 16 : kScanBlocks;
  const int gt = gated ? 1 : 0;
  hipLaunchKernelGGL(k_cell_count, grid(gb, g), dim3(kBlock), 0, g.stream, g.d, gt);
  hipLaunchKernelGGL(k_cell_scan, grid(gs, g), dim3(1024), 0, g.stream, g.d, gt);
  hipLaunchKernelGGL(k_cell_scatter, grid(gb, g), dim3(kBlock), 0, g.stream, g.d, gt);
  hipLaunchKernelGGL(k_cell_rank, grid(gb, g), dim3(kBlock), 0, g.stream, g.d, gt);
  hipLaunchKernelGGL(k_nlist_build, grid(gl, g), dim3(kBlock), 0, g.stream, g.d, gt);
}

void launch_sort_pos(const Group &g) {
  hipLaunchKernelGGL(k_sort_pos, grid(g.np_blocks, g), dim3(kBlock), 0, g.stream, g.d);
}

void launch_mc_place(const Group &g, int natm, const int *ia, const double *rtm,
                     double *ro_stage) {
  hipLaunchKernelGGL(k_mc_place, dim3((natm + 255) / 256), dim3(256), 0, g.stream, natm, ia, rtm,
                     ro_stage);
}

// points per thread, blocks, moved particles whose factors a block holds at a
// time (as many as 32 KB of LDS take beside the roots) and dynamic LDS of a
// pass over the spectrum
struct McPass {
  int P, nb, chunk;
  size_t lds;
};
static McPass mc_plan(const Group &g, int natm, bool table) {
  const int hx = g.mc_s[0] / 2 + 1;
  const size_t n = (size_t)hx * g.mc_s[1] * g.mc_s[2];
  McPass p;
  p.P = table && n < 256 * 256 * kMcPoints ? 1 : kMcPoints;
  p.nb = (int)std::min<size_t>((n + 256 * p.P - 1) / (256 * p.P), kMcRecBlocks);
  const size_t per = 2 * (size_t)(hx + mc_rows(hx, p.P)) * sizeof(double2);
  p.chunk = (int)std::max<size_t>(1, std::min<size_t>(natm, (32 * 1024) / per));
  p.lds = p.chunk * per;
  if (!table) p.lds += (size_t)(g.mc_s[0] + g.mc_s[1] + g.mc_s[2]) * sizeof(double2);
  return p;
}

void allow_lds(const void *kernel, size_t lds) {
  if (lds > 60 * 1024)
    (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

// the instance of the engine's precision and spline order
#define MFE_MC_CASES(T)                                                          \
  switch (g.order) {                                                             \
    MFE_MC(T, 3) MFE_MC(T, 4) MFE_MC(T, 5) MFE_MC(T, 6) MFE_MC(T, 7) MFE_MC(T, 8) \
  }

int mc_table_min() { return kMcTable; }

int launch_mc_rec(const Group &g, const McMove &mv, void *spec, double *old, void *fac,
                  double *part) {
  const McPass p = mc_plan(g, mv.natm, fac != nullptr);
  const int ns = g.mc_s[0] + g.mc_s[1] + g.mc_s[2];
  const int nf = (int)std::min(((long long)mv.natm * 2 * ns + 255) / 256, 1024ll);
  double2 *f2 = (double2 *)fac, *s2 = (double2 *)spec;
#define MFE_MC(T, O)                                                                        \
  case O:                                                                                   \
    if (fac) {                                                                              \
      hipLaunchKernelGGL((k_mc_fac<T, O>), dim3(nf), dim3(256), ns * sizeof(double2),       \
                         g.stream, g.d, mv, f2);                                            \
      break;                                                                                \
    }                                                                                       \
    allow_lds((const void *)k_mc_rec<T, O>, p.lds);                                      \
    hipLaunchKernelGGL((k_mc_rec<T, O>), dim3(p.nb), dim3(256), p.lds, g.stream, g.d, mv,   \
                       p.chunk, s2, old, part);                                             \
    break;
  if (g.prec == MFE_PREC_MIXED) { MFE_MC_CASES(float) }
  else { MFE_MC_CASES(double) }
#undef MFE_MC
  if (fac && p.P == 1)
    hipLaunchKernelGGL(k_mc_tab<1>, dim3(p.nb), dim3(256), p.lds, g.stream, g.d, mv.natm,
                       p.chunk, s2, (const double2 *)f2, part);
  else if (fac)
    hipLaunchKernelGGL(k_mc_tab<kMcPoints>, dim3(p.nb), dim3(256), p.lds, g.stream, g.d,
                       mv.natm, p.chunk, s2, (const double2 *)f2, part);
  return p.nb;
}

void launch_mc_accept(const Group &g, const McMove &mv, bool place, void *spec, double *old,
                      const void *fac) {
  const McPass p = spec ? mc_plan(g, mv.natm, fac != nullptr) : McPass{kMcPoints, 0, 1, 0};
  const int nset = place ? g.np_blocks : 0, nb = nset + p.nb;
  if (!nb) return;
  double2 *s2 = (double2 *)spec;
  if (spec && fac) {
    const double2 *f2 = (const double2 *)fac;
    if (p.P == 1)
      hipLaunchKernelGGL(k_mc_accept_tab<1>, dim3(nb), dim3(kBlock), p.lds, g.stream, g.d, mv,
                         nset, p.chunk, s2, f2);
    else
      hipLaunchKernelGGL(k_mc_accept_tab<kMcPoints>, dim3(nb), dim3(kBlock), p.lds, g.stream,
                         g.d, mv, nset, p.chunk, s2, f2);
    return;
  }
#define MFE_MC(T, O)                                                                       \
  case O:                                                                                  \
    allow_lds((const void *)k_mc_accept<T, O>, p.lds);                                  \
    hipLaunchKernelGGL((k_mc_accept<T, O>), dim3(nb), dim3(kBlock), p.lds, g.stream, g.d,  \
                       mv, nset, p.chunk, s2, old);                                        \
    return;
  if (spec && g.prec == MFE_PREC_MIXED) { MFE_MC_CASES(float) }
  else if (spec) { MFE_MC_CASES(double) }
  // without a spectrum any instance places the move
  switch (4) { MFE_MC(double, 4) }
#undef MFE_MC
}
#undef MFE_MC_CASES

void launch_mc_pair(const Group &g, const McMove &mv, double *out, double *part, bool all) {
  if (!all) {
    hipLaunchKernelGGL(k_mc_pair, grid(1, g), dim3(256), 0, g.stream, g.d, mv, out, part);
    return;
  }
  hipLaunchKernelGGL(k_mc_pair, dim3(kMcPairBlocks), dim3(256), 0, g.stream, g.d, mv, out, part);
  hipLaunchKernelGGL(k_mc_pair_sum, dim3(1), dim3(64), 0, g.stream, part, kMcPairBlocks, out);
}

void launch_pair(const Group &g, bool energy, bool sort_pos, bool skin) {
  if (sort_pos)
    hipLaunchKernelGGL(k_sort_pos, grid(g.np_blocks, g), dim3(kBlock), 0, g.stream, g.d);
  const int pgrid = std::max(g.pair_blocks, 1);
  const dim3 gr = grid(pgrid + (skin ? (g.np_blocks + 1) / 2 : 0), g);
  const int e1 = energy ? 1 : 0, s1 = skin ? 1 : 0;
#define MFE_PAIR(NT, CF)                                                                  \
  hipLaunchKernelGGL((k_pair<NT, CF>), gr, dim3(kPairBlock), g.lds_pair, g.stream, g.d, e1, \
                     pgrid, s1)
#define MFE_PAIR_CF(NT) \
  do { if (g.pair_cf_lds) MFE_PAIR(NT, true); else MFE_PAIR(NT, false); } while (0)
  // the skin blocks ride on the first of the (one or two) launches; the
  // second has no blocks beyond pgrid
  const dim3 gr0 = grid(pgrid, g);
#define MFE_PAIRF(NT, CF, KN, P64, GR, SK)                                                 \
  hipLaunchKernelGGL((k_pair_f<NT, CF, KN, P64>), GR, dim3(kPairBlock), g.lds_pair, g.stream, \
                     g.d, e1, pgrid, SK)
#define MFE_PAIRF_LN(NT, CF, KN)                                         \
  do {                                                                   \
    if (g.pair_any32) MFE_PAIRF(NT, CF, KN, false, gr, s1);              \
    if (g.pair_any64) {                                                  \
      if (g.pair_any32) MFE_PAIRF(NT, CF, KN, true, gr0, 0);             \
      else MFE_PAIRF(NT, CF, KN, true, gr, s1);                          \
    }                                                                    \
  } while (0)
#define MFE_PAIRF_KN(NT, CF) \
  do { if (g.knots) MFE_PAIRF_LN(NT, CF, true); else MFE_PAIRF_LN(NT, CF, false); } while (0)
#define MFE_PAIRF_CF(NT) \
  do { if (g.pair_cf_lds) MFE_PAIRF_KN(NT, true); else MFE_PAIRF_KN(NT, false); } while (0)
  const int nt = g.pair_npt;
  if (g.prec == MFE_PREC_MIXED) {
    if (nt <= 3) MFE_PAIRF_CF(3);
    else if (nt <= 4) MFE_PAIRF_CF(4);
    else MFE_PAIRF_CF(8);
  } else {
    if (nt <= 3) MFE_PAIR_CF(3);
    else if (nt <= 4) MFE_PAIR_CF(4);
    else MFE_PAIR_CF(8);
  }
#undef MFE_PAIRF_CF
#undef MFE_PAIRF_KN
#undef MFE_PAIRF_LN
#undef MFE_PAIRF
#undef MFE_PAIR_CF
#undef MFE_PAIR
}

template <typename R>
static void spme_stages(const Group &g, bool energy, int first, int last, int gmode,
                        const FinArgs *fin) {
  for (int st = first; st <= last; ++st) {
    switch (st) {
      case SP_BIN:
        // counts, the last count block's scan, records
        hipLaunchKernelGGL(k_spme_count,
                           grid((g.np_blocks * kBlock + kCountThreads - 1) / kCountThreads, g),
                           dim3(kCountThreads), 0, g.stream, g.d);
        hipLaunchKernelGGL(k_spme_scatter<R>, grid(g.np_blocks, g), dim3(kBlock), 0, g.stream,
                           g.d);
        if (last == SP_BIN)
          hipLaunchKernelGGL(k_spme_clear, grid((g.bricks + kBlock - 1) / kBlock, g), dim3(kBlock),
                             0, g.stream, g.d);
        break;
      case SP_SPREAD:
        switch (g.order) {
#define MFE_SPREAD(O)                                                                   \
  case O:                                                                               \
    hipLaunchKernelGGL((k_spread<R, O>), grid(g.bricks, g), dim3(kSpreadThreads),          \
                       g.lds_spread,                                                    \
                       g.stream, g.d);                                                  \
    break;
          MFE_SPREAD(3) MFE_SPREAD(4) MFE_SPREAD(5) MFE_SPREAD(6) MFE_SPREAD(7) MFE_SPREAD(8)
#undef MFE_SPREAD
        }
        break;
      case SP_FFTX: fft_x_forward(g); break;
      case SP_FFTY: fft_y(g, 0); break;
      case SP_CONV: fft_conv(g, energy); break;
      case SP_IFFTY: fft_y(g, 1); break;
      case SP_IFFTX: fft_x_inverse(g); break;
      case SP_GATHER: {
        const FinArgs fa = fin ? *fin : FinArgs{0, 0, 0, 0, 0.0};
        switch (g.order) {
#define MFE_GATHER(O)                                                                   \
  case O:                                                                               \
    if (fin)                                                                            \
      hipLaunchKernelGGL((k_gather<R, O, GM_FORCE, true>), grid(g.bricks + 1, g),       \
                         dim3(kGatherLanes), g.lds_gather, g.stream, g.d, fa);          \
    else if (gmode == GM_POT)                                                           \
      hipLaunchKernelGGL((k_gather<R, O, GM_POT, false>), grid(g.bricks, g),            \
                         dim3(kGatherLanes), g.lds_gather, g.stream, g.d, fa);          \
    else if (gmode == GM_FIELD)                                                         \
      hipLaunchKernelGGL((k_gather<R, O, GM_FIELD, false>), grid(g.bricks, g),          \
                         dim3(kGatherLanes), g.lds_gather, g.stream, g.d, fa);          \
    else if (gmode == GM_POTONLY)                                                       \
      hipLaunchKernelGGL((k_gather<R, O, GM_POTONLY, false>), grid(g.bricks, g),        \
                         dim3(kGatherLanes), g.lds_gather, g.stream, g.d, fa);          \
    else                                                                                \
      hipLaunchKernelGGL((k_gather<R, O, GM_FORCE, false>), grid(g.bricks, g),          \
                         dim3(kGatherLanes), g.lds_gather, g.stream, g.d, fa);          \
    break;
          MFE_GATHER(3) MFE_GATHER(4) MFE_GATHER(5) MFE_GATHER(6) MFE_GATHER(7) MFE_GATHER(8)
#undef MFE_GATHER
        }
        break;
      }
    }
  }
}

void launch_spme(const Group &g, bool energy, int first, int last, int gmode,
                 const FinArgs *fin) {
  if (g.prec == MFE_PREC_MIXED) spme_stages<float>(g, energy, first, last, gmode, fin);
  else spme_stages<double>(g, energy, first, last, gmode, fin);
}

void launch_pair_sk(const Group &g, bool energy, bool skin) {
  const int pgrid = std::max(g.pair_blocks, 1);
  const int npb = pgrid + (skin ? (g.np_blocks + 1) / 2 : 0);
  const int e1 = energy ? 1 : 0, s1 = skin ? 1 : 0;
  const int nt = g.pair_npt <= 3 ? 3 : (g.pair_npt <= 4 ? 4 : 8);
#define MFE_PSK(NT, P64)                                                                   \
  hipLaunchKernelGGL((k_pair_sk<NT, P64>), grid(npb + g.kvec, g), dim3(kPairBlock),        \
                     g.lds_pair, g.stream, g.d, e1, pgrid, s1, npb)
#define MFE_PSK_NT(P64)          \
  if (nt == 3) MFE_PSK(3, P64);  \
  else if (nt == 4) MFE_PSK(4, P64); \
  else MFE_PSK(8, P64);
  if (g.pair_any64) { MFE_PSK_NT(true) }
  else { MFE_PSK_NT(false) }
#undef MFE_PSK_NT
#undef MFE_PSK
}

void launch_std_factors(const Group &g) {
  hipLaunchKernelGGL(k_ewald_sk, grid(g.kvec, g), dim3(kSkThreads), 0, g.stream, g.d, 1);
}

void launch_std_forces(const Group &g) {
  const dim3 gr = grid((g.np_blocks * kBlock + kEwParticles - 1) / kEwParticles, g);
  const size_t lds = (size_t)kEwParticles * 3 * (g.ncut + 1) * sizeof(double2);
  if (lds <= 64 * 1024)
    hipLaunchKernelGGL(k_ewald_force<true>, gr, dim3(64 * kEwParticles), lds, g.stream, g.d);
  else
    hipLaunchKernelGGL(k_ewald_force<false>, gr, dim3(64 * kEwParticles), 0, g.stream, g.d);
}

void launch_bonds(const Group &g) {
  hipLaunchKernelGGL(k_bonds, grid(g.np_blocks, g), dim3(kBlock), 0, g.stream, g.d, 1);
}

void launch_surf(const Group &g) {
  hipLaunchKernelGGL(k_surf_sum, grid(g.np_blocks, g), dim3(kBlock), 0, g.stream, g.d);
}

void launch_reduce(const Group &g, unsigned flags, bool skin, bool bd) {
  const int energy = (flags & (MFE_ENERGY | MFE_VIRIAL)) ? 1 : 0;
  hipLaunchKernelGGL(k_reduce, grid(1, g), dim3(kReduceThreads), 0, g.stream, g.d, energy,
                     skin ? 1 : 0, bd ? 1 : 0);
}

void launch_reduce_finalize(const Group &g, unsigned flags, bool skin, bool bd, int mode,
                            double dt, bool split) {
  const int energy = (flags & (MFE_ENERGY | MFE_VIRIAL)) ? 1 : 0;
  const int F = (g.np_blocks * kBlock + kReduceThreads - 1) / kReduceThreads;
  hipLaunchKernelGGL(k_reduce_finalize, grid(F + 1, g), dim3(kReduceThreads), 0, g.stream, g.d,
                     energy, skin ? 1 : 0, bd ? 1 : 0, mode, dt, split ? 1 : 0);
}

bool launch_finalize_rebuild(const Group &g, unsigned flags, bool bd, int mode, double dt,
                             bool split, int *hflags) {
  if (!(g.R == 1 && g.rebuild_bar && g.flags && g.ncu > 1)) return false;
  const int energy = (flags & (MFE_ENERGY | MFE_VIRIAL)) ? 1 : 0;
  hipLaunchKernelGGL(k_finalize_rebuild, dim3(g.ncu), dim3(kReduceThreads), 0, g.stream, g.d,
                     energy, bd ? 1 : 0, mode, dt, split ? 1 : 0, g.rebuild_bar,
                     g.sync_spin >= 0 ? g.sync_spin : kGridSpin, hflags);
  return true;
}

// the fused pair + gather launch (Group::fuse_pg)
void launch_pair_gather(const Group &g, bool energy, bool skin) {
  const int pgrid = std::max(g.pair_blocks, 1);
  const int npb = (pgrid + (skin ? (g.np_blocks + 1) / 2 : 0) + 7) / 8 * 8;
  const dim3 gr = grid(npb + g.bricks, g);
  const size_t lds = std::max(g.lds_pair, g.lds_gather);
  const int e1 = energy ? 1 : 0, s1 = skin ? 1 : 0;
  const int nt = g.pair_npt <= 3 ? 3 : (g.pair_npt <= 4 ? 4 : 8);
#define MFE_PG(NT, O)                                                                      \
  hipLaunchKernelGGL((k_pair_gather<NT, O>), gr, dim3(kPairBlock), lds, g.stream, g.d, e1, \
                     pgrid, s1, npb)
#define MFE_PG_NT(O)                \
  case O:                           \
    if (nt == 3) MFE_PG(3, O);      \
    else if (nt == 4) MFE_PG(4, O); \
    else MFE_PG(8, O);              \
    break;
  switch (g.order) {
    MFE_PG_NT(3) MFE_PG_NT(4) MFE_PG_NT(5) MFE_PG_NT(6) MFE_PG_NT(7) MFE_PG_NT(8)
  }
#undef MFE_PG_NT
#undef MFE_PG
}

void launch_finalize(const Group &g, int mode, double dt) {
  hipLaunchKernelGGL(k_finalize, grid(g.np_blocks, g), dim3(kBlock), 0, g.stream, g.d, mode,
                     dt);
}

void launch_move(const Group &g, double dt, int bd) {
  hipLaunchKernelGGL(k_move, grid(g.np_blocks, g), dim3(kBlock), 0, g.stream, g.d, dt, bd);
}

// flags[0..3] and en[0..nen) of every replica into one array each
__global__ void k_collect(const SysDev *__restrict__ sys, int *fl, double *en, int nen) {
  const SysDev &V = sys[blockIdx.z];
  for (int k = threadIdx.x; k < 4; k += blockDim.x) fl[4 * blockIdx.z + k] = V.flags[k];
  for (int k = threadIdx.x; k < nen; k += blockDim.x) en[(size_t)nen * blockIdx.z + k] = V.en[k];
}

// The persistent batched BD launch: blocks workgroups of kPersistThreads
// taking replicas from the queue (zeroed by the fill launch before it).
void launch_bd_persistent(const Group &g, const int *order, int nrep, int nsteps, int energy,
                          int *queue, int blocks, size_t lds) {
  PersistArgs a{g.d, order, nrep, nsteps, energy, queue, (int)lds};
  launch_fill_int(queue, 1, 0, g.stream);
  switch (g.order) {
#define MFE_PERSIST(O)                                                                      \
  case O:                                                                                  \
    hipLaunchKernelGGL(k_bd_persistent<O>, dim3(blocks), dim3(kPersistThreads), lds, g.stream, \
                       a);                                                                 \
    break;
    MFE_PERSIST(3) MFE_PERSIST(4) MFE_PERSIST(5) MFE_PERSIST(6) MFE_PERSIST(7) MFE_PERSIST(8)
#undef MFE_PERSIST
  }
}

// dynamic LDS above the default 64 KB for the persistent launch (the
// attribute only ever grows)
bool persist_allow_lds(int order, size_t bytes) {
  static size_t allowed[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (order < 3 || order > 8) return false;
  if (bytes <= 64 * 1024 || bytes <= allowed[order]) return true;
  const void *f = nullptr;
  switch (order) {
    case 3: f = (const void *)&k_bd_persistent<3>; break;
    case 4: f = (const void *)&k_bd_persistent<4>; break;
    case 5: f = (const void *)&k_bd_persistent<5>; break;
    case 6: f = (const void *)&k_bd_persistent<6>; break;
    case 7: f = (const void *)&k_bd_persistent<7>; break;
    default: f = (const void *)&k_bd_persistent<8>; break;
  }
  if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) !=
      hipSuccess)
    return false;
  allowed[order] = bytes;
  return true;
}

void launch_collect(const Group &g, int *fl, double *en, int nen) {
  hipLaunchKernelGGL(k_collect, grid(1, g), dim3(64), 0, g.stream, g.d, fl, en, nen);
}

// the sums of the spline coefficients
static size_t adjoint_lds(int nk) { return (size_t)std::max(nk, 1) * sizeof(double); }

void launch_adjoint(const Group &g, int np, int npt, int ncol, double *part, double *out,
                    double *dro) {
  const size_t lds = adjoint_lds(ncol - 1 - 2 * npt);
  allow_lds((const void *)k_adjoint, lds);
  hipLaunchKernelGGL(k_adjoint, grid(g.np_blocks * kAdjLanes, g), dim3(kBlock), lds, g.stream,
                     g.d);
  double *zpart = part + (size_t)adjoint_blocks(np) * ncol;
  hipLaunchKernelGGL(k_adjoint_q, grid(g.np_blocks, g), dim3(kBlock), 0, g.stream, g.d, zpart,
                     dro);
  hipLaunchKernelGGL(k_adjoint_sum, dim3((ncol + kSumCols - 1) / kSumCols), dim3(kSumThreads), 0,
                     g.stream, part, adjoint_blocks(np), ncol, out);
  hipLaunchKernelGGL(k_adjoint_sum, dim3((npt + kSumCols - 1) / kSumCols), dim3(kSumThreads), 0,
                     g.stream, zpart, g.np_blocks, npt, out + ncol);
}
int adjoint_blocks(int np) { return (np + kAdjPer - 1) / kAdjPer; }
bool adjoint_fits(int nk) {
  return adjoint_lds(nk) + (kBlock / 64 + 3 * MFE_MAX_TYPES) * sizeof(double) <= kCuLds;
}

void launch_set_positions(const Group &g, const double *ro_new) {
  hipLaunchKernelGGL(k_set_positions, grid(g.np_blocks, g), dim3(kBlock), 0, g.stream, g.d,
                     ro_new);
}

void launch_skin(const Group &g) {
  hipLaunchKernelGGL(k_skin_blocks, grid(g.np_blocks, g), dim3(kBlock), 0, g.stream, g.d);
}

}  // namespace mfe

// Bricks above 64 KB of LDS (meshes whose only divisors >= order-1 are
// large, e.g. 2*23) need the per-kernel dynamic LDS limit raised.
void mfe_allow_big_spread_lds(int prec, int bytes) {
  // the attribute only ever grows (per precision): a smaller brick set up
  // later must not take the room of an earlier, larger one
  static int allowed[2] = {0, 0};
  int &al = allowed[prec == MFE_PREC_MIXED ? 1 : 0];
  if (bytes <= al) return;
  al = bytes;
  // the gather with the finalize phase has static LDS of its own
  const int fin = std::min(bytes, (int)(mfe::kCuLds - mfe::kGatherFinLds));
#define MFE_ATTR(R, O)                                                              \
  (void)hipFuncSetAttribute((const void *)mfe::k_spread_ptr<R, O>(),                 \
                            hipFuncAttributeMaxDynamicSharedMemorySize, bytes);        \
  for (int gm = 0; gm < 4; ++gm)                                                     \
    (void)hipFuncSetAttribute(mfe::k_gather_ptr<R, O>(gm, false),                     \
                              hipFuncAttributeMaxDynamicSharedMemorySize, bytes);      \
  (void)hipFuncSetAttribute(mfe::k_gather_ptr<R, O>(mfe::GM_FORCE, true),             \
                            hipFuncAttributeMaxDynamicSharedMemorySize, fin);          \
  (void)hipFuncSetAttribute(mfe::k_fm_spread_ptr<R, O>(),                             \
                            hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (prec == MFE_PREC_MIXED) {
    MFE_ATTR(float, 3) MFE_ATTR(float, 4) MFE_ATTR(float, 5)
    MFE_ATTR(float, 6) MFE_ATTR(float, 7) MFE_ATTR(float, 8)
  } else {
    MFE_ATTR(double, 3) MFE_ATTR(double, 4) MFE_ATTR(double, 5)
    MFE_ATTR(double, 6) MFE_ATTR(double, 7) MFE_ATTR(double, 8)
  }
#undef MFE_ATTR
}
