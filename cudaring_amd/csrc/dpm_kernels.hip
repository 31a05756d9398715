// dpm_kernels.hip -- gfx950 kernels of the DPM2D vertex engine.
//
// Work decomposition.  Vertices are cut into ring-aligned tiles of at most 64
// vertices (whole rings, one system per tile).  A step launches one workgroup per
// tile with nw wavefronts (the autotuned "waves per tile"):
//   * wave 0, one lane per vertex, does the ring geometry and the shape force:
//     ring perimeters, areas and centres are segmented wave scans, ring
//     neighbours (prev/next vertex, their angles and rest lengths) come from lane
//     shuffles, so the reference's three shape kernels collapse into one pass;
//     it also draws the ring's Philox numbers;
//   * meanwhile waves 1..nw-1 share the interparticle gather (with nw = 1 wave 0
//     does it itself): in loops over the tile's near list, one evaluation per
//     lane (dpm_near.h), in single force calls over the rows of the ELL neighbour
//     list; the partial forces are added through LDS in a fixed order;
//   * wave 0 applies the integrator epilogue (thermostat, kicks, drift,
//     displacement test).
// Neighbour rows and near lists are rebuilt inside the step kernel when the
// system's rebuild flag is set, each tile's by its own workgroup before its
// gather starts.  In the step loops the cells searched are those of the list
// positions (the positions of the system's last rebuild, binned by that rebuild:
// md_cells), so a step is one launch with no binning and no host
// synchronisation; the split FIRE step bins the current positions in a k_bin
// launch before each step kernel.
// This file: list builds, loop starts, reductions, stage kernels, the split FIRE
// step and the moves of rigid and tile-parallel FIRE.  dpm_step.hip holds the step
// kernel, dpm_fire.hip the persistent FIRE kernel, dpm_forces.h what they share.
#include "dpm_forces.h"
#include "dpm_launch.h"
#include "dpm_near.h"

namespace dpm {

// --------------------------------------------------------- neighbours ---
// cell_of, prev_pair, row_insert and build_row live in dpm_rows.h (shared with the adjoint).

// Bin the positions of flagged systems into the cells of this parity.  Thread 0 first bumps
// the RNG call counters of the step and clears the other parity's flags (they were consumed
// by the previous step).
__global__ void k_bin(View V, CellGrid G, int* count, const int* flagCur, const int* anyCur, int* flagOther,
                      int* anyOther, unsigned long long* ctr, int bumpT, int bumpA, int* err) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t == 0) {
    ctr[0] += bumpT;
    ctr[1] += bumpA;
    *anyOther = 0;
  }
  if (t < V.nsys) flagOther[t] = 0;
  if (*anyCur == 0) return;
  if (t >= V.nv) return;
  const int s = V.vsys[t];
  if (!flagCur[s] || G.brute[s]) return;
  const Box B = box_of(V, s);
  int cx, cy;
  cell_of(V.x[t], V.y[t], B, G.ncx[s], G.ncy[s], cx, cy);
  const int c = G.coff[s] + cy * G.ncx[s] + cx;
  const int slot = atomicAdd(&count[c], 1);
  if (slot < G.cap) G.slots[(long)c * G.cap + slot] = t;
  else atomicOr(err, ERR_CELL_OVERFLOW);
}

// Host-driven rebuild of the flagged systems' rows (calcNeighborList / checkNeighbors), one
// workgroup per tile whose waves share the cell search (build_rows_tile), or, without LDS for rows
// of width W (rowsLds = 0) or without cells, one lane per vertex (build_row).  Latency-bound: with
// one lane per vertex throughout, a lane inserts its row entry by entry in memory.
__global__ __launch_bounds__(WAVE* ROWS_WAVES) void k_build_rows(View V, Params P, CellGrid G, const int* count,
                                                                 const int* flagCur, int* updateCount,
                                                                 int countUpdates, int rowsLds, int* err, int* maxcnt) {
  extern __shared__ int rows[];
  const int w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  Lane L;
  lane_ctx(V, blockIdx.x, threadIdx.x & (WAVE - 1), L);
  if (!flagCur[L.s]) return;
  if (countUpdates && L.tile == V.stile[L.s] && threadIdx.x == 0) updateCount[L.s] += 1;
  const Box B = box_of(V, L.s);
  if (rowsLds && !G.brute[L.s])
    build_rows_tile<-1>(V, P, G, count, G.slots, L, w, nw, B, V.x[L.v], V.y[L.v], rows, err, maxcnt, NearRows{});
  else if (w == 0 && L.act)
    build_row(V, P, G, count, G.slots, L.v, L.s, B, err, maxcnt);
}

// ------------------------------------------------------------ wide rings ---
// Ring sums of the rings of more than 64 vertices, whose slices k_step and k_shape read: area,
// perimeter and centre by ring_shape's unwrapped walk (exclusive prefix sums of the minimum-image
// segments from the ring's first vertex), here a block-wide scan over chunks of 256 vertices.
// One 256-thread block per wide ring.
__global__ __launch_bounds__(256) void k_wide_rings(View V, const int* wide) {
  __shared__ double wsum[2][4];
  __shared__ double red[4][4];
  const int r = wide[blockIdx.x];
  const int f = V.rfirst[r], n = V.rnv[r];
  const Box B = box_of(V, V.rsys[r]);
  const int t = threadIdx.x, lane = t & (WAVE - 1), wv = t / WAVE;
  double carryX = 0, carryY = 0;  // unwrapped offset of the chunk's first vertex
  double aP = 0, aS = 0, aX = 0, aY = 0;
  for (int b = 0; b < n; b += 256) {
    const int i = b + t;
    const bool act = i < n;
    double dnx = 0, dny = 0;
    if (act) {
      const int v = f + i, vn = (i + 1 == n) ? f : v + 1;
      dnx = pbx(V.x[vn] - V.x[v], B);
      dny = pby(V.y[vn] - V.y[v], B);
    }
    double ix = dnx, iy = dny;
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
      const double tx = __shfl_up(ix, d, WAVE), ty = __shfl_up(iy, d, WAVE);
      if (lane >= d) {
        ix += tx;
        iy += ty;
      }
    }
    if (lane == WAVE - 1) {
      wsum[0][wv] = ix;
      wsum[1][wv] = iy;
    }
    __syncthreads();
    double ox = carryX, oy = carryY;
    for (int q = 0; q < wv; q++) {
      ox += wsum[0][q];
      oy += wsum[1][q];
    }
    const double ux = ox + (ix - dnx), uy = oy + (iy - dny);
    for (int q = 0; q < 4; q++) {
      carryX += wsum[0][q];
      carryY += wsum[1][q];
    }
    __syncthreads();
    if (act) {
      aP += sqrt(dnx * dnx + dny * dny);
      aS += ux * dny - dnx * uy;
      aX += ux;
      aY += uy;
    }
  }
  aP = wave_sum(aP);
  aS = wave_sum(aS);
  aX = wave_sum(aX);
  aY = wave_sum(aY);
  if (lane == 0) {
    red[0][wv] = aP;
    red[1][wv] = aS;
    red[2][wv] = aX;
    red[3][wv] = aY;
  }
  __syncthreads();
  if (t == 0) {
    const double perim = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    const double shoe = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    const double sux = red[2][0] + red[2][1] + red[2][2] + red[2][3];
    const double suy = red[3][0] + red[3][1] + red[3][2] + red[3][3];
    const double ind = 1.0 / (double)n;
    V.area[r] = fabs(shoe) * 0.5;
    V.perim[r] = perim;
    V.cx[r] = V.x[f] + sux * ind;
    V.cy[r] = V.y[f] + suy * ind;
  }
}

// smooth interaction energy of each wide ring: the sum of its vertices' shares, which the
// slices of k_step store per vertex
__global__ __launch_bounds__(256) void k_wide_pe(View V, const int* wide) {
  __shared__ double red[4];
  const int r = wide[blockIdx.x];
  const int f = V.rfirst[r], n = V.rnv[r];
  double acc = 0;
  for (int i = threadIdx.x; i < n; i += 256) acc += V.es[f + i];
  acc = wave_sum(acc);
  if ((threadIdx.x & (WAVE - 1)) == 0) red[threadIdx.x / WAVE] = acc;
  __syncthreads();
  if (threadIdx.x == 0) V.pe[r] = red[0] + red[1] + red[2] + red[3];
}

// The step loop's row rebuild of k_step as a launch of its own, for sets with wide rings under
// the vertex-segment interaction: the last lane of a slice reads the row of a vertex in another
// tile, so every flagged row is complete before the step kernel starts (which then skips its
// rebuild, A.rowsBuilt).  One thread per vertex.
__global__ void k_rows_loop(View V, Params P, StepArgs A, CellGrid G) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V.nv) return;
  const int s = V.vsys[v];
  const int flag = A.flagCur[s];
  if ((flag & 1) == 0) return;
  const Box B = box_of(V, s);
  const bool allPairs = A.staleCheck && (flag & FLAG_FAR) != 0;
  const int* cnt = A.cellCur;  // FIRE: cells of these positions
  const int* slots = A.slotsCur;
  if (A.genCur) {
    // step loop: the cells of the list positions (md_cells); the step kernel after this launch
    // advances the system's generation
    const MdCells M = md_cells(A.cellCur, A.slotsCur, G, A.genCur[s]);
    const double x = V.x[v], y = V.y[v];
    if (!allPairs) md_stale_test(V, P, B, v, x, y, A.err);
    bin_vertex(G, B, M.binCnt, M.binSlots, v, s, x, y, A.err);
    if (!G.brute[s]) {
      const int n = G.ncx[s] * G.ncy[s];
      for (int c = v - V.svoff[s]; c < n; c += V.svoff[s + 1] - V.svoff[s]) M.clear[G.coff[s] + c] = 0;
    }
    cnt = M.cnt;
    slots = M.slots;
  }
  build_row(V, P, G, cnt, slots, v, s, B, A.err, A.maxcnt, allPairs);
}

// geometry only (calcParticleShape + calcParticlePositions)
template <bool WIDE>
__global__ void k_shape(View V, Params P) {
  Lane L;
  const int tile = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  if (tile >= V.ntiles) return;
  lane_ctx<WIDE>(V, tile, threadIdx.x & (WAVE - 1), L);
  ring_shape(V, P, L, box_of(V, L.s), V.x[L.v], V.y[L.v], true);
}

// Prologue of a step loop's cell protocol for vertex v of system s at positions (x, y): its list
// position binned into list 0 (generation 0), and the rebuild flag of (x, y) (the displacement
// test, with FLAG_FAR where (x, y) lies more than 2 cutoff / 3 from the list position, beyond what
// the cells allow for)
__device__ __forceinline__ void md_prologue(const View& V, const Params& P, const CellGrid& G, const StepArgs& A,
                                            const Box& B, int v, int s, double x, double y, int* flag, int* any) {
  const double lx = V.lx[v], ly = V.ly[v];
  bin_vertex(G, B, A.cellCur, A.slotsCur, v, s, lx, ly, A.err);
  moved_test(P, B, x - lx, y - ly, flag, any);
}

// Start of a step loop, one workgroup per tile: wave 0 takes the loop's opening move, all waves
// build the tile's near list from its rows at the list positions (when the loop uses them).
//   START_VERLET, START_BAOAB: the first half step from the stored force (velocity Verlet, or
//     BAOAB's B A O A with the draw of call ctr[0] + ctrOffT; BAOAB::integrate, Simulator.cu:112-120,
//     up to its force evaluation) into A.xout;
//   START_RIGID: the rigid loop's first half step from the stored ring force and torque (RigidNVE /
//     RigidLangevin::integrate, Simulator.cu:241-252, 316-326, up to the vertex move), every lane
//     moving its ring redundantly, the ring's first lane storing it;
//   START_STAY: the overdamped loops and rigid FIRE, whose first step starts from the current positions;
//   START_NEAR: the near lists only.
// All but START_NEAR run the loop's cell protocol (md_prologue on the positions the first step
// reads, whose flags go to A.flagOut; generation 0 into A.genOut; A.flagClear cleared).
// Latency-bound.  The rigid start took one thread per ring, which moved its vertices one after another:
// 48 us for 1,024 rings.
enum : int { START_VERLET, START_BAOAB, START_RIGID, START_STAY, START_NEAR };

template <int KIND, int INTER>
__global__ __launch_bounds__(WAVE* START_WAVES) void k_loop_start(View V, Params P, CellGrid G, StepArgs A) {
  __shared__ unsigned long long mask[2 * WAVE];
  const int w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  Lane L;
  lane_ctx(V, blockIdx.x, threadIdx.x & (WAVE - 1), L);
  const int v = L.v, s = L.s;
  const Box B = box_of(V, s);
  if constexpr (KIND != START_NEAR) {
    for (int t = gid; t < V.nsys; t += gridDim.x * blockDim.x) {
      if (A.flagClear) A.flagClear[t] = 0;
      A.genOut[t] = 0;
    }
  }
  if (KIND != START_NEAR && w == 0 && L.act) {
    const double x = V.x[v], y = V.y[v];
    double xn = x, yn = y;
    if constexpr (KIND == START_VERLET || KIND == START_BAOAB) {
      double vx = V.vx[v] + A.h * V.fx[v];
      double vy = V.vy[v] + A.h * V.fy[v];
      if constexpr (KIND == START_BAOAB) {
        double z0, z1;
        gauss_pair(P.seed, (uint32_t)s, TAG_THERMAL, A.ctr[0] + (unsigned long long)A.ctrOffT,
                   (uint32_t)(L.r - V.sroff[s]), z0, z1);
        const double xa = x + vx * A.h, ya = y + vy * A.h;
        vx = P.gamma * vx + P.noise * z0;
        vy = P.gamma * vy + P.noise * z1;
        xn = xa + vx * A.h;
        yn = ya + vy * A.h;
      } else {
        xn = x + A.dt * vx;
        yn = y + A.dt * vy;
      }
      V.vx[v] = vx;
      V.vy[v] = vy;
    }
    if constexpr (KIND == START_RIGID) {
      const Rigid R = *V.rg;
      const int r = L.r;
      double vx = R.pvx[r], vy = R.pvy[r], om = R.pw[r];
      double z0 = 0, z1 = 0;
      if (A.rigidLangevin)
        gauss_pair(P.seed, (uint32_t)s, TAG_THERMAL, A.ctr[0] + (unsigned long long)A.ctrOffT,
                   (uint32_t)(r - V.sroff[s]), z0, z1);
      rigid_kick(A.rigidLangevin, A.h, P.gamma, R.pfx[r], R.pfy[r], R.ptq[r], z0, z1, vx, vy, om);
      const double cx = V.cx[r], cy = V.cy[r], ang = V.ang[r];
      const double ncx = cx + A.dt * vx, ncy = cy + A.dt * vy, nang = ang + A.dt * om;
      const double dth = nang - ang;
      rigid_move(B, x, y, cx, cy, ncx, ncy, cos(dth), sin(dth), xn, yn);
      if (L.lane == L.segS) {  // every lane of the ring has read the old state
        R.plx[r] = cx;
        R.ply[r] = cy;
        R.pla[r] = ang;
        R.pvx[r] = vx;
        R.pvy[r] = vy;
        R.pw[r] = om;
        V.ang[r] = nang;
        V.cx[r] = ncx;
        V.cy[r] = ncy;
      }
    }
    if constexpr (KIND != START_STAY) {
      A.xout[v] = xn;
      A.yout[v] = yn;
      if (A.recx) {
        A.recx[v] = xn;
        A.recy[v] = yn;
      }
      far_test(P, B, xn - x, yn - y, A.flagOut + s);
    }
    md_prologue(V, P, G, A, B, v, s, xn, yn, A.flagOut + s, A.anyOut);
  }
  if (A.near.task) build_near_tile<INTER>(V, P, A.near, L, w, nw, B, V.lx, V.ly, G.brute[s] != 0, mask);
}

// RigidLangevin::injectKineticEnergy (Simulator.cu:254-261), one workgroup per system: a
// Gaussian pair of the given amplitude per ring (counter `call`), minus the system's mean ring
// velocity (kernelConserveParticleMomentum, cudaKernel.cuh:1998-2027, over every ring)
__global__ __launch_bounds__(256) void k_rigid_inject(View V, Params P, double amplitude, unsigned long long call) {
  const Rigid R = *V.rg;
  __shared__ double red[2][256 / WAVE];
  const int s = blockIdx.x, tid = threadIdx.x;
  const int r0 = V.sroff[s], r1 = V.sroff[s + 1];
  double mx = 0, my = 0;
  for (int r = r0 + tid; r < r1; r += blockDim.x) {
    double z0, z1;
    gauss_pair(P.seed, (uint32_t)s, TAG_INJECT, call, (uint32_t)(r - r0), z0, z1);
    R.pvx[r] = amplitude * z0;
    R.pvy[r] = amplitude * z1;
    mx += R.pvx[r];
    my += R.pvy[r];
  }
  mx = wave_sum(mx);
  my = wave_sum(my);
  if ((tid & (WAVE - 1)) == 0) {
    red[0][tid / WAVE] = mx;
    red[1][tid / WAVE] = my;
  }
  __syncthreads();
  mx = 0;
  my = 0;
  for (int q = 0; q < (int)(blockDim.x / WAVE); q++) {
    mx += red[0][q];
    my += red[1][q];
  }
  mx /= (r1 - r0);
  my /= (r1 - r0);
  for (int r = r0 + tid; r < r1; r += blockDim.x) {
    R.pvx[r] -= mx;
    R.pvy[r] -= my;
  }
}

// RNG call counters advanced by the draws of a finished loop
__global__ void k_ctr_add(unsigned long long* ctr, long long addT, long long addA) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ctr[0] += (unsigned long long)addT;
    ctr[1] += (unsigned long long)addA;
  }
}

__global__ void k_fill_int(int* p, int value, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}

__global__ void k_copy_lastpos(View V) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V.nv) return;
  V.lx[v] = V.x[v];
  V.ly[v] = V.y[v];
}

// ---------------------------------------------------------- reductions ---
// Per-system sums, fixed striding and tree order (deterministic):
// out[s*8 + q]: 0 sum e_v, 1 sum pe, 2 sum v^2, 3 max F_c^2, 4 sum F^2,
//               5 sum area, 6 sum a0, 7 sum vertex-disk area r^2 (n/2 - 1)
// One block per REDUCE_CHUNK vertices of a system (block b serves system chunkSys[b]; its first block
// is chunkOff[s]) and the same share of its rings.  A system of one block is summed here; those of
// more leave partials that k_reduce_final adds.  (One block per system read a large system through
// one CU: 613 us for 524,288 vertices, 23 us for 19,456.)
__device__ __forceinline__ double reduce_op(int q, double a, double b) { return q == 3 ? fmax(a, b) : a + b; }

__global__ __launch_bounds__(512) void k_reduce(View V, const int* chunkSys, const int* chunkOff, double* part,
                                                double* out) {
  const int s = chunkSys[blockIdx.x], c = blockIdx.x - chunkOff[s], n = chunkOff[s + 1] - chunkOff[s];
  __shared__ double sh[8][8];
  double acc[8] = {0, 0, 0, -1, 0, 0, 0, 0};
  const int b0 = V.svoff[s] + c * REDUCE_CHUNK, b1 = min(V.svoff[s + 1], b0 + REDUCE_CHUNK);
  for (int v = b0 + threadIdx.x; v < b1; v += 512) {
    const double vx = V.vx[v], vy = V.vy[v], fx = V.fx[v], fy = V.fy[v];
    acc[0] += V.ev[v];
    acc[2] += vx * vx + vy * vy;
    acc[3] = fmax(acc[3], fmax(fx * fx, fy * fy));
    acc[4] += fx * fx + fy * fy;
  }
  const int r0 = V.sroff[s];
  const long nr = V.sroff[s + 1] - r0;
  const int q0 = r0 + (int)(nr * c / n), q1 = r0 + (int)(nr * (c + 1) / n);
  for (int r = q0 + threadIdx.x; r < q1; r += 512) {
    acc[1] += V.pe[r];
    acc[5] += V.area[r];
    acc[6] += V.a0[r];
    const double rr = V.rad[V.rfirst[r]];
    acc[7] += rr * rr * (0.5 * V.rnv[r] - 1);
  }
  const int w = threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const double t = (q == 3) ? wave_max(acc[q]) : wave_sum(acc[q]);
    if (lane == 0) sh[q][w] = t;
  }
  __syncthreads();
  if (threadIdx.x < 8) {
    const int q = threadIdx.x;
    double t = sh[q][0];
    for (int i = 1; i < 8; i++) t = reduce_op(q, t, sh[q][i]);
    if (n == 1) out[s * 8 + q] = t;
    else part[(long)blockIdx.x * 8 + q] = t;
  }
}

// lane 8 i + q adds the partials i, i + 8, ... of sum q
__global__ __launch_bounds__(WAVE) void k_reduce_final(const int* chunkOff, const double* part, double* out) {
  const int s = blockIdx.x, q = threadIdx.x & 7;
  const int c0 = chunkOff[s], c1 = chunkOff[s + 1];
  if (c1 - c0 == 1) return;
  double t = q == 3 ? -1 : 0;
  for (int c = c0 + (int)(threadIdx.x >> 3); c < c1; c += 8) t = reduce_op(q, t, part[(long)c * 8 + q]);
#pragma unroll
  for (int d = 32; d >= 8; d >>= 1) t = reduce_op(q, t, __shfl_xor(t, d, WAVE));
  if (threadIdx.x < 8) out[s * 8 + q] = t;
}

// Langevin::injectKineticEnergy, Simulator.cu:32-52: per-ring Gaussian velocity
__global__ void k_inject(View V, Params P, double amplitude, unsigned long long call) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V.nv) return;
  const int r = V.vring[v], s = V.vsys[v];
  double z0, z1;
  gauss_pair(P.seed, (uint32_t)s, TAG_INJECT, call, (uint32_t)(r - V.sroff[s]), z0, z1);
  V.vx[v] = amplitude * z0;
  V.vy[v] = amplitude * z1;
}

// Stages of the reference's Langevin integrator for callers that drive them one by one
// (Simulator.cu:85-95 kernelUpdateVertexPos / kernelUpdateVertexVel, 54-77 updateThermalVel):
// x += dt v; v += dt F; F += noise xi_ring - gamma v with the ring's draw of call `call`
__global__ void k_update_pos(View V, double dt) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V.nv) return;
  V.x[v] += dt * V.vx[v];
  V.y[v] += dt * V.vy[v];
}

__global__ void k_update_vel(View V, double dt) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V.nv) return;
  V.vx[v] += dt * V.fx[v];
  V.vy[v] += dt * V.fy[v];
}

__global__ void k_thermal_force(View V, Params P, const unsigned long long* ctr) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V.nv) return;
  const int r = V.vring[v], s = V.vsys[v];
  double z0, z1;
  gauss_pair(P.seed, (uint32_t)s, TAG_THERMAL, ctr[0], (uint32_t)(r - V.sroff[s]), z0, z1);
  V.fx[v] += P.noise * z0 - P.gamma * V.vx[v];
  V.fy[v] += P.noise * z1 - P.gamma * V.vy[v];
}

// subtract the per-system mean velocity
__global__ __launch_bounds__(256) void k_sub_mean(View V) {
  const int s = blockIdx.x;
  __shared__ double sh[2][4];
  __shared__ double mean[2];
  const int b0 = V.svoff[s], b1 = V.svoff[s + 1];
  double ax = 0, ay = 0;
  for (int v = b0 + threadIdx.x; v < b1; v += 256) { ax += V.vx[v]; ay += V.vy[v]; }
  const int w = threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
  ax = wave_sum(ax); ay = wave_sum(ay);
  if (lane == 0) { sh[0][w] = ax; sh[1][w] = ay; }
  __syncthreads();
  if (threadIdx.x < 2) {
    double t = 0;
    for (int i = 0; i < 4; i++) t += sh[threadIdx.x][i];
    mean[threadIdx.x] = t / (b1 - b0);
  }
  __syncthreads();
  for (int v = b0 + threadIdx.x; v < b1; v += 256) { V.vx[v] -= mean[0]; V.vy[v] -= mean[1]; }
}

// v *= scale[s]
__global__ void k_scale_vel(View V, const double* scale) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V.nv) return;
  const double sc = scale[V.vsys[v]];
  V.vx[v] *= sc;
  V.vy[v] *= sc;
}

// scaleVertices, DPM2D.cu:1802-1811 + kernelScaleVertexPositions, cudaKernel.cuh:1644-1658
__global__ void k_scale_vertices(View V, const double* scale) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < V.nv) {
    const int r = V.vring[v];
    const double sc = scale[V.vsys[v]];
    V.x[v] += (sc - 1) * (V.x[v] - V.cx[r]);
    V.y[v] += (sc - 1) * (V.y[v] - V.cy[r]);
    V.l0[v] *= sc;
    V.rad[v] *= sc;
  }
  if (v < V.np) {
    const double sc = scale[V.rsys[v]];
    V.a0[v] *= sc * sc;
    V.area[v] *= sc * sc;
  }
}

// scaleBox, DPM2D.cu:1693-1719, with translateVertices (kernelTranslateVertices,
// cudaKernel.cuh:1678-1693): every vertex moves by the shift of its ring's centre to
// centre / scale, a box distance in the new box (uploaded before this launch); the centres
// themselves are divided in k_scale_centres, launched after
__global__ void k_scale_box(View V, const double* scale) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V.nv) return;
  const int r = V.vring[v], s = V.vsys[v];
  const Box B = box_of(V, s);
  const double cx = V.cx[r], cy = V.cy[r], sc = scale[s];
  V.x[v] += pbx(cx / sc - cx, B);
  V.y[v] += pby(cy / sc - cy, B);
}

__global__ void k_scale_centres(View V, const double* scale) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= V.np) return;
  const double sc = scale[V.rsys[r]];
  V.cx[r] /= sc;
  V.cy[r] /= sc;
}

// --------------------------------------------------------------- FIRE ---
// sum of the per-tile partials q of system s, all 64 lanes striding over the tiles; the
// xor-butterfly leaves the same value in every lane (addition is commutative)
__device__ __forceinline__ double sys_sum(const double* part, int q, int t0, int t1, int lane) {
  double acc = 0;
  for (int t = t0 + lane; t < t1; t += WAVE) acc += part[t * 4 + q];
  return wave_sum(acc);
}

__device__ __forceinline__ double sys_max(const double* part, int q, int t0, int t1, int lane) {
  double acc = -1;
  for (int t = t0 + lane; t < t1; t += WAVE) acc = fmax(acc, part[t * 4 + q]);
  return wave_max(acc);
}

// --------------------------------------------------------- rigid FIRE ---
__global__ void k_rigid_fire_partials(View V, double* part) {
  const Rigid R = *V.rg;
  Lane L;
  if (!wave_tile_ctx(V, L)) return;
  const bool head = L.act && L.lane == L.segS;
  double vx = 0, vy = 0, Fx = 0, Fy = 0;
  if (head) {
    vx = R.pvx[L.r];
    vy = R.pvy[L.r];
    Fx = R.pfx[L.r];
    Fy = R.pfy[L.r];
  }
  rigid_fire_partials(L, head, vx, vy, Fx, Fy, part);
}

// One rigid FIRE iteration up to the vertex move, one wave per tile (FIRE::minimizerRigidLoop,
// FIRE.cu:279-291, with checkRigidFIREParams 217-254 and bendRigidVelocityTowardsForce 256-277).
// Every wave derives its system's FIRE update from the tile partials of the state after the
// previous iteration (power P = sum v.F decides; on a restart the centres and angles step back by
// half the already-decreased step and both velocities clear), and the bend ratio from
// |v'|^2 = h^2 |F|^2 after a restart, else |v|^2 + 2 h P + h^2 |F|^2, the half-kicked velocities'
// norm.  Each lane moves its ring redundantly and its vertex with it; the ring's first lane
// stores the ring, the system's first tile the new FIRE state (fout; fin stays as it was).
// The last centres and angles are the ones at the start of the iteration.
__global__ void k_rigid_fire_move(View V, Params P, FireParams fp, const FireState* fin, FireState* fout,
                                  const double* part, double* xo, double* yo, int* flagOut, int* anyOut) {
  const Rigid R = *V.rg;
  Lane L;
  if (!wave_tile_ctx(V, L)) return;
  const int t0 = V.stile[L.s], t1 = V.stile[L.s + 1];
  const double P0 = sys_sum(part, 0, t0, t1, L.lane);
  const double VV = sys_sum(part, 1, t0, t1, L.lane);
  const double FF = sys_sum(part, 2, t0, t1, L.lane);
  FireState f = fin[L.s];
  const bool restart = !(P0 > 0);
  if (!restart) {
    f.numStep++;
    if (f.numStep > fp.minStep) {
      f.dt = fmin(f.dt * fp.f_inc, fp.dt_max);
      f.a *= fp.f_a;
    }
  } else {
    f.numStep = 0;
    f.dt = fmax(f.dt * fp.f_dec, fp.dt_max / 10);
    f.a = fp.a_start;
  }
  const double h = 0.5 * f.dt;
  if (L.tile == t0 && L.lane == 0) {
    FireState o = f;
    o.P = P0;
    o.iters = f.iters + 1;
    fout[L.s] = o;
  }
  if (!L.act) return;
  const double VV1 = restart ? h * h * FF : VV + 2 * h * P0 + h * h * FF;
  double cx = V.cx[L.r], cy = V.cy[L.r], ang = V.ang[L.r];
  double vx = R.pvx[L.r], vy = R.pvy[L.r], w = R.pw[L.r];
  const double Fx = R.pfx[L.r], Fy = R.pfy[L.r];
  const double lcx = cx, lcy = cy, lang = ang;
  if (restart) {
    cx -= h * vx;
    cy -= h * vy;
    ang -= h * w;
    vx = vy = w = 0;
  }
  rigid_kick(false, h, 0.0, Fx, Fy, R.ptq[L.r], 0.0, 0.0, vx, vy, w);
  if (FF > 0) {
    const double ratio = sqrt(VV1 / FF);
    vx = (1 - f.a) * vx + f.a * Fx * ratio;
    vy = (1 - f.a) * vy + f.a * Fy * ratio;
  }
  cx += f.dt * vx;
  cy += f.dt * vy;
  ang += f.dt * w;
  const Box B = box_of(V, L.s);
  const double dth = ang - lang;
  double xn, yn;
  rigid_move(B, V.x[L.v], V.y[L.v], lcx, lcy, cx, cy, cos(dth), sin(dth), xn, yn);
  xo[L.v] = xn;
  yo[L.v] = yn;
  moved_test(P, B, xn - V.lx[L.v], yn - V.ly[L.v], flagOut + L.s, anyOut);
  if (L.lane == L.segS) {
    R.plx[L.r] = lcx;
    R.ply[L.r] = lcy;
    R.pla[L.r] = lang;
    V.cx[L.r] = cx;
    V.cy[L.r] = cy;
    V.ang[L.r] = ang;
    R.pvx[L.r] = vx;
    R.pvy[L.r] = vy;
    R.pw[L.r] = w;
  }
}

// FIRE::minimizerVertexLoop, FIRE.cu:397-411, split at its two global reductions.
// fire_begin: checkFIREParams (338-371) + half kick + partial |v|^2, |F|^2.
// With tol >= 0 a system whose max |F_c| <= tol (or that reached maxIter) is frozen.
__global__ void k_fire_begin(View V, FireParams fp, const FireState* fin, FireState* fout, double* part) {
  Lane L;
  if (!wave_tile_ctx(V, L)) return;
  FireState fs = fin[L.s];
  const int t0 = V.stile[L.s], t1 = V.stile[L.s + 1];
  const double Psum = sys_sum(part, 0, t0, t1, L.lane);
  if (!fs.converged && fp.tol >= 0) {
    const double fmax2 = sys_max(part, 3, t0, t1, L.lane);
    if (sqrt(fmax2) <= fp.tol || fs.iters >= fp.maxIter) fs.converged = 1;
  }
  bool reset = false;
  if (!fs.converged) {
    fs.P = Psum;
    if (Psum > 0) {
      fs.numStep++;
      if (fs.numStep > fp.minStep) {
        fs.dt = fmin(fs.dt * fp.f_inc, fp.dt_max);
        fs.a *= fp.f_a;
      }
    } else {
      fs.numStep = 0;
      fs.dt = fmax(fs.dt * fp.f_dec, fp.dt_max / 10);
      fs.a = fp.a_start;
      reset = true;
    }
    fs.iters++;
  }
  if (L.tile == t0 && L.lane == 0) fout[L.s] = fs;
  double vx = 0, vy = 0, fx = 0, fy = 0;
  if (L.act) {
    vx = V.vx[L.v]; vy = V.vy[L.v]; fx = V.fx[L.v]; fy = V.fy[L.v];
    if (!fs.converged) {
      if (reset) {
        const double hb = 0.5 * fs.dt;
        V.x[L.v] -= hb * vx;
        V.y[L.v] -= hb * vy;
        vx = 0; vy = 0;
      }
      const double h = 0.5 * fs.dt;
      vx += h * fx;
      vy += h * fy;
      V.vx[L.v] = vx;
      V.vy[L.v] = vy;
    }
  }
  const double tv = wave_sum(vx * vx + vy * vy);
  const double tf = wave_sum(fx * fx + fy * fy);
  if (L.lane == 0) {
    part[L.tile * 4 + 1] = tv;
    part[L.tile * 4 + 2] = tf;
  }
}

// fire_mid: bendVertexVelocityTowardsForce (374-394) + drift + displacement test
__global__ void k_fire_mid(View V, Params P, const FireState* fcur, const double* part, double* xo, double* yo,
                           int* flagOut, int* anyOut) {
  Lane L;
  if (!wave_tile_ctx(V, L)) return;
  const FireState fs = fcur[L.s];
  const int t0 = V.stile[L.s], t1 = V.stile[L.s + 1];
  const double vv = sys_sum(part, 1, t0, t1, L.lane);
  const double ff = sys_sum(part, 2, t0, t1, L.lane);
  if (!L.act) return;
  double vx = V.vx[L.v], vy = V.vy[L.v];
  const double x = V.x[L.v], y = V.y[L.v];
  if (fs.converged) {
    xo[L.v] = x;
    yo[L.v] = y;
    return;
  }
  if (ff > 0) {
    const double ratio = sqrt(vv / ff);
    const double fa = fs.a;
    vx = (1 - fa) * vx + fa * V.fx[L.v] * ratio;
    vy = (1 - fa) * vy + fa * V.fy[L.v] * ratio;
  }
  const double xn = x + fs.dt * vx, yn = y + fs.dt * vy;
  V.vx[L.v] = vx;
  V.vy[L.v] = vy;
  xo[L.v] = xn;
  yo[L.v] = yn;
  const Box B = box_of(V, L.s);
  if (moved_past(P, B, xn - V.lx[L.v], yn - V.ly[L.v])) {
    atomicOr(&flagOut[L.s], 1);
    atomicOr(anyOut, 1);
  }
}

// per-tile partials of P = v.F and max F_c^2 for the current state (start of a FIRE call)
__global__ void k_fire_partials(View V, double* part) {
  Lane L;
  if (!wave_tile_ctx(V, L)) return;
  double pvf = 0, f2 = -1;
  if (L.act) {
    const double vx = V.vx[L.v], vy = V.vy[L.v], fx = V.fx[L.v], fy = V.fy[L.v];
    pvf = vx * fx + vy * fy;
    f2 = fmax(fx * fx, fy * fy);
  }
  const double tP = wave_sum(pvf);
  const double tM = wave_max(f2);
  if (L.lane == 0) {
    part[L.tile * 4 + 0] = tP;
    part[L.tile * 4 + 3] = tM;
  }
}

// An iteration of FIRE on every tile up to the drift (the step kernel of MODE_FIRE | MODE_NEAR follows):
// `per` blocks a system, of one wave per tile.  Every block sums its whole system
// first, over the vertices in the order of the persistent kernel with as many waves (so that both follow
// the same path to the last bit), then takes the stopping rule and the parameter update and moves its
// vertices into the other position buffer and vxn, vyn (other blocks still sum vx, vy), with the step
// loop's flags.  A system that has stopped only keeps its positions in the buffer that is read next.  Look
// `look` (not 0) notes whether a system goes on, and the launch after it tells the host.
__global__ __launch_bounds__(WAVE* FS_WAVES) void k_fire_move(View V, Params P, FireParams fp, int per,
                                                              const FireState* fin, FireState* fout, double* xo,
                                                              double* yo, double* vxn, double* vyn, int* flagOut,
                                                              int* anyOut, int* open, int look, int* told,
                                                              int tell) {
  __shared__ double red[FS_WAVES][5];
  const int s = blockIdx.x / per, w = threadIdx.x / WAVE, nw = blockDim.x / WAVE, lane = threadIdx.x & (WAVE - 1);
  const int t0 = V.stile[s], t1 = V.stile[s + 1], tile = t0 + (blockIdx.x % per) * nw + w;
  FireState fs = fin[s];  // (before the store below, which would take it from the scalar cache)
  // what the launch before, look `tell`, found, for the host (pinned memory)
  if (tell && blockIdx.x == 0 && threadIdx.x == 0) *(volatile int*)told = 2 * tell + (*open == tell);
  FireSums sum{0, -1, 0, 0, 0};
  bool reset = false;
  if (!fs.converged) {
    const FireNext next(fp, fs);
    FireSums a{0, -1, 0, 0, 0};
    for (int t = t0 + w; t < t1; t += nw) {
      const int v = V.tile_v0[t] + lane;
      if (v < V.tile_v1[t]) fire_add(a, next, V.vx[v], V.vy[v], V.fx[v], V.fy[v]);
    }
    sum = fire_block_sums(a, red, nw);
    reset = fire_update(fs, fp, sum);
  }
  if (tile == t0 && lane == 0) {
    fout[s] = fs;
    if (look && !fs.converged) *open = look;
  }
  if (tile >= t1) return;
  const int v = V.tile_v0[tile] + lane;
  if (v >= V.tile_v1[tile]) return;
  const double x = V.x[v], y = V.y[v];
  double xn = x, yn = y;
  if (!fs.converged) {
    double vx = V.vx[v], vy = V.vy[v];
    fire_move(fs, sum, reset, V.fx[v], V.fy[v], xn, yn, vx, vy);
    vxn[v] = vx;
    vyn[v] = vy;
    moved_test(P, box_of(V, s), xn - V.lx[v], yn - V.ly[v], flagOut + s, anyOut);
  }
  xo[v] = xn;
  yo[v] = yn;
}

// a new minimisation call tests every system's stopping rule again (the driver's loop condition
// is evaluated per call, compressFIRE.cpp:121-131)
__global__ void k_fire_resume(FireState* fs, int nsys) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < nsys) fs[s].converged = 0;
}

// --------------------------------------------------------- launchers ---

template <int INTER>
static hipError_t step_pot(dpm_set_s* S, int mode, const StepArgs& A) {
  switch (S->P.potential) {
    case POT_HARMONIC: return step_launch<INTER, POT_HARMONIC>(S, mode, A);
    case POT_LJ: return step_launch<INTER, POT_LJ>(S, mode, A);
    case POT_ADHESIVE: return step_launch<INTER, POT_ADHESIVE>(S, mode, A);
    case POT_WCA: return step_launch<INTER, POT_WCA>(S, mode, A);
  }
  return hipErrorInvalidValue;
}

template <int INTER>
static hipError_t fire_pot(dpm_set_s* S, int chunk, int threads) {
  switch (S->P.potential) {
    case POT_HARMONIC: return fire_launch<INTER, POT_HARMONIC>(S, chunk, threads);
    case POT_LJ: return fire_launch<INTER, POT_LJ>(S, chunk, threads);
    case POT_ADHESIVE: return fire_launch<INTER, POT_ADHESIVE>(S, chunk, threads);
    default: return fire_launch<INTER, POT_WCA>(S, chunk, threads);
  }
}

static hipError_t launch_step_kernel(dpm_set_s* S, int mode, const StepArgs& A);

// Sets with wide rings (more than 64 vertices) run, around each step kernel, the ring sums
// of their slices before it (and, under the vertex-segment interaction inside loops, the row
// rebuild), and the wide rings' interaction energies after it.
hipError_t launch_step(dpm_set_s* S, int mode, const StepArgs& A0) {
  if (S->nwide == 0) return launch_step_kernel(S, mode, A0);
  if ((mode & MODE_RIGID) || S->P.particle == PART_ACTIVE || S->P.particle == PART_ACTIVE_SHAPE)
    return hipErrorInvalidValue;  // refused by the entry points before this point
  StepArgs A = A0;
  const bool smooth = S->P.interaction == INT_SMOOTH;
  if (smooth && A.manage) {
    if (!A.flagCur || !A.cellCur || !A.slotsCur || !A.err || !A.maxcnt) return hipErrorInvalidValue;
    k_rows_loop<<<grid_v(S->nv), 256, 0, S->stream>>>(S->V, S->P, A, S->G);
    A.rowsBuilt = 1;
  }
  k_wide_rings<<<(int)S->nwide, 256, 0, S->stream>>>(S->V, S->d_wide);
  hipError_t e = launch_step_kernel(S, mode, A);
  if (e != hipSuccess) return e;
  if (smooth) k_wide_pe<<<(int)S->nwide, 256, 0, S->stream>>>(S->V, S->d_wide);
  return hipGetLastError();
}

static hipError_t launch_step_kernel(dpm_set_s* S, int mode, const StepArgs& A0) {
  // refuse argument sets the chosen epilogue would dereference as null
  if (!A0.ctr) return hipErrorInvalidValue;
  // in-loop rebuilds by the whole workgroup need LDS for the tile's rows (rows_lds_ints), in the
  // region the gather's results use afterwards (W <= 64)
  StepArgs A = A0;
  A.rowsLdsW = (A.manage && S->V.W <= 64) ? S->V.W : 0;
  if (S->P.particle == PART_ACTIVE_SHAPE && !S->V.l0r) return hipErrorInvalidValue;
  if ((mode & MODE_FIRE) && (!A.fire || !A.part)) return hipErrorInvalidValue;
  if ((mode & MODE_RIGID) && S->P.interaction == INT_ALL) return hipErrorInvalidValue;
  if ((mode & MODE_NEAR) && (!A.near.task || S->V.W > 64)) return hipErrorInvalidValue;  // masks of 64 entries
  if ((mode & MODE_START) && (!A.xout || !A.yout || !A.flagOut || !A.anyOut)) return hipErrorInvalidValue;
  if (A.manage && (!A.flagCur || !A.cellCur || !A.slotsCur || (A.genCur && !A.genOut) || !A.err || !A.maxcnt ||
                   !A.updateCount))
    return hipErrorInvalidValue;
  switch (S->P.interaction) {
    case INT_VV: return step_pot<INT_VV>(S, mode, A);
    case INT_SMOOTH: return step_pot<INT_SMOOTH>(S, mode, A);
    case INT_ALL: return step_pot<INT_ALL>(S, mode, A);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_shape_only(dpm_set_s* S) {
  if (S->nwide > 0) {
    k_wide_rings<<<(int)S->nwide, 256, 0, S->stream>>>(S->V, S->d_wide);
    k_shape<true><<<grid_w(S->V.ntiles), 256, 0, S->stream>>>(S->V, S->P);
  } else {
    k_shape<false><<<grid_w(S->V.ntiles), 256, 0, S->stream>>>(S->V, S->P);
  }
  return hipGetLastError();
}

template <int KIND>
static hipError_t loop_start(dpm_set_s* S, const View& Vn, const StepArgs& A) {
  if (KIND != START_NEAR && (!A.genOut || !A.flagOut || !A.anyOut || !A.cellCur || !A.slotsCur || !A.ctr))
    return hipErrorInvalidValue;
  if (KIND != START_NEAR && KIND != START_STAY && (!A.xout || !A.yout || !A.flagClear)) return hipErrorInvalidValue;
  const int threads = WAVE * (A.near.task ? START_WAVES : 1);
  if (S->P.interaction == INT_SMOOTH)
    k_loop_start<KIND, INT_SMOOTH><<<S->V.ntiles, threads, 0, S->stream>>>(Vn, S->P, S->G, A);
  else
    k_loop_start<KIND, INT_VV><<<S->V.ntiles, threads, 0, S->stream>>>(Vn, S->P, S->G, A);
  return hipGetLastError();
}

hipError_t launch_start_baoab(dpm_set_s* S, const StepArgs& A) { return loop_start<START_BAOAB>(S, S->V, A); }

hipError_t launch_start_md(dpm_set_s* S, const StepArgs& A) { return loop_start<START_VERLET>(S, S->V, A); }

// the start of the loops that begin at the positions of Vn as they are: their flags into `flag`,
// generation 0 into `genOut`
hipError_t launch_bin_flag(dpm_set_s* S, const View& Vn, int* count, int* slots, int* flag, int* genOut,
                           const NearRows& near) {
  StepArgs A{};
  A.ctr = S->d_ctr;
  A.cellCur = count;
  A.slotsCur = slots;
  A.flagOut = flag;
  A.anyOut = S->d_any + 2;  // not read by the loop
  A.genOut = genOut;
  A.err = S->d_err;
  A.near = near;
  return loop_start<START_STAY>(S, Vn, A);
}

// the near lists at the list positions
hipError_t launch_near(dpm_set_s* S) {
  StepArgs A{};
  A.near = S->N;
  return loop_start<START_NEAR>(S, S->V, A);
}

hipError_t launch_ctr_add(dpm_set_s* S, long long addT, long long addA) {
  k_ctr_add<<<1, 64, 0, S->stream>>>(S->d_ctr, addT, addA);
  return hipGetLastError();
}

hipError_t launch_bin(dpm_set_s* S, int bumpThermal, int bumpActive) {
  const int b = S->cur;
  long n = S->nv > S->nsys ? S->nv : S->nsys;
  k_bin<<<grid_v(n), 256, 0, S->stream>>>(S->V, S->G, S->G.count[b], S->d_flag[b], S->d_any + b,
                                          S->d_flag[1 - b], S->d_any + 1 - b, S->d_ctr, bumpThermal, bumpActive,
                                          S->d_err);
  return hipGetLastError();
}

// k_bin on positions other than the set's current buffer (the adjoint's recorded positions),
// with the flags and cells of `parity`; no RNG counter bump.
hipError_t launch_bin_view(dpm_set_s* S, const View& Vn, int parity) {
  long n = S->nv > S->nsys ? S->nv : S->nsys;
  k_bin<<<grid_v(n), 256, 0, S->stream>>>(Vn, S->G, S->G.count[parity], S->d_flag[parity], S->d_any + parity,
                                          S->d_flag[1 - parity], S->d_any + 1 - parity, S->d_ctr, 0, 0, S->d_err);
  return hipGetLastError();
}

hipError_t launch_build_rows(dpm_set_s* S, int countUpdates) {
  return launch_build_rows_view(S, S->V, S->cur, countUpdates);
}

// k_build_rows on positions other than the set's current buffer (the list positions), with the
// flags and cells of `parity`
hipError_t launch_build_rows_view(dpm_set_s* S, const View& Vn, int parity, int countUpdates) {
  const int rowsLds = Vn.W <= 64;
  const size_t sh = rowsLds ? (size_t)rows_lds_ints(Vn.W, false) * sizeof(int) : 0;
  k_build_rows<<<Vn.ntiles, rowsLds ? WAVE * ROWS_WAVES : WAVE, sh, S->stream>>>(
      Vn, S->P, S->G, S->G.count[parity], S->d_flag[parity], S->d_updateCount, countUpdates, rowsLds, S->d_err,
      S->d_maxcnt);
  return hipGetLastError();
}

hipError_t launch_fill_int(int* p, int value, long n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  k_fill_int<<<grid_v(n), 256, 0, st>>>(p, value, n);
  return hipGetLastError();
}

hipError_t launch_reduce(dpm_set_s* S) {
  k_reduce<<<S->redBlocks, 512, 0, S->stream>>>(S->V, S->d_chunkSys, S->d_chunkOff, S->d_red, S->h_red);
  if (S->redBlocks > S->nsys) k_reduce_final<<<(int)S->nsys, WAVE, 0, S->stream>>>(S->d_chunkOff, S->d_red, S->h_red);
  return hipGetLastError();
}

hipError_t launch_inject(dpm_set_s* S, double amplitude, unsigned long long call) {
  k_inject<<<grid_v(S->nv), 256, 0, S->stream>>>(S->V, S->P, amplitude, call);
  return hipGetLastError();
}

hipError_t launch_update_pos(dpm_set_s* S, double dt) {
  k_update_pos<<<grid_v(S->nv), 256, 0, S->stream>>>(S->V, dt);
  return hipGetLastError();
}

hipError_t launch_update_vel(dpm_set_s* S, double dt) {
  k_update_vel<<<grid_v(S->nv), 256, 0, S->stream>>>(S->V, dt);
  return hipGetLastError();
}

hipError_t launch_thermal_force(dpm_set_s* S) {
  k_thermal_force<<<grid_v(S->nv), 256, 0, S->stream>>>(S->V, S->P, S->d_ctr);
  return hipGetLastError();
}

hipError_t launch_sub_mean(dpm_set_s* S) {
  k_sub_mean<<<(int)S->nsys, 256, 0, S->stream>>>(S->V);
  return hipGetLastError();
}

hipError_t launch_scale_vel(dpm_set_s* S) {
  k_scale_vel<<<grid_v(S->nv), 256, 0, S->stream>>>(S->V, S->d_scale);
  return hipGetLastError();
}

hipError_t launch_scale_vertices(dpm_set_s* S) {
  long n = S->nv > S->np ? S->nv : S->np;
  k_scale_vertices<<<grid_v(n), 256, 0, S->stream>>>(S->V, S->d_scale);
  return hipGetLastError();
}

hipError_t launch_scale_box(dpm_set_s* S) {
  k_scale_box<<<grid_v(S->nv), 256, 0, S->stream>>>(S->V, S->d_scale);
  k_scale_centres<<<grid_v(S->np), 256, 0, S->stream>>>(S->V, S->d_scale);
  return hipGetLastError();
}

hipError_t launch_rigid_start(dpm_set_s* S, bool langevin, const StepArgs& A) {
  StepArgs B = A;
  B.rigidLangevin = langevin ? 1 : 0;
  return loop_start<START_RIGID>(S, S->V, B);
}

hipError_t launch_rigid_inject(dpm_set_s* S, double amplitude, unsigned long long call) {
  k_rigid_inject<<<(int)S->nsys, 256, 0, S->stream>>>(S->V, S->P, amplitude, call);
  return hipGetLastError();
}

hipError_t launch_rigid_fire_partials(dpm_set_s* S) {
  k_rigid_fire_partials<<<grid_w(S->V.ntiles), 256, 0, S->stream>>>(S->V, S->d_part);
  return hipGetLastError();
}

hipError_t launch_rigid_fire_move(dpm_set_s* S, int* flagOut, int* anyOut) {
  if (!flagOut || !anyOut) return hipErrorInvalidValue;
  const int nb = 1 - S->cur;
  k_rigid_fire_move<<<grid_w(S->V.ntiles), 256, 0, S->stream>>>(
      S->V, S->P, S->fp, S->d_rfire[S->rfireCur], S->d_rfire[1 - S->rfireCur], S->d_part, S->pos[nb][0],
      S->pos[nb][1], flagOut, anyOut);
  return hipGetLastError();
}

hipError_t launch_copy_lastpos(dpm_set_s* S) {
  k_copy_lastpos<<<grid_v(S->nv), 256, 0, S->stream>>>(S->V);
  return hipGetLastError();
}

hipError_t launch_fire_begin(dpm_set_s* S) {
  k_fire_begin<<<grid_w(S->V.ntiles), 256, 0, S->stream>>>(S->V, S->fp, S->d_fire[S->fireCur],
                                                            S->d_fire[1 - S->fireCur], S->d_part);
  return hipGetLastError();
}

hipError_t launch_fire_mid(dpm_set_s* S) {
  const int nb = 1 - S->cur;
  k_fire_mid<<<grid_w(S->V.ntiles), 256, 0, S->stream>>>(S->V, S->P, S->d_fire[S->fireCur], S->d_part,
                                                          S->pos[nb][0], S->pos[nb][1], S->d_flag[nb],
                                                          S->d_any + nb);
  return hipGetLastError();
}

hipError_t launch_fire_move(dpm_set_s* S, int most, int waves, int* flagOut, int* anyOut, int look, int tell) {
  if (!flagOut || !anyOut || waves < 1 || waves > FS_WAVES) return hipErrorInvalidValue;
  const int nb = 1 - S->cur;
  const int per = (most + waves - 1) / waves;
  k_fire_move<<<(unsigned)(S->nsys * per), WAVE * waves, 0, S->stream>>>(
      S->V, S->P, S->fp, per, S->d_fire[S->fireCur], S->d_fire[1 - S->fireCur], S->pos[nb][0], S->pos[nb][1], S->d_fireVel,
      S->d_fireVel + S->V.nv, flagOut, anyOut, S->d_look, look, &S->h_stat->look, tell);
  return hipGetLastError();
}

hipError_t launch_fire_partials(dpm_set_s* S) {
  k_fire_partials<<<grid_w(S->V.ntiles), 256, 0, S->stream>>>(S->V, S->d_part);
  return hipGetLastError();
}

hipError_t launch_fire_sys(dpm_set_s* S, int chunk, int waves) {
  const int threads = WAVE * (waves < 1 ? 1 : (waves > FS_WAVES ? FS_WAVES : waves));
  switch (S->P.interaction) {
    case INT_VV: return fire_pot<INT_VV>(S, chunk, threads);
    case INT_SMOOTH: return fire_pot<INT_SMOOTH>(S, chunk, threads);
    default: return fire_pot<INT_ALL>(S, chunk, threads);
  }
}

hipError_t launch_fire_resume(dpm_set_s* S) {
  k_fire_resume<<<grid_v(S->nsys), 256, 0, S->stream>>>(S->d_fire[S->fireCur], (int)S->nsys);
  return hipGetLastError();
}

StepArgs loop_args(dpm_set_s* S) {
  const int b = S->cur;
  StepArgs A{};
  A.h = 0.5 * S->P.dt;
  A.dt = S->P.dt;
  A.xout = S->pos[1 - b][0];
  A.yout = S->pos[1 - b][1];
  A.flagCur = S->d_flag[b];
  A.flagOut = S->d_flag[1 - b];
  A.anyOut = S->d_any + 1 - b;
  A.cellCur = S->G.count[b];
  A.slotsCur = S->G.slots;
  A.cellOther = S->G.count[1 - b];
  A.ctr = S->d_ctr;
  A.ctrOffT = -1;  // k_bin has bumped the counters of this step
  A.ctrOffA = -1;
  A.err = S->d_err;
  A.maxcnt = S->d_maxcnt;
  A.updateCount = S->d_updateCount;
  A.manage = 1;
  A.xcd = S->xcdMap;
  return A;
}

hipError_t launch_fire_step(dpm_set_s* S) {
  StepArgs A = loop_args(S);
  A.fire = S->d_fire[S->fireCur];
  A.part = S->d_part;
  return launch_step(S, MODE_FIRE, A);
}

}  // namespace dpm
