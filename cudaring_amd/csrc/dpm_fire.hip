// dpm_fire.hip -- the persistent FIRE kernel, compiled once per (interaction, potential): FIRE_INTER and
// FIRE_POT select the instance.
#include <algorithm>

#include "dpm_forces.h"
#include "dpm_launch.h"
#include "dpm_near.h"

namespace dpm {

// One workgroup per system runs whole FIRE iterations (FIRE::minimizerVertexLoop,
// FIRE.cu:397-411) back to back, separated by workgroup barriers only: systems share nothing,
// so no grid-wide synchronisation is needed and a converged system's workgroup simply exits.
// Each wave walks the system's ring-aligned tiles.  At most `chunk` iterations per launch; every
// thread carries the system's FIRE state and decides the loop exit from the same values, so all
// waves leave together.
//
// Bound by the vector instructions of one CU: a system of 200 rings is 60 tiles on 16 waves.  So an
// iteration is one pass over the vertices up to the drift and one for the force, with two barriers:
//   * the force phase evaluates the tile's near list (dpm_near.h) instead of whole rows;
//   * |v|^2 after the half kick is summed with v.F at the end of the iteration before (FireSums);
//   * NEAR: the system's positions live in LDS (16 bytes a vertex), where the pair terms read them;
//   * energies, ring geometry and the positions in memory are written once, when the launch ends.
// Terms and sums keep the reference's order of operations and its rounding (quot, root): a minimiser
// amplifies last bits, a thousandfold per ten iterations of a stiff contact.  The loops' short forms and
// |v|^2 + 2 h P + h^2 |F|^2 took 512 packings of 16 to 256 rings through 2 x 60 iterations in 10.0 ms,
// this takes 15.3 (whole rows from memory, four barriers: 19.1), but there single packings of a set left
// the path: forces off by up to 9e-4 after a second compression.
// MAXW: a lane may hold 256 registers with up to 8 waves (200 to 214 in use, nothing spills), 168 with up to
// 12 (23 to 49 spill), 128 with 16 (63 to 114).  Against the 16-wave build alone: 512 packings of 16 to 256
// rings, 200 iterations, 4 waves 93.1 -> 79.2 ms, 8 waves 63.4 -> 51.0, 12 waves 54.1 -> 45.1 (16 waves take
// 47.7); 512 packings of 16 to 24 rings (5 to 9 tiles), 8 waves 8.4 -> 7.5, 9 waves 10.2 -> 7.8.
// Without near lists (rows of more than 64 entries, systems of more vertices than LDS holds, the
// all-pairs interaction) it gathers over whole rows from memory.

// Force on the lane's vertex of tile t (and, STORE, its energy and the ring geometry into memory).
template <int INTER, int POT, bool NEAR, bool STORE, class X>
__device__ __forceinline__ void tile_force(const View& V, const Params& P, const NearRows& N, const Box& B,
                                           const Lane& L, X pos, double* res, double& fx, double& fy) {
  const double2 r = pos(L.v);
  double e = 0, es = 0, qx = 0, qy = 0, qnx = 0, qny = 0;  // sets with wide rings do not run this kernel
  fx = fy = 0;
  if constexpr (NEAR)
    near_wave<INTER, POT, true, STORE>(V, P, N, B, L, pos, res, fx, fy, INTER == INT_SMOOTH ? es : e, qx, qy);
  else
    gather_pairs<INTER, POT, true>(V, P, L, B, r.x, r.y, 0, 1, fx, fy, e, es, qx, qy, qnx, qny);
  const ShapeOut so = ring_shape(V, P, L, B, r.x, r.y, STORE);
  if constexpr (INTER == INT_SMOOTH) {
    fx += shfl_d(qx, L.nl);
    fy += shfl_d(qy, L.nl);
    if constexpr (STORE) {
      const double pe = seg_sum(L.act ? es : 0.0, L.lane, L.segS, L.segE);
      if (L.act) {
        V.es[L.v] = es;
        if (L.lane == L.segS) V.pe[L.r] = pe;
      }
    }
  }
  fx = so.fx + fx;
  fy = so.fy + fy;
  if (STORE && L.act) V.ev[L.v] = so.e + e;
}

template <int INTER, int POT, bool NEAR, int MAXW>
__global__ __launch_bounds__(WAVE* MAXW) void k_fire_sys(View V, Params P, FireParams fp, CellGrid G, NearRows N,
                                                             FireState* fst, int chunk, int* updateCount, int* err,
                                                             int* maxcnt, const int* order) {
  // NEAR: per wave near_wave_doubles, then the positions, both read and written as double2
  extern __shared__ __align__(16) double dyn[];
  static_assert(__alignof__(dyn) % alignof(double2) == 0, "128-bit LDS accesses");
  __shared__ double red[MAXW][5];
  __shared__ int movedFlag[2];
  const int s = order[blockIdx.x];
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  const int t0 = V.stile[s], t1 = V.stile[s + 1], b0 = V.svoff[s];
  const Box B = box_of(V, s);
  double* res = dyn + w * near_wave_doubles<INTER>();
  double2* lpos = (double2*)(dyn + nw * near_wave_doubles<INTER>());
  auto pos = [&](int v) -> double2 {
    if constexpr (NEAR) return lpos[v - b0];
    else return make_double2(V.x[v], V.y[v]);
  };
  FireState fs = fst[s];
  FireSums a{0, -1, 0, 0, 0};
  const FireNext first(fp, fs);
  if (threadIdx.x < 2) movedFlag[threadIdx.x] = 0;
  for (int t = t0 + w; t < t1; t += nw) {
    Lane L;
    lane_ctx(V, t, lane, L);
    if (L.act) {
      fire_add(a, first, V.vx[L.v], V.vy[L.v], V.fx[L.v], V.fy[L.v]);
      if constexpr (NEAR) lpos[L.v - b0] = make_double2(V.x[L.v], V.y[L.v]);
    }
    if constexpr (NEAR) build_near_wave<INTER>(V, P, N, L, B, V.lx, V.ly, G.brute[s] != 0);
  }
  FireSums sum = fire_block_sums(a, red, nw);
  bool ran = false;
  for (int it = 0; it < chunk; it++) {
    // ---- checkFIREParams (FIRE.cu:338-371) and the stopping rule
    const bool reset = fire_update(fs, fp, sum);
    if (fs.converged) break;
    ran = true;
    const double h = 0.5 * fs.dt;
    // ---- back-step on reset, half kick, mixing, drift, displacement test
    int moved = 0;
    for (int t = t0 + w; t < t1; t += nw) {
      const int v = V.tile_v0[t] + lane;
      if (v < V.tile_v1[t]) {
        double vx = V.vx[v], vy = V.vy[v];
        const double fx = V.fx[v], fy = V.fy[v], lx = V.lx[v], ly = V.ly[v];
        double2 r = pos(v);
        fire_move(fs, sum, reset, fx, fy, r.x, r.y, vx, vy);
        V.vx[v] = vx;
        V.vy[v] = vy;
        if constexpr (NEAR) {
          lpos[v - b0] = r;
        } else {
          V.x[v] = r.x;
          V.y[v] = r.y;
        }
        if (moved_past(P, B, r.x - lx, r.y - ly)) moved = 1;
      }
    }
    if (moved) movedFlag[it & 1] = 1;
    __syncthreads();
    const bool rebuild = movedFlag[it & 1] != 0;
    if (threadIdx.x == 0) movedFlag[1 - (it & 1)] = 0;
    // ---- checkNeighbors: rebuild the system's rows from cells binned here (DPM2D.cu:1408-1423)
    if (rebuild) {
      const int ncx = G.ncx[s], ncy = G.ncy[s];
      int* count = G.count[0];
      for (int t = t0 + w; t < t1; t += nw) {
        const int v = V.tile_v0[t] + lane;
        if (v < V.tile_v1[t]) {
          const double2 r = pos(v);
          if constexpr (NEAR) {
            V.x[v] = r.x;
            V.y[v] = r.y;
          }
          bin_vertex(G, B, count, G.slots, v, s, r.x, r.y, err);
        }
      }
      __syncthreads();
      for (int t = t0 + w; t < t1; t += nw) {
        Lane L;
        lane_ctx(V, t, lane, L);
        if (L.act) build_row(V, P, G, count, G.slots, L.v, s, B, err, maxcnt);
        if constexpr (NEAR) build_near_wave<INTER>(V, P, N, L, B, V.x, V.y, G.brute[s] != 0);
      }
      __syncthreads();
      if (!G.brute[s])
        for (int c = threadIdx.x; c < ncx * ncy; c += blockDim.x) count[G.coff[s] + c] = 0;
      if (threadIdx.x == 0) updateCount[s] += 1;
    }
    // ---- calcForceEnergy (shape + interaction) and the second half kick
    a = FireSums{0, -1, 0, 0, 0};
    const FireNext next(fp, fs);
    for (int t = t0 + w; t < t1; t += nw) {
      Lane L;
      lane_ctx(V, t, lane, L);
      double fx, fy;
      tile_force<INTER, POT, NEAR, false>(V, P, N, B, L, pos, res, fx, fy);
      if (L.act) {
        const double vx = V.vx[L.v] + h * fx, vy = V.vy[L.v] + h * fy;
        V.fx[L.v] = fx;
        V.fy[L.v] = fy;
        V.vx[L.v] = vx;
        V.vy[L.v] = vy;
        fire_add(a, next, vx, vy, fx, fy);
      }
    }
    sum = fire_block_sums(a, red, nw);
  }
  if (ran) {  // what the last force phase left out
    for (int t = t0 + w; t < t1; t += nw) {
      Lane L;
      lane_ctx(V, t, lane, L);
      double fx, fy;
      tile_force<INTER, POT, NEAR, true>(V, P, N, B, L, pos, res, fx, fy);
      if (NEAR && L.act) {
        const double2 r = pos(L.v);
        V.x[L.v] = r.x;
        V.y[L.v] = r.y;
      }
    }
  }
  if (threadIdx.x == 0) fst[s] = fs;
}

#if !defined(FIRE_INTER) || !defined(FIRE_POT)
#error "compile with -DFIRE_INTER and -DFIRE_POT"
#endif
template <int MAXW>
static hipError_t fire_waves_launch(dpm_set_s* S, int chunk, int threads) {
  const unsigned g = (unsigned)S->nsys;
#if FIRE_INTER != 3
  int most = 0;
  for (long s = 0; s < S->nsys; s++) most = std::max(most, S->h_svoff[s + 1] - S->h_svoff[s]);
  const size_t lds = (size_t)(threads / WAVE) * near_wave_doubles<FIRE_INTER>() * sizeof(double) +
                     (size_t)most * sizeof(double2);
  if (S->N.task && lds <= kFireLds) {
    auto k = k_fire_sys<FIRE_INTER, FIRE_POT, true, MAXW>;
    hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFireLds);
    if (e != hipSuccess) return e;
    k<<<g, threads, lds, S->stream>>>(S->V, S->P, S->fp, S->G, S->N, S->d_fire[S->fireCur], chunk, S->d_updateCount,
                                      S->d_err, S->d_maxcnt, S->d_sysOrder);
    return hipGetLastError();
  }
#endif
  k_fire_sys<FIRE_INTER, FIRE_POT, false, MAXW>
      <<<g, threads, 0, S->stream>>>(S->V, S->P, S->fp, S->G, S->N, S->d_fire[S->fireCur], chunk, S->d_updateCount,
                                     S->d_err, S->d_maxcnt, S->d_sysOrder);
  return hipGetLastError();
}

template <>
hipError_t fire_launch<FIRE_INTER, FIRE_POT>(dpm_set_s* S, int chunk, int threads) {
  if (threads <= WAVE * FS_WAVES_FEW) return fire_waves_launch<FS_WAVES_FEW>(S, chunk, threads);
  if (threads <= WAVE * FS_WAVES_SOME) return fire_waves_launch<FS_WAVES_SOME>(S, chunk, threads);
  return fire_waves_launch<FS_WAVES>(S, chunk, threads);
}

}  // namespace dpm
