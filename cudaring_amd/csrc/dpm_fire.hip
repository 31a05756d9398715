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
//   * the force phase evaluates the tile's near list (dpm_near.h), in the loops' short forms where the
//     contacts are soft (a minimiser amplifies last bits a thousandfold per ten iterations of a stiff
//     one, and the split FIRE step keeps the reference's order);
//   * |v|^2 after the half kick is |v|^2 + 2 h P + h^2 |F|^2 (h^2 |F|^2 after a restart), from the sums
//     made with P at the end of the iteration before: P > 0, so nothing cancels;
//   * NEAR: the system's positions live in LDS (16 bytes a vertex), where the pair terms read them;
//   * energies, ring geometry and the positions in memory are written once, when the launch ends.
// Without near lists (rows of more than 64 entries, systems of more vertices than LDS holds, the
// all-pairs interaction) it gathers over whole rows from memory.

struct FireSums {
  double P, vv, ff, m;  // v.F, |v|^2, |F|^2, max F_c^2
};

// workgroup sums of P, vv, ff and maximum of m (fixed order: lanes by butterfly, waves by index);
// every thread passes another barrier between two calls
__device__ __forceinline__ FireSums block_sums(FireSums a, double (*red)[4]) {
  const int w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    a.P += __shfl_xor(a.P, d, WAVE);
    a.vv += __shfl_xor(a.vv, d, WAVE);
    a.ff += __shfl_xor(a.ff, d, WAVE);
    a.m = fmax(a.m, __shfl_xor(a.m, d, WAVE));
  }
  if ((threadIdx.x & (WAVE - 1)) == 0) {
    red[w][0] = a.P;
    red[w][1] = a.vv;
    red[w][2] = a.ff;
    red[w][3] = a.m;
  }
  __syncthreads();
  FireSums s{0, 0, 0, -1};
  for (int q = 0; q < nw; q++) {
    s.P += red[q][0];
    s.vv += red[q][1];
    s.ff += red[q][2];
    s.m = fmax(s.m, red[q][3]);
  }
  return s;
}

__device__ __forceinline__ void add_vertex(FireSums& a, double vx, double vy, double fx, double fy) {
  a.P += vx * fx + vy * fy;
  a.vv += vx * vx + vy * vy;
  a.ff += fx * fx + fy * fy;
  a.m = fmax(a.m, fmax(fx * fx, fy * fy));
}

template <int INTER, int POT>
constexpr bool fire_ref() {
  return INTER == INT_SMOOTH || POT == POT_LJ || POT == POT_WCA;
}

// Force on the lane's vertex of tile t (and, STORE, its energy and the ring geometry into memory).
template <int INTER, int POT, bool NEAR, bool STORE, class X>
__device__ __forceinline__ void tile_force(const View& V, const Params& P, const NearRows& N, const Box& B,
                                           const Lane& L, X pos, double* res, double& fx, double& fy) {
  constexpr bool REF = fire_ref<INTER, POT>();
  const double2 r = pos(L.v);
  double e = 0, es = 0, qx = 0, qy = 0, qnx = 0, qny = 0;  // sets with wide rings do not run this kernel
  fx = fy = 0;
  if constexpr (NEAR)
    near_wave<INTER, POT, REF, STORE>(V, P, N, B, L, pos, res, fx, fy, INTER == INT_SMOOTH ? es : e, qx, qy);
  else
    gather_pairs<INTER, POT, REF>(V, P, L, B, r.x, r.y, 0, 1, fx, fy, e, es, qx, qy, qnx, qny);
  ShapeOut so;
  if constexpr (REF) so = ring_shape(V, P, L, B, r.x, r.y, STORE);
  else so = ring_shape_n(V, P, L, B, r.x, r.y, STORE);
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

template <int INTER, int POT, bool NEAR>
__global__ __launch_bounds__(WAVE* FS_WAVES) void k_fire_sys(View V, Params P, FireParams fp, CellGrid G, NearRows N,
                                                             FireState* fst, int chunk, int* updateCount, int* err,
                                                             int* maxcnt, const int* order) {
  extern __shared__ double dyn[];  // NEAR: per wave near_wave_doubles, then the positions
  __shared__ double red[FS_WAVES][4];
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
  FireSums a{0, 0, 0, -1};
  if (threadIdx.x < 2) movedFlag[threadIdx.x] = 0;
  for (int t = t0 + w; t < t1; t += nw) {
    Lane L;
    lane_ctx(V, t, lane, L);
    if (L.act) {
      add_vertex(a, V.vx[L.v], V.vy[L.v], V.fx[L.v], V.fy[L.v]);
      if constexpr (NEAR) lpos[L.v - b0] = make_double2(V.x[L.v], V.y[L.v]);
    }
    if constexpr (NEAR) build_near_wave<INTER>(V, P, N, L, B, V.lx, V.ly, G.brute[s] != 0);
  }
  FireSums sum = block_sums(a, red);
  bool ran = false;
  for (int it = 0; it < chunk; it++) {
    // ---- checkFIREParams (FIRE.cu:338-371) and the stopping rule
    if (!fs.converged && (sqrt(sum.m) <= fp.tol || fs.iters >= fp.maxIter)) fs.converged = 1;
    if (fs.converged) break;
    ran = true;
    const bool reset = !(sum.P > 0);
    fs.P = sum.P;
    if (!reset) {
      fs.numStep++;
      if (fs.numStep > fp.minStep) {
        fs.dt = fmin(fs.dt * fp.f_inc, fp.dt_max);
        fs.a *= fp.f_a;
      }
    } else {
      fs.numStep = 0;
      fs.dt = fmax(fs.dt * fp.f_dec, fp.dt_max / 10);
      fs.a = fp.a_start;
    }
    fs.iters++;
    const double dt = fs.dt, h = 0.5 * dt, fa = fs.a;
    // ---- back-step on reset (with the decreased dt), half kick, bendVertexVelocityTowardsForce
    // (FIRE.cu:374-394), drift, displacement test
    const double VV = reset ? h * h * sum.ff : sum.vv + 2 * h * sum.P + h * h * sum.ff;
    const double bend = sum.ff > 0 ? fa * sqrt(VV / sum.ff) : 0.0, keep = sum.ff > 0 ? 1 - fa : 1.0;
    int moved = 0;
    for (int t = t0 + w; t < t1; t += nw) {
      const int v = V.tile_v0[t] + lane;
      if (v < V.tile_v1[t]) {
        double vx = V.vx[v], vy = V.vy[v];
        const double fx = V.fx[v], fy = V.fy[v], lx = V.lx[v], ly = V.ly[v];
        double2 r = pos(v);
        if (reset) {
          r.x -= h * vx;
          r.y -= h * vy;
          vx = 0;
          vy = 0;
        }
        vx = keep * (vx + h * fx) + bend * fx;
        vy = keep * (vy + h * fy) + bend * fy;
        r.x += dt * vx;
        r.y += dt * vy;
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
    a = FireSums{0, 0, 0, -1};
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
        add_vertex(a, vx, vy, fx, fy);
      }
    }
    sum = block_sums(a, red);
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
template <>
hipError_t fire_launch<FIRE_INTER, FIRE_POT>(dpm_set_s* S, int chunk, int threads) {
  const unsigned g = (unsigned)S->nsys;
#if FIRE_INTER != 3
  int most = 0;
  for (long s = 0; s < S->nsys; s++) most = std::max(most, S->h_svoff[s + 1] - S->h_svoff[s]);
  const size_t lds = (size_t)(threads / WAVE) * near_wave_doubles<FIRE_INTER>() * sizeof(double) +
                     (size_t)most * sizeof(double2);
  if (S->N.task && lds <= kFireLds) {
    auto k = k_fire_sys<FIRE_INTER, FIRE_POT, true>;
    hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFireLds);
    if (e != hipSuccess) return e;
    k<<<g, threads, lds, S->stream>>>(S->V, S->P, S->fp, S->G, S->N, S->d_fire[S->fireCur], chunk, S->d_updateCount,
                                      S->d_err, S->d_maxcnt, S->d_sysOrder);
    return hipGetLastError();
  }
#endif
  k_fire_sys<FIRE_INTER, FIRE_POT, false>
      <<<g, threads, 0, S->stream>>>(S->V, S->P, S->fp, S->G, S->N, S->d_fire[S->fireCur], chunk, S->d_updateCount,
                                     S->d_err, S->d_maxcnt, S->d_sysOrder);
  return hipGetLastError();
}

}  // namespace dpm
