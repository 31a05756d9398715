// dpm_fire.hip -- the persistent FIRE kernel, compiled once per (interaction, potential): FIRE_INTER and
// FIRE_POT select the instance.
#include "dpm_forces.h"
#include "dpm_launch.h"

namespace dpm {

// ------------------------------------------------------- persistent FIRE ---
// One workgroup per system runs whole FIRE iterations (FIRE::minimizerVertexLoop,
// FIRE.cu:397-411) back to back, separated by workgroup barriers only: systems share nothing,
// so no grid-wide synchronisation is needed and a converged system's workgroup simply exits.
// Each wave walks the system's ring-aligned tiles; the force phase is the step kernel's
// (ring_shape + gather_pairs).  At most `chunk` iterations per launch; every thread decides the
// loop exit from the same FIRE state, so all waves leave together.
// Two builds: up to 8 waves per system (about 190 VGPRs, no spills) and up to 16 (the 1024-lane
// workgroup caps a wave at 128 VGPRs, so 40-75 of them spill to scratch; halving the tiles each
// wave walks still makes an iteration about 12% shorter on systems of 76 tiles).

// Workgroup reductions of the persistent kernel, with one barrier each: a caller alternates two
// exchange buffers `red`, so that between two exchanges through the same buffer every thread
// passes another barrier (no exchange overwrites one that a wave is still reading).
// workgroup sum of a and maximum of b (fixed order: lanes by butterfly, waves by index)
__device__ __forceinline__ void block_sum_max(double a, double b, double (*red)[2], double& sa, double& mb) {
  const int w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  a = wave_sum(a);
  b = wave_max(b);
  if ((threadIdx.x & (WAVE - 1)) == 0) {
    red[w][0] = a;
    red[w][1] = b;
  }
  __syncthreads();
  double s = 0, m = -1;
  for (int q = 0; q < nw; q++) {
    s += red[q][0];
    m = fmax(m, red[q][1]);
  }
  sa = s;
  mb = m;
}

// workgroup sums of a and of b in one exchange (the order of block_sum_max's sum for each)
__device__ __forceinline__ void block_sum_sum(double a, double b, double (*red)[2], double& sa, double& sb) {
  const int w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  a = wave_sum(a);
  b = wave_sum(b);
  if ((threadIdx.x & (WAVE - 1)) == 0) {
    red[w][0] = a;
    red[w][1] = b;
  }
  __syncthreads();
  double s = 0, t = 0;
  for (int q = 0; q < nw; q++) {
    s += red[q][0];
    t += red[q][1];
  }
  sa = s;
  sb = t;
}

// P = v.F and max F_c^2 over the system's vertices
__device__ __forceinline__ void fire_power(const View& V, int t0, int t1, double (*red)[2], double& P, double& Fm) {
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  double p = 0, m = -1;
  for (int t = t0 + w; t < t1; t += nw) {
    const int v = V.tile_v0[t] + lane;
    if (v < V.tile_v1[t]) {
      const double fx = V.fx[v], fy = V.fy[v];
      p += V.vx[v] * fx + V.vy[v] * fy;
      m = fmax(m, fmax(fx * fx, fy * fy));
    }
  }
  block_sum_max(p, m, red, P, Fm);
}

template <int INTER, int POT, int MAXW>
__global__ __launch_bounds__(WAVE* MAXW) void k_fire_sys(View V, Params P, FireParams fp, CellGrid G,
                                                         FireState* fst, int chunk, int* updateCount, int* err,
                                                         int* maxcnt, const int* order) {
  // exchange buffers: [0] for |v|^2 and |F|^2 after the half kick, [1] for P and max F_c^2 after
  // the force (between two exchanges through one buffer every thread passes the other's barrier
  // and the displacement test's)
  __shared__ double red[2][MAXW][2];
  const int s = order[blockIdx.x];
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  const int t0 = V.stile[s], t1 = V.stile[s + 1];
  const Box B = box_of(V, s);
  // every thread carries the system's FIRE state and updates it from the same reduced values in
  // the same order, so all hold the same state and take the same exit without a barrier
  FireState fs = fst[s];
  double Pv, Fm;
  fire_power(V, t0, t1, red[1], Pv, Fm);
  for (int it = 0; it < chunk; it++) {
    // ---- checkFIREParams (FIRE.cu:338-371) and the stopping rule
    if (!fs.converged && (sqrt(Fm) <= fp.tol || fs.iters >= fp.maxIter)) fs.converged = 1;
    if (fs.converged) break;
    int reset = 0;
    fs.P = Pv;
    if (Pv > 0) {
      fs.numStep++;
      if (fs.numStep > fp.minStep) {
        fs.dt = fmin(fs.dt * fp.f_inc, fp.dt_max);
        fs.a *= fp.f_a;
      }
    } else {
      fs.numStep = 0;
      fs.dt = fmax(fs.dt * fp.f_dec, fp.dt_max / 10);
      fs.a = fp.a_start;
      reset = 1;
    }
    fs.iters++;
    const double dt = fs.dt, h = 0.5 * dt, fa = fs.a;
    // ---- back-step on reset (with the decreased dt), half kick, |v|^2 and |F|^2
    double vv = 0, ff = 0;
    for (int t = t0 + w; t < t1; t += nw) {
      const int v = V.tile_v0[t] + lane;
      if (v < V.tile_v1[t]) {
        double vx = V.vx[v], vy = V.vy[v];
        const double fx = V.fx[v], fy = V.fy[v];
        if (reset) {
          V.x[v] -= h * vx;
          V.y[v] -= h * vy;
          vx = 0;
          vy = 0;
        }
        vx += h * fx;
        vy += h * fy;
        V.vx[v] = vx;
        V.vy[v] = vy;
        vv += vx * vx + vy * vy;
        ff += fx * fx + fy * fy;
      }
    }
    double VV, FF;
    block_sum_sum(vv, ff, red[0], VV, FF);
    // ---- bendVertexVelocityTowardsForce (FIRE.cu:374-394), drift, displacement test
    int moved = 0;
    for (int t = t0 + w; t < t1; t += nw) {
      const int v = V.tile_v0[t] + lane;
      if (v < V.tile_v1[t]) {
        double vx = V.vx[v], vy = V.vy[v];
        if (FF > 0) {
          const double ratio = sqrt(VV / FF);
          vx = (1 - fa) * vx + fa * V.fx[v] * ratio;
          vy = (1 - fa) * vy + fa * V.fy[v] * ratio;
        }
        const double xn = V.x[v] + dt * vx, yn = V.y[v] + dt * vy;
        V.vx[v] = vx;
        V.vy[v] = vy;
        V.x[v] = xn;
        V.y[v] = yn;
        if (moved_past(P, B, xn - V.lx[v], yn - V.ly[v])) moved = 1;
      }
    }
    // ---- checkNeighbors: rebuild the system's rows from cells binned here (DPM2D.cu:1408-1423)
    if (__syncthreads_or(moved)) {
      const int ncx = G.ncx[s], ncy = G.ncy[s];
      int* count = G.count[0];
      if (!G.brute[s]) {
        for (int t = t0 + w; t < t1; t += nw) {
          const int v = V.tile_v0[t] + lane;
          if (v < V.tile_v1[t]) {
            int cx, cy;
            cell_of(V.x[v], V.y[v], B, ncx, ncy, cx, cy);
            const int c = G.coff[s] + cy * ncx + cx;
            const int slot = atomicAdd(&count[c], 1);
            if (slot < G.cap) G.slots[(long)c * G.cap + slot] = v;
            else atomicOr(err, ERR_CELL_OVERFLOW);
          }
        }
      }
      __syncthreads();
      for (int t = t0 + w; t < t1; t += nw) {
        const int v = V.tile_v0[t] + lane;
        if (v < V.tile_v1[t]) build_row(V, P, G, count, G.slots, v, s, B, err, maxcnt);
      }
      __syncthreads();
      if (!G.brute[s])
        for (int c = threadIdx.x; c < ncx * ncy; c += blockDim.x) count[G.coff[s] + c] = 0;
      if (threadIdx.x == 0) updateCount[s] += 1;
    }
    // ---- calcForceEnergy (shape + interaction) and the second half kick
    double p = 0, m = -1;
    for (int t = t0 + w; t < t1; t += nw) {
      Lane L;
      lane_ctx(V, t, lane, L);
      const double x = V.x[L.v], y = V.y[L.v];
      double fx = 0, fy = 0, e = 0, es = 0, qx = 0, qy = 0;
      double qnx = 0, qny = 0;  // sets with wide rings do not run this kernel
      gather_pairs<INTER, POT, true>(V, P, L, B, x, y, 0, 1, fx, fy, e, es, qx, qy, qnx, qny);
      const ShapeOut so = ring_shape(V, P, L, B, x, y, true);
      if constexpr (INTER == INT_SMOOTH) {
        fx += shfl_d(qx, L.nl);
        fy += shfl_d(qy, L.nl);
        const double pe = seg_sum(L.act ? es : 0.0, L.lane, L.segS, L.segE);
        if (L.act) {
          V.es[L.v] = es;
          if (L.lane == L.segS) V.pe[L.r] = pe;
        }
      }
      fx = so.fx + fx;
      fy = so.fy + fy;
      if (L.act) {
        const double vx = V.vx[L.v] + h * fx, vy = V.vy[L.v] + h * fy;
        V.fx[L.v] = fx;
        V.fy[L.v] = fy;
        V.ev[L.v] = so.e + e;
        V.vx[L.v] = vx;
        V.vy[L.v] = vy;
        p += vx * fx + vy * fy;
        m = fmax(m, fmax(fx * fx, fy * fy));
      }
    }
    block_sum_max(p, m, red[1], Pv, Fm);
  }
  if (threadIdx.x == 0) fst[s] = fs;
}

#if !defined(FIRE_INTER) || !defined(FIRE_POT)
#error "compile with -DFIRE_INTER and -DFIRE_POT"
#endif
template <>
hipError_t fire_launch<FIRE_INTER, FIRE_POT>(dpm_set_s* S, int chunk, int threads) {
  if (threads > WAVE * FS_WAVES)
    k_fire_sys<FIRE_INTER, FIRE_POT, FS_WAVES_WIDE><<<(unsigned)S->nsys, threads, 0, S->stream>>>(
        S->V, S->P, S->fp, S->G, S->d_fire[S->fireCur], chunk, S->d_updateCount, S->d_err, S->d_maxcnt,
        S->d_sysOrder);
  else
    k_fire_sys<FIRE_INTER, FIRE_POT, FS_WAVES><<<(unsigned)S->nsys, threads, 0, S->stream>>>(
        S->V, S->P, S->fp, S->G, S->d_fire[S->fireCur], chunk, S->d_updateCount, S->d_err, S->d_maxcnt,
        S->d_sysOrder);
  return hipGetLastError();
}

}  // namespace dpm
