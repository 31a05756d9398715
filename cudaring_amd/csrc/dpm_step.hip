// dpm_step.hip -- the step kernel, compiled once per (interaction, potential): STEP_INTER and
// STEP_POT select the instance, whose launcher is a specialisation of step_launch.
#include "dpm_forces.h"
#include "dpm_launch.h"
#include "dpm_near.h"

namespace dpm {

// Single force calls and the vertex FIRE steps keep the reference's order of operations, over whole rows
// with a fixed number of waves too (whose sums they set).
template <int MODE>
constexpr bool step_ref() {
  return (MODE & (MODE_KICK | MODE_BROWN)) == 0 && (MODE & (MODE_RIGID | MODE_NEAR)) != (MODE_RIGID | MODE_NEAR);
}

// Whether the launch stores the force, energies, ring geometry and wall forces: what is read after a
// loop.  A step of a velocity-Verlet, Langevin, BAOAB or rigid loop other than its last consumes the
// force it computes (the closing and next opening half kicks); on near lists the overdamped loops and
// FIRE store in a launch of MODE_OUT only.
template <int MODE>
constexpr bool step_store() {
  if ((MODE & MODE_NEAR) != 0 && (MODE & MODE_RIGID) == 0 && (MODE & (MODE_BROWN | MODE_FIRE)) != 0)
    return (MODE & MODE_OUT) != 0;
  return (MODE & MODE_START) == 0 || (MODE & MODE_BROWN) != 0;
}

template <int INTER, int POT, int MODE>
__global__ __launch_bounds__(WAVE* MAXSPLIT) void k_step(View V, Params P, StepArgs A, CellGrid G) {
  // partials of gather waves 1..nw-1: red[((w - 1) * 6 + q) * WAVE + lane], sized by the launch; near
  // lists' results as double2
  extern __shared__ __align__(16) double red[];
  static_assert(__alignof__(red) % alignof(double2) == 0, "128-bit LDS accesses");
  const int w = threadIdx.x / WAVE;
  const int nw = blockDim.x / WAVE;
  Lane L;
  constexpr bool WIDE = (MODE & MODE_WIDE) != 0;
  constexpr bool NEAR = (MODE & MODE_NEAR) != 0;
  constexpr bool REF = step_ref<MODE>();
  constexpr int MB = MODE & ~(MODE_WIDE | MODE_NEAR | MODE_OUT);  // the integrator mode
  constexpr bool STORE = step_store<MODE>();
  lane_ctx<WIDE>(V, A.xcd ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x, threadIdx.x & (WAVE - 1), L);
  const Box B = box_of(V, L.s);
  // own position first: the row rebuild below does not change it, so its load overlaps the
  // rebuild-flag load instead of waiting behind it
  const double x = V.x[L.v], y = V.y[L.v];

  // loop bookkeeping: clear flags (and cells) for later steps, count this step's rebuild, rebuild rows
  if (A.manage) {
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (A.cellOther)
      for (int c = gid; c < G.ncells; c += gridDim.x * blockDim.x) A.cellOther[c] = 0;
    if (A.flagClear)
      for (int t = gid; t < V.nsys; t += gridDim.x * blockDim.x) A.flagClear[t] = 0;
    const int flag = A.flagCur[L.s];
    const bool rebuild = (flag & 1) != 0;
    // a system flagged FLAG_FAR searches all its vertices instead of cells that may miss a
    // neighbour (the reference's all-pairs search)
    const bool allPairs = A.staleCheck && (flag & FLAG_FAR) != 0;
    const int* cells = A.cellCur;
    const int* slots = A.slotsCur;
    if (A.genCur) {
      // step loop: rows from the cells of the list positions (md_cells)
      const int g = A.genCur[L.s];
      if (L.tile == V.stile[L.s] && threadIdx.x == 0) A.genOut[L.s] = rebuild ? g + 1 : g;
      if (rebuild) {
        const MdCells M = md_cells(A.cellCur, A.slotsCur, G, g);
        cells = M.cnt;
        slots = M.slots;
        if (!A.rowsBuilt) {
          if (w == 0 && L.act && !allPairs) md_stale_test(V, P, B, L.v, x, y, A.err);
        }
      }
    }
    if (rebuild && L.tile == V.stile[L.s] && threadIdx.x == 0) A.updateCount[L.s] += 1;
    // the cell search shared by the tile's waves (rows in LDS) where the launch sized LDS for it
    const bool tileBuild = rebuild && !A.rowsBuilt && !allPairs && A.rowsLdsW == V.W && !G.brute[L.s];
    if (tileBuild) {
      build_rows_tile<NEAR ? INTER : -1>(V, P, G, cells, slots, L, w, nw, B, x, y, (int*)red, A.err, nullptr, A.near);
    } else if (rebuild && w == 0 && L.act && !A.rowsBuilt) {
      build_row(V, P, G, cells, slots, L.v, L.s, B, A.err, nullptr, allPairs);
    }
    if (rebuild) __syncthreads();
    if constexpr (NEAR) {
      if (rebuild && !tileBuild) {
        build_near_tile<INTER>(V, P, A.near, L, w, nw, B, V.x, V.y, G.brute[L.s] != 0, red);
        __syncthreads();
      }
    }
    if (rebuild && A.genCur && !A.rowsBuilt && w == nw - 1)
      md_bin_rebuilt(V, G, md_cells(A.cellCur, A.slotsCur, G, A.genCur[L.s]), L, B, x, y, A.err);
  }
  // FIRE on every tile: a converged system's positions, forces and partials stay as they are
  if constexpr (NEAR && (MODE & MODE_FIRE) != 0 && (MODE & (MODE_RIGID | MODE_OUT)) == 0)
    if (A.fire[L.s].converged) return;
  // wave 0's epilogue operands, fetched before the force work (lastPos after the rebuild above)
  double vx = 0, vy = 0, lx = 0, ly = 0;
  if (w == 0) {
    if constexpr (MB != MODE_FORCE && (MODE & MODE_RIGID) == 0) {
      constexpr bool MOVED = NEAR && MB == MODE_FIRE;  // the velocities k_fire_move wrote
      vx = MOVED ? A.vel[L.v] : V.vx[L.v];
      vy = MOVED ? A.vel[V.nv + L.v] : V.vy[L.v];
    }
    if constexpr ((MODE & MODE_START) != 0) {
      lx = V.lx[L.v];
      ly = V.ly[L.v];
    }
  }

  // gather partials: force on v, vertex-vertex energy, smooth energy, share for prev(v)
  double fx = 0, fy = 0, e = 0, es = 0, qx = 0, qy = 0, qnx = 0, qny = 0;
  const int g0 = nw > 1 ? 1 : 0;
  const int ng = nw - g0;
  // partials per gather wave: six, eight when the tile is a slice of a wide ring
  constexpr int nq = (INTER == INT_SMOOTH && WIDE) ? 8 : 6;
  int2 cnt = make_int2(0, 0);
  int spanT = 0, spanO = 0;
  if constexpr (NEAR) {
    cnt = A.near.tcnt[L.tile];
    if (w == 0 && L.act) {
      spanT = A.near.span[L.v];
      if constexpr (INTER == INT_SMOOTH) spanO = A.near.span[V.nv + L.v];
    }
    if (w >= g0) eval_near<INTER, POT, REF, STORE>(V, P, A.near, B, L.tile, L.v0, cnt, 0, L.lane, w - g0, ng, red);
  } else {
    if (w >= g0) gather_pairs<INTER, POT, REF>(V, P, L, B, x, y, w - g0, ng, fx, fy, e, es, qx, qy, qnx, qny);
    if (nw > 1 && w > 0) {
      double* r = red + (w - 1) * nq * WAVE + L.lane;
      r[0 * WAVE] = fx;
      r[1 * WAVE] = fy;
      if constexpr (STORE) {  // energies are outputs only: a step that stores none leaves them out
        r[2 * WAVE] = e;
        r[3 * WAVE] = es;
      }
      r[4 * WAVE] = qx;
      r[5 * WAVE] = qy;
      if (nq == 8) {
        r[6 * WAVE] = qnx;
        r[7 * WAVE] = qny;
      }
    }
  }

  // ---- wave 0: work that does not need the gather, overlapped with it
  ShapeOut so{0, 0, 0};
  double zt0 = 0, zt1 = 0, ang = 0;
  if (w == 0) {
    if constexpr ((MODE & MODE_RIGID) != 0) so = ring_centre(V, L, B, x, y, STORE);
    else if constexpr (REF) so = ring_shape(V, P, L, B, x, y, STORE);
    else so = ring_shape_n(V, P, L, B, x, y, STORE);
    // one thermal draw per integrate call and ring: Langevin::updateThermalVel (Simulator.cu:54-77)
    // and Brownian::updateThermalVel (156-179) after this call's force, counter = call index;
    // BAOAB::updateThermalVel (122-144) in the next call's first half, whose index is one more
    const unsigned long long callT = A.ctr[0] + (unsigned long long)A.ctrOffT;
    const unsigned long long callA = A.ctr[1] + (unsigned long long)A.ctrOffA;
    if constexpr ((MODE & MODE_LANGEVIN) != 0 || ((MODE & MODE_BAOAB) != 0 && (MODE & MODE_START) != 0))
      gauss_pair(P.seed, (uint32_t)L.s, TAG_THERMAL, callT, (uint32_t)(L.r - V.sroff[L.s]), zt0, zt1);
    // rigid Langevin: this step's pair (RigidLangevin::integrate draws it before its first half)
    if constexpr ((MODE & MODE_RIGID) != 0 && (MODE & MODE_KICK) != 0)
      if (A.rigidLangevin)
        gauss_pair(P.seed, (uint32_t)L.s, TAG_THERMAL, callT, (uint32_t)(L.r - V.sroff[L.s]), zt0, zt1);
    if (P.geometry != GEOM_NORMAL) {  // walls, after the interactions (DPM2D.cu:2090-2103)
      double wfx, wfy;
      so.e += wall_forces(P, B, x, y, V.rad[L.v], so.fx, so.fy, wfx, wfy);
      if (STORE && L.act) {
        V.wfx[L.v] = wfx;
        V.wfy[L.v] = wfy;
      }
    }
    if (P.particle == PART_ACTIVE_SHAPE && L.act) {  // updateRestLength, DPM2D.cu:2037-2056
      double z0, z1;
      gauss_pair(P.seed, (uint32_t)L.s, TAG_SHAPE, callA, (uint32_t)(L.r - V.sroff[L.s]), z0, z1);
      const double l0v = V.l0[L.v];
      V.l0[L.v] = l0v + ((l0v - V.l0r[L.v]) / P.l0Tau + sqrt(2. * P.l0Diff / P.dt) * z0) * P.dt;
    }
    if (P.particle == PART_ACTIVE) {  // addSelfPropulsion, DPM2D.cu:1995-2035
      const double amplitude = (P.taup != 0) ? sqrt(2.0 * P.dt / P.taup) : 0.0;
      double z0, z1;
      gauss_pair(P.seed, (uint32_t)L.s, TAG_ACTIVE, callA, (uint32_t)(L.r - V.sroff[L.s]), z0, z1);
      ang = V.ang[L.r];
      ang += amplitude * z0;
      ang = ang + kPI;
      ang = ang - 2.0 * kPI * floor(ang / (2.0 * kPI));
      ang = ang - kPI;
      // the store depends on every lane's load of the old angle, which has returned
      if (L.act && L.lane == L.segS) V.ang[L.r] = ang;
    }
  }
  if constexpr (NEAR) {
    // windows of NEAR_WIN evaluations per role (one, unless the tile is unusually crowded)
    const int most = max(cnt.x, cnt.y);
    for (int base = 0;;) {
      __syncthreads();
      if (w == 0) sum_near<INTER, STORE>(spanT, spanO, base, red, fx, fy, INTER == INT_SMOOTH ? es : e, qx, qy);
      base += NEAR_WIN;
      if (base >= most) break;
      __syncthreads();
      if (w >= g0) eval_near<INTER, POT, REF, STORE>(V, P, A.near, B, L.tile, L.v0, cnt, base, L.lane, w - g0, ng, red);
    }
    if (w > 0) return;
  } else if (nw > 1) {
    __syncthreads();
    if (w > 0) return;
    for (int q = 1; q < nw; q++) {
      const double* r = red + (q - 1) * nq * WAVE + L.lane;
      fx += r[0 * WAVE];
      fy += r[1 * WAVE];
      if constexpr (STORE) {
        e += r[2 * WAVE];
        es += r[3 * WAVE];
      }
      qx += r[4 * WAVE];
      qy += r[5 * WAVE];
      if (nq == 8) {
        qnx += r[6 * WAVE];
        qny += r[7 * WAVE];
      }
    }
  }

  // ---- wave 0: assemble F = shape + interparticle (+ shares from the next lane)
  if constexpr (INTER == INT_SMOOTH) {
    const double sx = shfl_d(qx, L.nl), sy = shfl_d(qy, L.nl);
    const bool fromMemory = L.wide && L.lane == L.segE;  // next(v) in another tile
    fx += fromMemory ? qnx : sx;
    fy += fromMemory ? qny : sy;
    if constexpr (STORE) {
      const double pe = seg_sum(L.act ? es : 0.0, L.lane, L.segS, L.segE);
      if (L.act) {
        V.es[L.v] = es;
        if (L.lane == L.segS && !L.wide) V.pe[L.r] = pe;  // wide rings: k_wide_pe sums es
      }
    }
  }
  if constexpr ((MODE & MODE_RIGID) != 0) {
    rigid_epilogue<MB, INTER == INT_VV, STORE>(V, P, A, L, B, x, y, fx, fy, e, so.cx, so.cy, lx, ly, zt0, zt1);
    return;
  }
  fx = so.fx + fx;
  fy = so.fy + fy;
  e = so.e + e;
  if (P.particle == PART_ACTIVE) {
    double sn, cs;
    sincos(ang, &sn, &cs);
    fx += P.driving * cs;
    fy += P.driving * sn;
  }

  if constexpr ((MODE & MODE_LANGEVIN) != 0 && (MODE & MODE_BROWN) == 0) {
    fx += P.noise * zt0 - P.gamma * vx;
    fy += P.noise * zt1 - P.gamma * vy;
  }
  if constexpr ((MODE & MODE_FIRE) != 0 && (MODE & MODE_OUT) != 0) {
    if (L.act) V.ev[L.v] = e;
    return;
  }
  if constexpr ((MODE & MODE_FIRE) != 0) {
    const FireState fs = A.fire[L.s];
    const double h = 0.5 * fs.dt;
    if (L.act && !fs.converged) {
      vx += h * fx;
      vy += h * fy;
    }
    if constexpr (!NEAR) {  // (the move on near lists sums over the vertices)
      const double pvf = L.act ? (vx * fx + vy * fy) : 0.0;
      const double f2 = L.act ? fmax(fx * fx, fy * fy) : -1.0;
      const double tP = wave_sum(pvf);
      const double tM = wave_max(f2);
      if (L.lane == 0) {
        A.part[L.tile * 4 + 0] = tP;
        A.part[L.tile * 4 + 3] = tM;
      }
    }
    if (!L.act) return;
    V.fx[L.v] = fx; V.fy[L.v] = fy;
    if constexpr (STORE) V.ev[L.v] = e;
    V.vx[L.v] = vx; V.vy[L.v] = vy;
    return;
  }
  if (!L.act) return;
  if constexpr (STORE) {
    V.fx[L.v] = fx;
    V.fy[L.v] = fy;
    V.ev[L.v] = e;
  }
  if constexpr (MB == MODE_FORCE) return;
  if constexpr ((MODE & MODE_BROWN) != 0) {
    // overdamped velocity (Brownian: (F + noise xi) / gamma; driven: F / gamma), then the drift
    if constexpr ((MODE & MODE_LANGEVIN) != 0) {
      vx = (fx + P.noise * zt0) / P.gamma;
      vy = (fy + P.noise * zt1) / P.gamma;
    } else {
      vx = fx / P.gamma;
      vy = fy / P.gamma;
    }
  }
  if constexpr ((MODE & MODE_KICK) != 0) {
    vx += A.h * fx;
    vy += A.h * fy;
  }
  if constexpr ((MODE & MODE_START) != 0) {
    double xn, yn;
    if constexpr ((MODE & MODE_BROWN) != 0) {
      xn = x + vx * A.dt;
      yn = y + vy * A.dt;
    } else if constexpr ((MODE & MODE_BAOAB) != 0) {
      // B, A (half), O, A (half)
      vx += A.h * fx;
      vy += A.h * fy;
      const double xa = x + vx * A.h, ya = y + vy * A.h;
      vx = P.gamma * vx + P.noise * zt0;
      vy = P.gamma * vy + P.noise * zt1;
      xn = xa + vx * A.h;
      yn = ya + vy * A.h;
    } else {
      vx += A.h * fx;
      vy += A.h * fy;
      xn = x + A.dt * vx;
      yn = y + A.dt * vy;
    }
    A.xout[L.v] = xn;
    A.yout[L.v] = yn;
    if (A.recx) {
      A.recx[L.v] = xn;
      A.recy[L.v] = yn;
    }
    if (moved_past(P, B, xn - lx, yn - ly)) {
      atomicOr(&A.flagOut[L.s], 1);
      atomicOr(A.anyOut, 1);
    }
    far_test(P, B, xn - x, yn - y, A.flagOut + L.s);
  }
  V.vx[L.v] = vx;
  V.vy[L.v] = vy;
}

// LDS of the step kernel: six partials per lane of each gather wave (eight with wide rings)
// (or the results of the near list's evaluations), and in the same region the rows under construction
template <int INTER, int MODE>
static inline size_t step_lds(const dpm_set_s* S, int nw) {
  constexpr bool STORE = step_store<MODE>();
  const size_t red = (MODE & MODE_NEAR) ? (size_t)near_slots_bytes<INTER, STORE>()
                                        : (size_t)(nw - 1) * (S->nwide > 0 ? 8 : 6) * WAVE * sizeof(double);
  const size_t rows = S->V.W <= 64 ? (size_t)rows_lds_ints(S->V.W, (MODE & MODE_NEAR) != 0) * sizeof(int) : 0;
  return red > rows ? red : rows;
}

template <int INTER, int POT, int MODE>
static hipError_t step_one(dpm_set_s* S, const StepArgs& A) {
  const int nw = step_ref<MODE>() && !(MODE & MODE_NEAR) ? S->split : loop_waves(S);
  k_step<INTER, POT, MODE>
      <<<S->V.ntiles, WAVE * nw, step_lds<INTER, MODE>(S, nw), S->stream>>>(S->V, S->P, A, S->G);
  return hipGetLastError();
}

// rigid-ring modes (sets of rings of at most 64 vertices only)
template <int INTER, int POT>
static hipError_t step_rigid(dpm_set_s* S, int mode, const StepArgs& A) {
  switch (mode) {
    case MODE_RIGID: return step_one<INTER, POT, MODE_RIGID>(S, A);
    case MODE_RIGID | MODE_KICK: return step_one<INTER, POT, MODE_RIGID | MODE_KICK>(S, A);
    case MODE_RIGID | MODE_KICK | MODE_START: return step_one<INTER, POT, MODE_RIGID | MODE_KICK | MODE_START>(S, A);
    case MODE_RIGID | MODE_FIRE: return step_one<INTER, POT, MODE_RIGID | MODE_FIRE>(S, A);
    case MODE_RIGID | MODE_KICK | MODE_NEAR: return step_one<INTER, POT, MODE_RIGID | MODE_KICK | MODE_NEAR>(S, A);
    case MODE_RIGID | MODE_KICK | MODE_START | MODE_NEAR:
      return step_one<INTER, POT, MODE_RIGID | MODE_KICK | MODE_START | MODE_NEAR>(S, A);
    case MODE_RIGID | MODE_FIRE | MODE_NEAR: return step_one<INTER, POT, MODE_RIGID | MODE_FIRE | MODE_NEAR>(S, A);
  }
  return hipErrorInvalidValue;
}

// the loop modes, on whole rows (XB: 0 or MODE_WIDE) or on the near lists (XB: MODE_NEAR)
template <int INTER, int POT, int XB>
static hipError_t step_loop_mode(dpm_set_s* S, int mode, const StepArgs& A) {
  switch (mode) {
    case MODE_KICK: return step_one<INTER, POT, MODE_KICK | XB>(S, A);
    case MODE_KICK | MODE_LANGEVIN: return step_one<INTER, POT, MODE_KICK | MODE_LANGEVIN | XB>(S, A);
    case MODE_KICK | MODE_START: return step_one<INTER, POT, MODE_KICK | MODE_START | XB>(S, A);
    case MODE_KICK | MODE_LANGEVIN | MODE_START:
      return step_one<INTER, POT, MODE_KICK | MODE_LANGEVIN | MODE_START | XB>(S, A);
    case MODE_KICK | MODE_BAOAB: return step_one<INTER, POT, MODE_KICK | MODE_BAOAB | XB>(S, A);
    case MODE_KICK | MODE_BAOAB | MODE_START:
      return step_one<INTER, POT, MODE_KICK | MODE_BAOAB | MODE_START | XB>(S, A);
    case MODE_BROWN | MODE_START: return step_one<INTER, POT, MODE_BROWN | MODE_START | XB>(S, A);
    case MODE_BROWN | MODE_LANGEVIN | MODE_START:
      return step_one<INTER, POT, MODE_BROWN | MODE_LANGEVIN | MODE_START | XB>(S, A);
  }
  if constexpr (XB == MODE_NEAR) {
    switch (mode) {
      case MODE_BROWN | MODE_START | MODE_OUT: return step_one<INTER, POT, MODE_BROWN | MODE_START | MODE_OUT | XB>(S, A);
      case MODE_BROWN | MODE_LANGEVIN | MODE_START | MODE_OUT:
        return step_one<INTER, POT, MODE_BROWN | MODE_LANGEVIN | MODE_START | MODE_OUT | XB>(S, A);
    }
  }
  return hipErrorInvalidValue;
}

template <int INTER, int POT>
static hipError_t step_mode(dpm_set_s* S, int mode, const StepArgs& A) {
  if (S->nwide > 0) {
    if (mode & (MODE_RIGID | MODE_NEAR)) return hipErrorInvalidValue;  // refused for wide sets before this point
    switch (mode) {
      case MODE_FORCE: return step_one<INTER, POT, MODE_FORCE | MODE_WIDE>(S, A);
      case MODE_FIRE: return step_one<INTER, POT, MODE_FIRE | MODE_WIDE>(S, A);
    }
    return step_loop_mode<INTER, POT, MODE_WIDE>(S, mode, A);
  }
  if (mode & MODE_RIGID) return step_rigid<INTER, POT>(S, mode, A);
  if (mode == (MODE_FIRE | MODE_NEAR)) return step_one<INTER, POT, MODE_FIRE | MODE_NEAR>(S, A);
  if (mode == (MODE_FIRE | MODE_NEAR | MODE_OUT)) return step_one<INTER, POT, MODE_FIRE | MODE_NEAR | MODE_OUT>(S, A);
  if (mode & MODE_NEAR) return step_loop_mode<INTER, POT, MODE_NEAR>(S, mode & ~MODE_NEAR, A);
  switch (mode) {
    case MODE_FORCE: return step_one<INTER, POT, MODE_FORCE>(S, A);
    case MODE_FIRE: return step_one<INTER, POT, MODE_FIRE>(S, A);
  }
  return step_loop_mode<INTER, POT, 0>(S, mode, A);
}

// all-pairs interaction (test mode): forces only
template <int POT, int WB>
static hipError_t step_all(dpm_set_s* S, int mode, const StepArgs& A) {
  if (mode != MODE_FORCE) return hipErrorInvalidValue;
  return step_one<INT_ALL, POT, MODE_FORCE | WB>(S, A);
}

#if !defined(STEP_INTER) || !defined(STEP_POT)
#error "compile with -DSTEP_INTER and -DSTEP_POT"
#endif
template <>
hipError_t step_launch<STEP_INTER, STEP_POT>(dpm_set_s* S, int mode, const StepArgs& A) {
#if STEP_INTER == 3
  return S->nwide > 0 ? step_all<STEP_POT, MODE_WIDE>(S, mode, A) : step_all<STEP_POT, 0>(S, mode, A);
#else
  return step_mode<STEP_INTER, STEP_POT>(S, mode, A);
#endif
}

}  // namespace dpm
