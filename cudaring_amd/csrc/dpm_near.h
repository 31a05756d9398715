// dpm_near.h -- the part of a tile's neighbour rows that can come into range before the next
// rebuild, as one flat list of pair evaluations per tile.
//
// A row holds the neighbours within (1 + cutDistance) radius sums, far beyond the potential's
// range.  Inside a loop no vertex is farther than cutoff / 3 from its list position when a force
// is evaluated (the displacement test rebuilds first), so a pair (or a vertex and a segment) whose
// distance at the list positions exceeds range + 2 cutoff / 3 cannot interact before the next
// rebuild: leaving it out changes no force.  The evaluations that remain lie one after another
// per tile, by vertex and then by neighbour, so that every lane of the gather holds one (a row per
// lane would wait for the tile's longest row: 18 entries where the mean is 4.4), and a lane finds
// its task at an address that depends on nothing but the tile.
#pragma once

#include "dpm_forces.h"

namespace dpm {

// widest range of the potential in radius sums
__device__ __forceinline__ double near_range(const Params& P) {
  switch (P.potential) {
    case POT_HARMONIC: return 1.0;
    case POT_LJ: return P.LJcutoff;
    case POT_ADHESIVE: return 1.0 + fmax(P.l1, P.l2);
    default: return kWCAcut;
  }
}

// whether i lies within r (r2 = r r) of the segment (p, j), divisions multiplied out; a segment too
// long for its minimum image to be the one the force takes counts as near
__device__ __forceinline__ bool seg_near(const Box& B, double xi, double yi, double xj, double yj, double xp,
                                         double yp, double r2) {
  const double sx = pbx(xj - xp, B), sy = pby(yj - yp, B);
  const double ix = pbx(xi - xp, B), iy = pby(yi - yp, B);
  const double l2 = sx * sx + sy * sy, lim = 0.25 * fmin(B.Lx, B.Ly);
  const double dot = ix * sx + iy * sy, i2 = ix * ix + iy * iy;
  const double jx = ix - sx, jy = iy - sy;
  const bool in = dot <= 0 ? i2 <= r2 : (dot >= l2 ? jx * jx + jy * jy <= r2 : i2 * l2 - dot * dot <= r2 * l2);
  return in || l2 > lim * lim;
}

// kernelCalcNeighborList's predicate -(1 - d / sum) < cutDistance (cudaKernel.cuh:1735-1763) from the
// squared distance: the division and the root only where the comparison of squares cannot tell
__device__ __forceinline__ bool in_list(const Params& P, double d2, double sum) {
  const double r = (1 + P.cutDistance) * sum, r2 = r * r;
  if (fabs(d2 - r2) > 1e-12 * r2 && r > 0) return d2 < r2;
  return -(1 - sqrt(d2) / sum) < P.cutDistance;
}

// reach of the near test for a radius sum: the widest range, the 2 cutoff / 3 by which two vertices
// can approach before the next rebuild, and a slack far above the rounding of the distances
struct NearReach {
  double R, d2;
  __device__ explicit NearReach(const Params& P) : R(near_range(P) + 1e-6), d2(2 * fmax(P.cutoff, 0.0) / 3) {}
  __device__ __forceinline__ double sq(double sum) const {
    const double r = R * sum + d2;
    return r * r;
  }
};

// LDS of the near masks in bytes: one bit per row entry, role and lane
constexpr int kNearMaskBytes = 2 * WAVE * 8;
// LDS ints of build_rows_tile
__host__ __device__ constexpr int rows_lds_ints(int W, bool near) {
  return near ? kNearMaskBytes / 4 + WAVE + 2 * WAVE * W : WAVE + WAVE * W;
}

// The task list of a tile: `bits(q)` the lane's mask of near row entries of role q (complete),
// `entry(k)` its k-th neighbour in ascending order, of n.
template <int INTER, class M, class F>
__device__ __forceinline__ void write_near_tile(const View& V, const NearRows& N, const Lane& L, int w, int nw, int n,
                                                M bits, F entry) {
  constexpr int NR = INTER == INT_SMOOTH ? 2 : 1;
  int total[2] = {0, 0};
#pragma unroll
  for (int q = 0; q < NR; q++) {
    const unsigned long long m = bits(q);
    const int c = __popcll(m);
    int end = c;  // inclusive scan over the lanes: vertices in order
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
      const int t = __shfl_up(end, d, WAVE);
      if (L.lane >= d) end += t;
    }
    const int start = end - c;
    total[q] = __shfl(end, WAVE - 1, WAVE);
    if (w == 0 && L.act) N.span[(long)q * V.nv + L.v] = start | (c << 16);
    int2* list = N.task + ((long)L.tile * 2 + q) * N.cap;
    for (int k = w; k < n; k += nw)
      if ((m >> k) & 1) {
        const int u = entry(k);
        int meta = L.lane;
        if constexpr (NR == 2) {
          int o1, o2;  // offsets within a ring of at most 64 vertices
          if (q == 0) {
            const int2 pp = prev_pair(V, u);
            o1 = u - pp.x;
            o2 = u - pp.y;
          } else {
            o1 = L.lane - L.pl;
            o2 = L.lane - ((L.pl > L.segS) ? L.pl - 1 : L.segE);
          }
          meta |= (o1 + 64) << 8 | (o2 + 64) << 16;
        }
        list[start + __popcll(m & ((1ull << k) - 1))] = make_int2(u, meta);
      }
  }
  if (w == 0 && L.lane == 0) N.tcnt[L.tile] = make_int2(total[0], total[1]);
}

// Near bits (role 0, role 1) of the lane's vertex at (x, y), whose ring's previous vertex is at
// (xp, yp), and its neighbour u; positions px, py.
template <int INTER>
__device__ __forceinline__ int near_bits(const View& V, const NearReach& R, const Box& B, double x, double y,
                                         double radv, double xp, double yp, int u, const double* px, const double* py) {
  const double xu = px[u], yu = py[u], r2 = R.sq(radv + V.rad[u]);
  if constexpr (INTER == INT_SMOOTH) {
    const int p = prev_pair(V, u).x;
    return (seg_near(B, x, y, xu, yu, px[p], py[p], r2) ? 1 : 0) | (seg_near(B, xu, yu, x, y, xp, yp, r2) ? 2 : 0);
  }
  const double dx = pbx(x - xu, B), dy = pby(y - yu, B);
  return dx * dx + dy * dy <= r2 ? 1 : 0;
}

// The task list of a tile from its rows in memory (complete and visible to the workgroup) and the
// list positions px, py; keepAll: every entry (systems narrower than three cells, where an entry may
// be near through another image).  Roles: 0, the pair (v, j) or the share of v from the segment
// (prev(u), u); 1 (vertex-segment only), the shares of v and prev(v) from u against the segment
// (prev(v), v).  An entry is (neighbour, lane of v | offsets of the segment's prev and second prev), a
// vertex's span its first entry and their number.  Every thread of the workgroup calls it, rows of
// at most 64 entries, kNearMaskBytes of LDS; the caller synchronises before the list is read or lds
// reused.
template <int INTER>
__device__ __forceinline__ void build_near_tile(const View& V, const Params& P, const NearRows& N, const Lane& L,
                                                int w, int nw, const Box& B, const double* px, const double* py,
                                                bool keepAll, void* lds) {
  unsigned long long* mask = (unsigned long long*)lds;
  if (w == 0) mask[L.lane] = mask[WAVE + L.lane] = 0;
  __syncthreads();
  const int n = L.act ? V.ncnt[L.v] : 0;
  const double x = px[L.v], y = py[L.v], radv = V.rad[L.v];
  const NearReach R(P);
  const int vp = L.act ? L.v0 + L.pl : L.v;
  const double xp = px[vp], yp = py[vp];
  for (int k = w; k < n; k += nw) {
    const int bits =
        keepAll ? 3 : near_bits<INTER>(V, R, B, x, y, radv, xp, yp, V.nbr[(long)k * V.nv + L.v], px, py);
    if (bits & 1) atomicOr(&mask[L.lane], 1ull << k);
    if (bits & 2) atomicOr(&mask[WAVE + L.lane], 1ull << k);
  }
  __syncthreads();
  write_near_tile<INTER>(V, N, L, w, nw, n, [&](int q) { return mask[q * WAVE + L.lane]; }, [&](int k) { return V.nbr[(long)k * V.nv + L.v]; });
}

// build_near_tile by one wave for its tile, each lane over its own row, the masks in registers.
template <int INTER>
__device__ __forceinline__ void build_near_wave(const View& V, const Params& P, const NearRows& N, const Lane& L,
                                                const Box& B, const double* px, const double* py, bool keepAll) {
  const int n = L.act ? V.ncnt[L.v] : 0;
  const double x = px[L.v], y = py[L.v], radv = V.rad[L.v];
  const NearReach R(P);
  const int vp = L.act ? L.v0 + L.pl : L.v;
  const double xp = px[vp], yp = py[vp];
  unsigned long long mask[2] = {0, 0};
  for (int k = 0; k < n; k++) {
    const int bits =
        keepAll ? 3 : near_bits<INTER>(V, R, B, x, y, radv, xp, yp, V.nbr[(long)k * V.nv + L.v], px, py);
    mask[0] |= (unsigned long long)(bits & 1) << k;
    mask[1] |= (unsigned long long)(bits >> 1) << k;
  }
  write_near_tile<INTER>(V, N, L, 0, 1, n, [&](int q) { return mask[q]; },
                         [&](int k) { return V.nbr[(long)k * V.nv + L.v]; });
}

// The rows of a tile's vertices (lane = vertex, L.act lanes), built by all nw waves of its
// workgroup: thread (w, lane) scans the cells w, w + nw, ... of the 3 x 3 block around its lane's
// vertex and appends the hits to the lane's list in LDS (an LDS counter
// per lane, so the order of arrival varies); after a barrier the waves share the entries of each
// list, place every one by its rank (the number of smaller entries of the list) and write it with
// its prev pair into the ELL row.  The same rows as build_row from the same cells (its predicate,
// ascending order).  NEAR: the interaction whose near list is built from the same entries while
// they are at hand (positions V.x, V.y are the new list positions), or -1.  Every thread of the
// workgroup calls it (it holds barriers); lds holds rows_lds_ints(W, NEAR >= 0) ints; the caller
// synchronises before reading the rows or reusing lds.
//
// Bound by latency: a chain of dependent loads (cell count, slots, positions), shortened by fetching
// ahead and four candidates at a time, and the fetch of its own instructions, which a rebuild runs cold
// (eight candidates unrolled took longer than one after another).  A vertex of the own ring is told by
// its index.  maxcnt: longest row for the host, or null (inside loops: one word for every tile).
template <int NEAR>
__device__ __forceinline__ void build_rows_tile(const View& V, const Params& P, const CellGrid& G, const int* count,
                                                const int* slots, const Lane& L, int w, int nw, const Box& B, double x,
                                                double y, int* lds, int* err, int* maxcnt, const NearRows& N) {
  const int W = V.W, lane = L.lane, v = L.v, s = L.s;
  unsigned long long* mask = (unsigned long long*)lds;
  int* lcnt = NEAR >= 0 ? lds + kNearMaskBytes / 4 : lds;
  int* lrow = lcnt + WAVE;
  int* srow = lrow + WAVE * W;
  if (w == 0) {
    lcnt[lane] = 0;
    if constexpr (NEAR >= 0) mask[lane] = mask[WAVE + lane] = 0;
  }
  __syncthreads();
  const double rv = V.rad[v];
  if (L.act) {
    const int ncx = G.ncx[s], ncy = G.ncy[s], c0 = G.coff[s];
    int cx, cy;
    cell_of(x, y, B, ncx, ncy, cx, cy);
    auto cell = [&](int k) {
      int yy = cy + k / 3 - 1, xx = cx + k % 3 - 1;
      yy += yy < 0 ? ncy : (yy >= ncy ? -ncy : 0);
      xx += xx < 0 ? ncx : (xx >= ncx ? -ncx : 0);
      return c0 + yy * ncx + xx;
    };
    // a cell's count and first four slots are fetched while the cell before it is searched (slots past
    // the count hold older vertices: in bounds, and not tested)
    int cl = cell(w);
    int m = count[cl];
    int4 sj = *(const int4*)(slots + (long)cl * G.cap);
#pragma unroll 1
    for (int k = w; k < 9; k += nw) {
      const int cn = cell(k + nw < 9 ? k + nw : k);
      const int mn = count[cn];
      const int4 sn = *(const int4*)(slots + (long)cn * G.cap);
      const int* sl = slots + (long)cl * G.cap;
      m = min(m, G.cap);
#pragma unroll 1
      for (int q = 0; q < m; q += 4) {
        const int j[4] = {sj.x, sj.y, sj.z, sj.w};
        double xj[4], yj[4], rj[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int u = q + i < m ? j[i] : v;
          xj[i] = V.x[u];
          yj[i] = V.y[u];
          rj[i] = V.rad[u];
        }
        if (q + 4 < m) sj = *(const int4*)(sl + q + 4);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const double dx = pbx(x - xj[i], B), dy = pby(y - yj[i], B);
          if (q + i < m && (unsigned)(j[i] - L.f) >= (unsigned)L.n && in_list(P, dx * dx + dy * dy, rv + rj[i])) {
            const int idx = atomicAdd(&lcnt[lane], 1);
            if (idx < W) lrow[idx * WAVE + lane] = j[i];
          }
        }
      }
      cl = cn;
      m = mn;
      sj = sn;
    }
  }
  double xp = 0, yp = 0;
  if constexpr (NEAR == INT_SMOOTH) {
    const int vp = L.act ? L.v0 + L.pl : v;
    xp = V.x[vp];
    yp = V.y[vp];
  }
  __syncthreads();
  const int c = L.act ? lcnt[lane] : 0;
  const int n = c < W ? c : W;
  if (w == 0 && L.act) {
    if (c > W) atomicOr(err, ERR_LIST_OVERFLOW);
    if (maxcnt) atomicMax(maxcnt, c);
    V.ncnt[v] = n;
    V.lx[v] = x;
    V.ly[v] = y;
  }
  const NearReach R(P);
  for (int k = w; k < n; k += nw) {
    const int j = lrow[k * WAVE + lane];
    int rank = 0;
    for (int q = 0; q < n; q++) rank += lrow[q * WAVE + lane] < j ? 1 : 0;
    V.nbr[(long)rank * V.nv + v] = j;
    V.nbrp[(long)rank * V.nv + v] = prev_pair(V, j);
    if constexpr (NEAR >= 0) {
      srow[rank * WAVE + lane] = j;
      const int bits = near_bits<NEAR>(V, R, B, x, y, rv, xp, yp, j, V.x, V.y);
      if (bits & 1) atomicOr(&mask[lane], 1ull << rank);
      if (bits & 2) atomicOr(&mask[WAVE + lane], 1ull << rank);
    }
  }
  if constexpr (NEAR >= 0) {
    __syncthreads();
    write_near_tile<NEAR>(V, N, L, w, nw, n, [&](int q) { return mask[q * WAVE + lane]; }, [&](int k) { return srow[k * WAVE + lane]; });
  }
}

// LDS results of a window of NEAR_WIN evaluations per role: forces on v of role 0, forces on v and
// on prev(v) of role 1, energies when the step stores them
#define NEAR_WIN 384
template <int INTER, bool ENERGY>
constexpr int near_slots_bytes() {
  return NEAR_WIN * ((INTER == INT_SMOOTH ? 48 : 16) + (ENERGY ? (INTER == INT_SMOOTH ? 16 : 8) : 0));
}

// Evaluations [base, base + NEAR_WIN) of both roles of a tile, dealt in chunks of 64 to the gather
// waves w of nw (roles alternate, so that the first chunks of both start at once).
template <int INTER, int POT, bool REF, bool ENERGY>
__device__ __forceinline__ void eval_near(const View& V, const Params& P, const NearRows& N, const Box& B, int tile,
                                          int v0, int2 cnt, int base, int lane, int w, int nw, void* lds) {
  constexpr int NR = INTER == INT_SMOOTH ? 2 : 1;
  double2* fT = (double2*)lds;
  double2* fO = fT + NEAR_WIN;
  double2* qO = fO + NEAR_WIN;
  double* eT = (double*)(fT + (NR == 2 ? 3 : 1) * NEAR_WIN);
  double* eO = eT + NEAR_WIN;
  const int nT = min(cnt.x - base, NEAR_WIN), nO = NR == 2 ? min(cnt.y - base, NEAR_WIN) : 0;
  const int2* list = N.task + (long)tile * 2 * N.cap;
  const int chunks = NR * ((max(nT, nO) + WAVE - 1) / WAVE);
  for (int c = w; c < chunks; c += nw) {
    const int i = (NR == 2 ? c >> 1 : c) * WAVE + lane;
    if (NR == 1 || (c & 1) == 0) {
      if (i < nT) {
        const int2 t = list[base + i];
        const int v = v0 + (t.y & 63), u = t.x;
        const double x = V.x[v], y = V.y[v], xu = V.x[u], yu = V.y[u];
        const double sum = V.rad[v] + V.rad[u];
        double fx = 0, fy = 0, e;
        if constexpr (NR == 1) {
          e = pair_of<POT, REF>(P, pbx(x - xu, B), pby(y - yu, B), sum, fx, fy);
        } else {
          const int p1 = u - (((t.y >> 8) & 255) - 64), p2 = u - (((t.y >> 16) & 255) - 64);
          e = smooth_this_of<POT, REF>(P, B, x, y, xu, yu, V.x[p1], V.y[p1], V.x[p2], V.y[p2], sum, fx, fy);
        }
        fT[i] = make_double2(fx, fy);
        if constexpr (ENERGY) eT[i] = e;
      }
    } else {
      if (i < nO) {
        const int2 t = list[N.cap + base + i];
        const int v = v0 + (t.y & 63), u = t.x;
        const int p1 = v - (((t.y >> 8) & 255) - 64), p2 = v - (((t.y >> 16) & 255) - 64);
        double fx = 0, fy = 0, qx = 0, qy = 0;
        const double e = smooth_op_of<POT, REF>(P, B, V.x[u], V.y[u], V.x[v], V.y[v], V.x[p1], V.y[p1], V.x[p2], V.y[p2],
                                             V.rad[v] + V.rad[u], fx, fy, qx, qy);
        fO[i] = make_double2(fx, fy);
        qO[i] = make_double2(qx, qy);
        if constexpr (ENERGY) eO[i] = e;
      }
    }
  }
}

// A lane's sums over its vertex's results of the window, in list order: the same values whatever
// the number of waves.
template <int INTER, bool ENERGY>
__device__ __forceinline__ void sum_near(int spanT, int spanO, int base, const void* lds, double& fx, double& fy,
                                         double& e, double& qx, double& qy) {
  constexpr int NR = INTER == INT_SMOOTH ? 2 : 1;
  const double2* fT = (const double2*)lds;
  const double2* fO = fT + NEAR_WIN;
  const double2* qO = fO + NEAR_WIN;
  const double* eT = (const double*)(fT + (NR == 2 ? 3 : 1) * NEAR_WIN);
  const double* eO = eT + NEAR_WIN;
  {
    const int s = (spanT & 0xffff) - base, a = max(s, 0), b = min(s + (spanT >> 16), NEAR_WIN);
    for (int k = a; k < b; k++) {
      const double2 f = fT[k];
      fx += f.x;
      fy += f.y;
      if constexpr (ENERGY) e += eT[k];
    }
  }
  if constexpr (NR == 2) {
    const int s = (spanO & 0xffff) - base, a = max(s, 0), b = min(s + (spanO >> 16), NEAR_WIN);
    for (int k = a; k < b; k++) {
      const double2 f = fO[k], q = qO[k];
      fx += f.x;
      fy += f.y;
      qx += q.x;
      qy += q.y;
      if constexpr (ENERGY) e += eO[k];
    }
  }
}

// One wave's evaluation of its tile's near list, 64 at a time, positions through pos(v) (a double2), the
// chunk's results handed to their lanes through `res` (near_wave_doubles of LDS, the wave's own).
template <int INTER>
__host__ __device__ constexpr int near_wave_doubles() {
  return WAVE * (INTER == INT_SMOOTH ? 5 : 3);
}
template <int INTER, int POT, bool REF, bool ENERGY, class X>
__device__ __forceinline__ void near_wave(const View& V, const Params& P, const NearRows& N, const Box& B,
                                          const Lane& L, X pos, double* res, double& fx, double& fy, double& e,
                                          double& qx, double& qy) {
  constexpr int NR = INTER == INT_SMOOTH ? 2 : 1;
  double2* f = (double2*)res;
  double2* g = f + WAVE;
  double* en = (double*)(f + NR * WAVE);
  const int2 cnt = N.tcnt[L.tile];
#pragma unroll
  for (int q = 0; q < NR; q++) {
    const int total = q ? cnt.y : cnt.x, span = L.act ? N.span[(long)q * V.nv + L.v] : 0;
    const int2* list = N.task + ((long)L.tile * 2 + q) * N.cap;
    for (int base = 0; base < total; base += WAVE) {
      if (base + L.lane < total) {
        const int2 t = list[base + L.lane];
        const int v = L.v0 + (t.y & 63), u = t.x;
        const double2 a = pos(v), b = pos(u);
        const double sum = V.rad[v] + V.rad[u];
        double ax = 0, ay = 0, bx = 0, by = 0, ee;
        if constexpr (NR == 1) {
          ee = pair_of<POT, REF>(P, pbx(a.x - b.x, B), pby(a.y - b.y, B), sum, ax, ay);
        } else {
          const int j = q ? v : u;
          const double2 p1 = pos(j - (((t.y >> 8) & 255) - 64)), p2 = pos(j - (((t.y >> 16) & 255) - 64));
          if (q == 0)
            ee = smooth_this_of<POT, REF>(P, B, a.x, a.y, b.x, b.y, p1.x, p1.y, p2.x, p2.y, sum, ax, ay);
          else
            ee = smooth_op_of<POT, REF>(P, B, b.x, b.y, a.x, a.y, p1.x, p1.y, p2.x, p2.y, sum, ax, ay, bx, by);
        }
        f[L.lane] = make_double2(ax, ay);
        if (q == 1) g[L.lane] = make_double2(bx, by);
        if constexpr (ENERGY) en[L.lane] = ee;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const int s = (span & 0xffff) - base, k0 = max(s, 0), k1 = min(s + (span >> 16), WAVE);
      for (int k = k0; k < k1; k++) {
        const double2 a = f[k];
        fx += a.x;
        fy += a.y;
        if (q == 1) {
          const double2 b = g[k];
          qx += b.x;
          qy += b.y;
        }
        if constexpr (ENERGY) e += en[k];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
}

}  // namespace dpm
