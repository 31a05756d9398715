// dpm_forces.h -- device functions of the step and FIRE kernels: ring geometry and shape forces,
// the interparticle gather, the step loop's cell lists and the rigid-ring moves.
#pragma once

#include "dpm_internal.h"
#include "dpm_rows.h"
#include "dpm_tile.h"

namespace dpm {

// wave-per-tile kernels (4 tiles per 256-thread block)
__device__ __forceinline__ bool wave_tile_ctx(const View& V, Lane& L) {
  const int tile = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  if (tile >= V.ntiles) return false;
  lane_ctx(V, tile, threadIdx.x & (WAVE - 1), L);
  return true;
}

// Ring geometry + shape force for one lane (wave-uniform call).  Restates
// kernelCalcParticleShape (cudaKernel.cuh:1571-1606), calcParticlePos (365-388)
// and kernelCalcShapeForceEnergy (474-529) with the area/perimeter/bending
// terms of 429-471.  Writes theta, length and the ring area/perimeter/centre.
struct ShapeOut {
  double fx, fy, e;
  double cx, cy;  // ring centre (calcParticlePos, cudaKernel.cuh:365-388)
};

// turning angle at a vertex from its own, next and previous positions (calcAngle 423-427)
__device__ __forceinline__ double vertex_theta(const Box& B, double x, double y, double xn, double yn, double xp,
                                               double yp) {
  const double dnx = pbx(xn - x, B), dny = pby(yn - y, B);
  const double psx = -pbx(xp - x, B), psy = -pby(yp - y, B);
  return atan2(dnx * psy - dny * psx, dnx * psx + dny * psy);
}

__device__ __forceinline__ ShapeOut ring_shape(const View& V, const Params& P, const Lane& L, const Box& B,
                                               double x, double y, bool write) {
  ShapeOut o;
  double xn, yn, xp, yp, theta, seglen, area, perim, comx, comy;
  int vn = 0, vp = 0;
  if (!L.wide) {
    xn = shfl_d(x, L.nl); yn = shfl_d(y, L.nl);
    xp = shfl_d(x, L.pl); yp = shfl_d(y, L.pl);
    const double xf = shfl_d(x, L.segS), yf = shfl_d(y, L.segS);
    // segments of the reference's unwrapped walk
    const double dnx = pbx(xn - x, B), dny = pby(yn - y, B);
    const double psx = -pbx(xp - x, B), psy = -pby(yp - y, B);
    theta = atan2(dnx * psy - dny * psx, dnx * psx + dny * psy);  // calcAngle 423-427
    seglen = root(dnx * dnx + dny * dny);
    // Unwrapped position relative to the first vertex: the reference walks the ring one
    // minimum-image segment at a time; here that walk is an exclusive segmented scan of the
    // segment vectors, valid for rings wider than half the box.
    const double Ix = seg_scan(L.act ? dnx : 0.0, L.lane, L.segS);
    const double Iy = seg_scan(L.act ? dny : 0.0, L.lane, L.segS);
    const double ux = L.act ? Ix - dnx : 0.0;
    const double uy = L.act ? Iy - dny : 0.0;
    const double shoe = L.act ? (ux * dny - dnx * uy) : 0.0;  // shoelace: cur x next = cur x delta
    perim = seg_sum(L.act ? seglen : 0.0, L.lane, L.segS, L.segE);
    const double shoeSum = seg_sum(shoe, L.lane, L.segS, L.segE);
    const double sux = seg_sum(ux, L.lane, L.segS, L.segE);
    const double suy = seg_sum(uy, L.lane, L.segS, L.segE);
    const double ind = quot(1.0, (double)L.n);
    area = fabs(shoeSum) * 0.5;
    comx = xf + sux * ind;
    comy = yf + suy * ind;
  } else {
    // a slice of a wide ring: ring neighbours from memory (this launch reads the current positions
    // only), the ring's area, perimeter and centre from k_wide_rings, launched just before
    vn = ring_next(L.v, L.f, L.n);
    vp = ring_prev(L.v, L.f, L.n);
    xn = V.x[vn]; yn = V.y[vn];
    xp = V.x[vp]; yp = V.y[vp];
    theta = vertex_theta(B, x, y, xn, yn, xp, yp);
    const double dnx = pbx(xn - x, B), dny = pby(yn - y, B);
    seglen = root(dnx * dnx + dny * dny);
    area = V.area[L.r];
    perim = V.perim[L.r];
    comx = V.cx[L.r];
    comy = V.cy[L.r];
  }
  o.cx = comx;
  o.cy = comy;
  if (write && L.act) {
    V.th[L.v] = theta;
    V.len[L.v] = seglen;
    if (L.lane == L.segS && !L.wide) {
      V.area[L.r] = area;
      V.perim[L.r] = perim;
      V.cx[L.r] = comx;
      V.cy[L.r] = comy;
    }
  }
  const double ind = quot(1.0, (double)L.n);
  // positions relative to the ring centre (getRelativeVertexPos 273-279)
  const double rvx = pbx(x - comx, B), rvy = pby(y - comy, B);
  const double rnx = pbx(xn - comx, B), rny = pby(yn - comy, B);
  const double rpx = pbx(xp - comx, B), rpy = pby(yp - comy, B);
  const double a0 = V.a0[L.r];
  // shape costs: the global ea, el, eb, or per-ring values when the caller set them
  const double ea = V.kr ? V.kr[L.r] : P.ea;
  const double el = V.kr ? V.kr[V.np + L.r] : P.el;
  const double eb = V.kr ? V.kr[2 * V.np + L.r] : P.eb;
  // area term (calcAreaForceEnergy 429-435)
  const double deltaA = quot(area, a0) - 1.;
  const double gmA = quot(ea * deltaA, a0);
  double fx = 0.5 * gmA * (rpy - rny);
  double fy = 0.5 * gmA * (rnx - rpx);
  double e = (0.5 * ea * deltaA * deltaA) * ind;
  // perimeter term (calcPerimeterForceEnergy 437-447 / FENE 449-455)
  const double nsx = rnx - rvx, nsy = rny - rvy;
  const double qsx = rvx - rpx, qsy = rvy - rpy;
  const double pLen = root(qsx * qsx + qsy * qsy);
  const double nLen = root(nsx * nsx + nsy * nsy);
  const double l0v = V.l0[L.v];
  const double l0s = shfl_d(l0v, L.pl);
  const double l0p = L.wide ? V.l0[vp] : l0s;
  if (P.monomer == MONO_HARMONIC) {
    const double pDelta = quot(pLen, l0p) - 1.;
    const double nDelta = quot(nLen, l0v) - 1.;
    const double cn = quot(nDelta, l0v * nLen), cp = quot(pDelta, l0p * pLen);
    fx += el * ((cn * (rnx - rvx)) - (cp * (rvx - rpx)));
    fy += el * ((cn * (rny - rvy)) - (cp * (rvy - rpy)));
    e += (0.5 * el * pDelta * pDelta);
  } else {
    const double c = 2 * el * P.stiff * P.extSq;
    fx += c * ((nLen / (P.extSq * l0v * l0v - nLen * nLen)) * (rnx - rvx) / nLen -
               (pLen / (P.extSq * l0p * l0p - pLen * pLen)) * (rvx - rpx) / pLen);
    fy += c * ((nLen / (P.extSq * l0v * l0v - nLen * nLen)) * (rny - rvy) / nLen -
               (pLen / (P.extSq * l0p * l0p - pLen * pLen)) * (rvy - rpy) / pLen);
    e += el * P.stiff * P.extSq * log(1 - pLen * pLen / (P.extSq * l0p * l0p));
  }
  // bending term (calcBendingForceEnergy 457-471)
  const double D = theta - V.th0[L.v];
  double Dp = shfl_d(D, L.pl), Dn = shfl_d(D, L.nl);
  if (L.wide) {  // the neighbours' angles from their own neighbours, as their lanes form them
    const int vpp = ring_prev(vp, L.f, L.n), vnn = ring_next(vn, L.f, L.n);
    Dp = vertex_theta(B, xp, yp, x, y, V.x[vpp], V.y[vpp]) - V.th0[vp];
    Dn = vertex_theta(B, xn, yn, V.x[vnn], V.y[vnn], x, y) - V.th0[vn];
  }
  const double preVar = quot(D - Dp, qsx * qsx + qsy * qsy);
  const double nextVar = quot(D - Dn, nsx * nsx + nsy * nsy);
  fx += eb * (preVar * qsy + nextVar * nsy);
  fy += eb * (preVar * (-qsx) + nextVar * (-nsx));
  e += (0.5 * eb * D * D);
  o.fx = fx; o.fy = fy; o.e = e;
  return o;
}

// Position (ux, uy) of the lane's vertex relative to its ring's first vertex along the reference's
// walk, one minimum-image segment (dnx, dny) at a time.  The walk of a ring narrower than half the box
// is the minimum image of the difference itself: taken when every segment of the wave's rings joins up
// with it, else the walk is an exclusive segmented scan of the segments (six dependent levels more).
__device__ __forceinline__ void ring_walk(const Lane& L, const Box& B, double x, double y, double xf, double yf,
                                          double dnx, double dny, double& ux, double& uy) {
  ux = L.act ? pbx(x - xf, B) : 0.0;
  uy = L.act ? pby(y - yf, B) : 0.0;
  const double gx = shfl_d(ux, L.nl) - ux - dnx, gy = shfl_d(uy, L.nl) - uy - dny;
  if (__all(!L.act || (fabs(gx) < 0.25 * B.Lx && fabs(gy) < 0.25 * B.Ly))) return;
  ux = L.act ? seg_scan(L.act ? dnx : 0.0, L.lane, L.segS) - dnx : 0.0;
  uy = L.act ? seg_scan(L.act ? dny : 0.0, L.lane, L.segS) - dny : 0.0;
}

// seg_scan of a pair as a loop: the walk's rare path, small rather than fast (a step's time is the
// length of its instruction stream, also of what it jumps over)
__device__ __forceinline__ void seg_scan_pair(double& a, double& b, int lane, int segS) {
#pragma unroll 1
  for (int d = 1; d < WAVE; d <<= 1) {
    const double s = __shfl_up(a, d, WAVE), t = __shfl_up(b, d, WAVE);
    if (lane - d >= segS) {
      a += s;
      b += t;
    }
  }
}

// ring_walk for ring_shape_n.  True when a ring of the wave reaches past half the box from its centre
// (cx, cy), set only then: there the reference's centre-relative positions, a minimum image each
// (getRelativeVertexPos 273-279), differ by a box length more than the segments.  Rings within a quarter
// of the box of the middle between their first vertex and the opposite one, the usual case down to packings
// of ten rings, are told by that: their centre lies there too, and the walk is the minimum image itself.
__device__ __forceinline__ bool ring_walk_past_half(const Lane& L, const Box& B, double x, double y, double dnx,
                                                    double dny, double& ux, double& uy, double& cx, double& cy) {
  const double xf = shfl_d(x, L.segS), yf = shfl_d(y, L.segS);
  ux = L.act ? pbx(x - xf, B) : 0.0;
  uy = L.act ? pby(y - yf, B) : 0.0;
  const int opposite = (L.segS + (L.n >> 1)) & (WAVE - 1);
  const double hx = __builtin_fma(-0.5, shfl_d(ux, opposite), ux), hy = __builtin_fma(-0.5, shfl_d(uy, opposite), uy);
  if (__all(!L.act || (fabs(hx) < 0.25 * B.Lx && fabs(hy) < 0.25 * B.Ly))) return false;
  double ax = L.act ? dnx : 0.0, ay = L.act ? dny : 0.0;  // the walk, one segment at a time
  seg_scan_pair(ax, ay, L.lane, L.segS);
  ux = L.act ? ax - dnx : 0.0;
  uy = L.act ? ay - dny : 0.0;
  ax = ux;
  ay = uy;
  seg_scan_pair(ax, ay, L.lane, L.segS);
  const double ind = quot(1.0, (double)L.n), mx = shfl_d(ax, L.segE) * ind, my = shfl_d(ay, L.segE) * ind;
  cx = xf + mx;
  cy = yf + my;
  return __any(L.act && !(fabs((ux - mx) * B.mx) < 0.4999 && fabs((uy - my) * B.my) < 0.4999));
}

// ring_shape for the step loops.  With dn = (v, next) and ps = (prev, v): the centre-relative differences of the reference's terms
// (getRelativeVertexPos 273-279) are sums of the two, so the force needs no centre (rings reaching past
// half the box from theirs excepted); the previous
// segment's factors are the previous lane's own.  `write`: theta, length, energy, and the ring's area,
// perimeter and centre, which nothing inside a step needs.
__device__ __forceinline__ ShapeOut ring_shape_n(const View& V, const Params& P, const Lane& L, const Box& B,
                                                 double x, double y, bool write) {
#pragma clang fp contract(fast)
  ShapeOut o{0, 0, 0, 0, 0};
  double xn, yn, xp, yp, area, perim = 0;
  int vn = 0, vp = 0;
  if (!L.wide) {
    xn = shfl_d(x, L.nl); yn = shfl_d(y, L.nl);
    xp = shfl_d(x, L.pl); yp = shfl_d(y, L.pl);
  } else {
    // a slice of a wide ring: ring neighbours from memory (this launch reads the current positions
    // only), the ring's area, perimeter and centre from k_wide_rings, launched just before
    vn = ring_next(L.v, L.f, L.n);
    vp = ring_prev(L.v, L.f, L.n);
    xn = V.x[vn]; yn = V.y[vn];
    xp = V.x[vp]; yp = V.y[vp];
  }
  double dnx = pbx(xn - x, B), dny = pby(yn - y, B);
  double psx = -pbx(xp - x, B), psy = -pby(yp - y, B);
  const double theta = atan2(dnx * psy - dny * psx, dnx * psx + dny * psy);  // calcAngle 423-427
  double n2 = dnx * dnx + dny * dny, in = rsqrt_n(n2), seglen = n2 > 0 ? sqrt_from(n2, in) : n2;
  bool past;  // a ring of the wave reaches past half the box from its centre (cx, cy)
  double cx = 0, cy = 0;
  if (!L.wide) {
    double ux, uy;
    past = ring_walk_past_half(L, B, x, y, dnx, dny, ux, uy, cx, cy);
    const double shoe = L.act ? (ux * dny - dnx * uy) : 0.0;  // shoelace: cur x next = cur x delta
    area = fabs(seg_sum(shoe, L.lane, L.segS, L.segE)) * 0.5;
    if (write) {
      const double xf = shfl_d(x, L.segS), yf = shfl_d(y, L.segS);
      perim = seg_sum(L.act ? seglen : 0.0, L.lane, L.segS, L.segE);
      const double ind = 1.0 / (double)L.n;
      o.cx = xf + seg_sum(ux, L.lane, L.segS, L.segE) * ind;
      o.cy = yf + seg_sum(uy, L.lane, L.segS, L.segE) * ind;
    }
  } else {
    area = V.area[L.r];
    cx = V.cx[L.r];
    cy = V.cy[L.r];
    const double rx = pbx(x - cx, B), ry = pby(y - cy, B);
    past = __any(L.act && !(fabs((rx + dnx) * B.mx) < 0.4999 && fabs((ry + dny) * B.my) < 0.4999 &&
                            fabs((rx - psx) * B.mx) < 0.4999 && fabs((ry - psy) * B.my) < 0.4999));
  }
  if (write && L.act) {
    V.th[L.v] = theta;
    V.len[L.v] = seglen;
    if (L.lane == L.segS && !L.wide) {
      V.area[L.r] = area;
      V.perim[L.r] = perim;
      V.cx[L.r] = o.cx;
      V.cy[L.r] = o.cy;
    }
  }
  if (past) {  // the terms' differences of centre-relative positions, as ring_shape forms them
    const double rvx = pbx(x - cx, B), rvy = pby(y - cy, B);
    dnx = pbx(xn - cx, B) - rvx;
    dny = pby(yn - cy, B) - rvy;
    psx = rvx - pbx(xp - cx, B);
    psy = rvy - pby(yp - cy, B);
    n2 = dnx * dnx + dny * dny;
    in = rsqrt_n(n2);
    seglen = n2 > 0 ? sqrt_from(n2, in) : n2;
  }
  const double a0 = V.a0[L.r], ia0 = recip(a0);
  // shape costs: the global ea, el, eb, or per-ring values when the caller set them
  const double ea = V.kr ? V.kr[L.r] : P.ea;
  const double el = V.kr ? V.kr[V.np + L.r] : P.el;
  const double eb = V.kr ? V.kr[2 * V.np + L.r] : P.eb;
  // area term (calcAreaForceEnergy 429-435)
  const double deltaA = div_from(area, a0, ia0) - 1.;
  const double gmA = ea * deltaA * ia0;
  double fx = -0.5 * gmA * (psy + dny);
  double fy = 0.5 * gmA * (dnx + psx);
  // perimeter term (calcPerimeterForceEnergy 437-447 / FENE 449-455): each segment's factor cn
  const double l0v = V.l0[L.v];
  const bool harmonic = P.monomer == MONO_HARMONIC;
  auto factor = [&](double l0, double d2, double len, double id) {
    if (harmonic) {
      const double il0 = recip(l0);
      return (div_from(len, l0, il0) - 1.) * il0 * id;
    }
    return 2 * P.stiff * P.extSq * recip(P.extSq * l0 * l0 - d2);
  };
  const double cn = factor(l0v, n2, seglen, in), in2 = in * in;
  const double D = theta - V.th0[L.v];
  double cp = shfl_d(cn, L.pl), ip2 = shfl_d(in2, L.pl), Dp = shfl_d(D, L.pl), Dn = shfl_d(D, L.nl);
  if (L.wide) {  // from memory; the neighbours' angles from their own neighbours, as their lanes form them
    const double p2 = psx * psx + psy * psy, ip = rsqrt_n(p2);
    cp = factor(V.l0[vp], p2, sqrt_from(p2, ip), ip);
    ip2 = ip * ip;
    const int vpp = ring_prev(vp, L.f, L.n), vnn = ring_next(vn, L.f, L.n);
    Dp = vertex_theta(B, xp, yp, x, y, V.x[vpp], V.y[vpp]) - V.th0[vp];
    Dn = vertex_theta(B, xn, yn, V.x[vnn], V.y[vnn], x, y) - V.th0[vn];
  }
  fx += el * (cn * dnx - cp * psx);
  fy += el * (cn * dny - cp * psy);
  // bending term (calcBendingForceEnergy 457-471)
  const double preVar = (D - Dp) * ip2, nextVar = (D - Dn) * in2;
  fx += eb * (preVar * psy + nextVar * dny);
  fy -= eb * (preVar * psx + nextVar * dnx);
  if (write) {  // the previous segment's perimeter energy
    double l0p = shfl_d(l0v, L.pl);
    if (L.wide) l0p = V.l0[vp];
    const double p2 = psx * psx + psy * psy;
    double e = 0.5 * ea * deltaA * deltaA / (double)L.n + 0.5 * eb * D * D;
    if (harmonic) {
      const double pDelta = sqrt(p2) / l0p - 1.;
      e += 0.5 * el * pDelta * pDelta;
    } else {
      e += el * P.stiff * P.extSq * log(1 - p2 / (P.extSq * l0p * l0p));
    }
    o.e = e;
  }
  o.fx = fx; o.fy = fy;
  return o;
}

// The ring centre alone (calcParticlePos, cudaKernel.cuh:365-388), as ring_shape computes it,
// stored by the ring's first lane: the rigid rings' shape pass
__device__ __forceinline__ ShapeOut ring_centre(const View& V, const Lane& L, const Box& B, double x, double y, bool write) {
  ShapeOut o{0, 0, 0, 0, 0};
  const double xn = shfl_d(x, L.nl), yn = shfl_d(y, L.nl);
  const double xf = shfl_d(x, L.segS), yf = shfl_d(y, L.segS);
  const double dnx = pbx(xn - x, B), dny = pby(yn - y, B);
  double ux, uy;
  ring_walk(L, B, x, y, xf, yf, dnx, dny, ux, uy);
  const double sux = seg_sum(ux, L.lane, L.segS, L.segE);
  const double suy = seg_sum(uy, L.lane, L.segS, L.segE);
  const double ind = 1.0 / (double)L.n;
  o.cx = xf + sux * ind;
  o.cy = yf + suy * ind;
  if (write && L.act && L.lane == L.segS) {
    V.cx[L.r] = o.cx;
    V.cy[L.r] = o.cy;
  }
  return o;
}

// the pair terms in the reference's order (REF) or in the loops' form
template <int POT, bool REF>
__device__ __forceinline__ double pair_of(const Params& P, double dx, double dy, double sum, double& fx, double& fy) {
  if constexpr (REF) return pair_force<POT>(P, dx, dy, sum, fx, fy);
  return pair_force_n<POT>(P, dx, dy, sum, fx, fy);
}
template <int POT, bool REF>
__device__ __forceinline__ double smooth_this_of(const Params& P, const Box& B, double tix, double tiy, double tjx,
                                                 double tjy, double tpx, double tpy, double tqx, double tqy,
                                                 double sum, double& fx, double& fy) {
  if constexpr (REF) return smooth_pair<POT, ROLE_THIS>(P, B, tix, tiy, tjx, tjy, tpx, tpy, tqx, tqy, sum, fx, fy);
  return smooth_this_n<POT>(P, B, tix, tiy, tjx, tjy, tpx, tpy, tqx, tqy, sum, fx, fy);
}
template <int POT, bool REF>
__device__ __forceinline__ double smooth_op_of(const Params& P, const Box& B, double tix, double tiy, double tjx,
                                               double tjy, double tpx, double tpy, double tqx, double tqy, double sum,
                                               double& fx, double& fy, double& px, double& py) {
  if constexpr (REF) return smooth_pair_op<POT>(P, B, tix, tiy, tjx, tjy, tpx, tpy, tqx, tqy, sum, fx, fy, px, py);
  return smooth_op_n<POT>(P, B, tix, tiy, tjx, tjy, tpx, tpy, tqx, tqy, sum, fx, fy, px, py);
}

// Interparticle gather of lane L's vertex over entries k0, k0 + kstep, ... of its row:
// accumulates the force on v, the vertex-vertex energy e, the smooth energy es and the share
// (qx, qy) that v's `other` evaluation owes prev(v) (handed to prev(v)'s lane by the caller).
// On the last lane of a wide ring's slice, whose next vertex lies in another tile, (qnx, qny)
// accumulates the share that next(v)'s evaluations owe v, from next(v)'s row (complete before
// the launch: wide sets rebuild rows in their own launch).
template <int INTER, int POT, bool REF>
__device__ __forceinline__ void gather_pairs(const View& V, const Params& P, const Lane& L, const Box& B, double x,
                                             double y, int k0, int kstep, double& fx, double& fy, double& e,
                                             double& es, double& qx, double& qy, double& qnx, double& qny) {
  const double radv = V.rad[L.v];
  // Row entries are fetched one iteration ahead, the first one before the row length is known:
  // rows are W entries wide (unused entries hold -1), so k < W keeps every fetch in bounds, and
  // an entry is only used once k < ncnt is known.
  if constexpr (INTER == INT_VV) {
    // kernelCalcVertexInteraction, cudaKernel.cuh:690-722
    int j = k0 < V.W ? V.nbr[(long)k0 * V.nv + L.v] : 0;
    const int c = L.act ? V.ncnt[L.v] : 0;
    for (int k = k0; k < c; k += kstep) {
      const int kn = k + kstep;
      const int jn = kn < V.W ? V.nbr[(long)kn * V.nv + L.v] : 0;
      e += pair_of<POT, REF>(P, pbx(x - V.x[j], B), pby(y - V.y[j], B), radv + V.rad[j], fx, fy);
      j = jn;
    }
  } else if constexpr (INTER == INT_SMOOTH) {
    // kernelCalcSmoothInteraction, cudaKernel.cuh:922-975, as a gather: for every u in list(v),
    // (v, segment of u) gives v's `this` share, and (u, segment (prev(v), v)) gives v's
    // `other` share and prev(v)'s `previous` share (handed to prev(v)'s lane by the caller).
    // Ring neighbours of v; inactive lanes past the tile end use v itself (in bounds).
    int vp = L.act ? L.v0 + L.pl : L.v;
    int vpp = L.act ? L.v0 + ((L.pl > L.segS) ? L.pl - 1 : L.segE) : L.v;
    if (L.wide && L.act) {
      vp = ring_prev(L.v, L.f, L.n);
      vpp = ring_prev(vp, L.f, L.n);
    }
    const double xp = V.x[vp], yp = V.y[vp];
    const double xpp = V.x[vpp], ypp = V.y[vpp];
    int u = 0;
    int2 pp = make_int2(0, 0);
    if (k0 < V.W) {
      u = V.nbr[(long)k0 * V.nv + L.v];
      pp = V.nbrp[(long)k0 * V.nv + L.v];
    }
    const int c = L.act ? V.ncnt[L.v] : 0;
    for (int k = k0; k < c; k += kstep) {
      const int kn = k + kstep;
      int un = 0;
      int2 ppn = make_int2(0, 0);
      if (kn < V.W) {
        un = V.nbr[(long)kn * V.nv + L.v];
        ppn = V.nbrp[(long)kn * V.nv + L.v];
      }
      const double xu = V.x[u], yu = V.y[u];
      const double radSum = radv + V.rad[u];
      es += smooth_this_of<POT, REF>(P, B, x, y, xu, yu, V.x[pp.x], V.y[pp.x], V.x[pp.y], V.y[pp.y], radSum, fx, fy);
      es += smooth_op_of<POT, REF>(P, B, xu, yu, x, y, xp, yp, xpp, ypp, radSum, fx, fy, qx, qy);
      u = un;
      pp = ppn;
    }
    if (L.wide && L.act && L.lane == L.segE) {
      // (u, segment (v, next(v))) for u in list(next(v)): next(v)'s `other` share is its own
      // lane's; the `previous` share is v's (the energy is counted by next(v)'s lane)
      const int j = ring_next(L.v, L.f, L.n);
      const double xj = V.x[j], yj = V.y[j], radj = V.rad[j];
      const int cj = V.ncnt[j];
      for (int k = k0; k < cj; k += kstep) {
        const int w = V.nbr[(long)k * V.nv + j];
        double ox = 0, oy = 0;
        (void)smooth_op_of<POT, REF>(P, B, V.x[w], V.y[w], xj, yj, x, y, xp, yp, radj + V.rad[w], ox, oy, qnx, qny);
      }
    }
  } else {
    // kernelCalcAllToAllVertexInteraction, cudaKernel.cuh:725-757 (test mode)
    if (L.act) {
      const int b0 = V.svoff[L.s], b1 = V.svoff[L.s + 1];
      for (int j = b0 + k0; j < b1; j += kstep) {
        if (V.vring[j] == L.r) continue;
        e += pair_of<POT, REF>(P, pbx(x - V.x[j], B), pby(y - V.y[j], B), radv + V.rad[j], fx, fy);
      }
    }
  }
}

// -------------------------------------------------------------- step ---
// Waves of a tile: with nw > 1, wave 0 does the ring geometry, shape force and random draws
// while waves 1..nw-1 share the neighbour gather; with nw == 1 wave 0 does both in turn.
// Whether a displacement exceeds k cutoff / 3 (checkDisplacement, DPM2D.cu:1390-1406), by squares; a
// negative cutoff is exceeded by any
__device__ __forceinline__ bool moved_past(const Params& P, const Box& B, double dx, double dy, double k = 1.0) {
  dx = pbx(dx, B);
  dy = pby(dy, B);
  const double c = k * P.cutoff;
  return 9 * (dx * dx + dy * dy) > c * fabs(c);
}

// A drift that moved a vertex more than cutoff / 3 marks its system FLAG_FAR: the next rebuild
// cannot rely on the cells of its list positions (md_cells)
__device__ __forceinline__ void far_test(const Params& P, const Box& B, double dx, double dy, int* flag) {
  if (moved_past(P, B, dx, dy)) atomicOr(flag, FLAG_FAR);
}

// Rebuild flag of a vertex (dx, dy) from its list position: the displacement test, with FLAG_FAR beyond the
// 2 cutoff / 3 that the cells of the list positions allow for, however the vertex came there
__device__ __forceinline__ void moved_test(const Params& P, const Box& B, double dx, double dy, int* flag, int* any) {
  if (moved_past(P, B, dx, dy)) {
    atomicOr(flag, moved_past(P, B, dx, dy, 2.0) ? 1 | FLAG_FAR : 1);
    if (any) atomicOr(any, 1);
  }
}

// The step loop's cell lists of a system whose list positions (the positions of its last
// rebuild) have generation g: its rows are rebuilt from list g % 3, the rebuild bins its own
// positions (the next list positions) into list (g + 1) % 3, cleared by the rebuild before, and
// clears list (g + 2) % 3, which that rebuild read.  The cells are wide enough for a vertex 2
// cutoff / 3 from its list position: at most cutoff / 3 before the drift that triggers the
// rebuild (the displacement test) plus cutoff / 3 in that drift (else FLAG_FAR, all pairs).
struct MdCells {
  const int *cnt, *slots;  // read
  int *binCnt, *binSlots;  // binned into
  int* clear;              // cleared
};
__device__ __forceinline__ MdCells md_cells(int* cells, int* slots, const CellGrid& G, int g) {
  const long C = G.ncells, CS = (long)G.ncells * G.cap;
  const int k0 = g % 3, k1 = (g + 1) % 3, k2 = (g + 2) % 3;
  return MdCells{cells + k0 * C, slots + k0 * CS, cells + k1 * C, slots + k1 * CS, cells + k2 * C};
}

// A rebuild's own cells, by one wave of its tile: its positions are the system's next list positions (its
// rows are built from them), binned into the next cell list, and the list after that cleared.  Nothing
// in the launch reads either: the wave calls it behind the rebuild's barriers, which would wait for the
// bins' atomics.
__device__ __forceinline__ void md_bin_rebuilt(const View& V, const CellGrid& G, const MdCells& M, const Lane& L,
                                               const Box& B, double x, double y, int* err) {
  if (L.act) bin_vertex(G, B, M.binCnt, M.binSlots, L.v, L.s, x, y, err);
  if (!G.brute[L.s]) {
    const int t0 = V.stile[L.s], nt = V.stile[L.s + 1] - t0;
    const int n = G.ncx[L.s] * G.ncy[L.s];
    int* clr = M.clear + G.coff[L.s];
    for (int c = (L.tile - t0) * WAVE + L.lane; c < n; c += nt * WAVE) clr[c] = 0;
  }
}

// a rebuilding vertex at (x, y) farther than 2 cutoff / 3 from its list position: its cells may
// miss a neighbour (cannot happen while the displacement and far tests hold)
__device__ __forceinline__ void md_stale_test(const View& V, const Params& P, const Box& B, int v, double x, double y,
                                              int* err) {
  if (moved_past(P, B, x - V.lx[v], y - V.ly[v], 2.0)) atomicOr(err, ERR_STALE_BINS);
}

// ------------------------------------------------------------------ FIRE ---
// Sums an iteration starts from: v.F, max F_c^2, |F|^2, and |v|^2 after the half kick.  The step of that
// kick is known before v.F but for its sign: h1 when it is positive, h2 of a restart (which clears v first),
// so one exchange carries both outcomes, each vertex's half-kicked velocity rounded as the kick rounds it.
struct FireSums {
  double P, m, ff, v1, v2;
};
struct FireNext {
  double h1, h2;
  __device__ __forceinline__ FireNext(const FireParams& fp, const FireState& fs)
      : h1(0.5 * (fs.numStep + 1 > fp.minStep ? fmin(fs.dt * fp.f_inc, fp.dt_max) : fs.dt)),
        h2(0.5 * fmax(fs.dt * fp.f_dec, fp.dt_max / 10)) {}
};
__device__ __forceinline__ void fire_add(FireSums& a, const FireNext& n, double vx, double vy, double fx, double fy) {
  const double ux = vx + n.h1 * fx, uy = vy + n.h1 * fy, wx = n.h2 * fx, wy = n.h2 * fy;
  a.P += vx * fx + vy * fy;
  a.m = fmax(a.m, fmax(fx * fx, fy * fy));
  a.ff += fx * fx + fy * fy;
  a.v1 += ux * ux + uy * uy;
  a.v2 += wx * wx + wy * wy;
}
// workgroup sums (fixed order: lanes by butterfly, the first nw waves by index); every thread passes
// another barrier between two calls
__device__ __forceinline__ FireSums fire_block_sums(FireSums a, double (*red)[5], int nw) {
  const int w = threadIdx.x / WAVE;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    a.P += __shfl_xor(a.P, d, WAVE);
    a.m = fmax(a.m, __shfl_xor(a.m, d, WAVE));
    a.ff += __shfl_xor(a.ff, d, WAVE);
    a.v1 += __shfl_xor(a.v1, d, WAVE);
    a.v2 += __shfl_xor(a.v2, d, WAVE);
  }
  if ((threadIdx.x & (WAVE - 1)) == 0) {
    red[w][0] = a.P;
    red[w][1] = a.m;
    red[w][2] = a.ff;
    red[w][3] = a.v1;
    red[w][4] = a.v2;
  }
  __syncthreads();
  FireSums s{0, -1, 0, 0, 0};
  for (int q = 0; q < nw; q++) {
    s.P += red[q][0];
    s.m = fmax(s.m, red[q][1]);
    s.ff += red[q][2];
    s.v1 += red[q][3];
    s.v2 += red[q][4];
  }
  return s;
}
// checkFIREParams (FIRE.cu:338-371) with the stopping rule; true when the iteration restarts
__device__ __forceinline__ bool fire_update(FireState& fs, const FireParams& fp, const FireSums& s) {
  if (!fs.converged && (sqrt(s.m) <= fp.tol || fs.iters >= fp.maxIter)) fs.converged = 1;
  if (fs.converged) return false;
  const bool reset = !(s.P > 0);
  fs.P = s.P;
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
  return reset;
}
// back-step on reset (with the decreased dt), half kick, bendVertexVelocityTowardsForce
// (FIRE.cu:374-394) and drift of one vertex
__device__ __forceinline__ void fire_move(const FireState& fs, const FireSums& s, bool reset, double fx, double fy,
                                          double& x, double& y, double& vx, double& vy) {
  const double h = 0.5 * fs.dt, fa = fs.a;
  if (reset) {
    x -= h * vx;
    y -= h * vy;
    vx = 0;
    vy = 0;
  }
  vx += h * fx;
  vy += h * fy;
  if (s.ff > 0) {
    const double ratio = sqrt((reset ? s.v2 : s.v1) / s.ff);
    vx = (1 - fa) * vx + fa * fx * ratio;
    vy = (1 - fa) * vy + fa * fy * ratio;
  }
  x += fs.dt * vx;
  y += fs.dt * vy;
}

// ---------------------------------------------------------- rigid rings ---
// Half kick of a rigid ring: RigidNVE::updateVelocity (Simulator.cu:348-366), or
// RigidLangevin::updateVelocity (263-286) with its unit Gaussian pair (z0, z1) of the step and
// d_thermalVel zero; the angular velocity takes the torque / moment of inertia.
__device__ __forceinline__ void rigid_kick(bool langevin, double h, double gamma, double Fx, double Fy, double T,
                                           double z0, double z1, double& vx, double& vy, double& w) {
  if (langevin) {
    vx += h * (Fx - vx * gamma);
    vx -= 0.5 * h * h * (Fx - vx * gamma) / gamma;
    vx += z0;
    vy += h * (Fy - vy * gamma);
    vy -= 0.5 * h * h * (Fy - vy * gamma) / gamma;
    vy += z1;
  } else {
    vx += h * Fx;
    vy += h * Fy;
  }
  w += h * T;
}

// A ring's vertex after the ring moved from centre (cx, cy) to (ncx, ncy) and turned by dth:
// translateVertices then rotateVertices (kernelTranslateVertices / kernelRotateVertices,
// cudaKernel.cuh:1678-1713), each difference a box distance.
__device__ __forceinline__ void rigid_move(const Box& B, double x, double y, double cx, double cy, double ncx,
                                           double ncy, double c, double sn, double& xn, double& yn) {
  const double x1 = x + pbx(ncx - cx, B), y1 = y + pby(ncy - cy, B);
  const double dx = pbx(x1 - ncx, B), dy = pby(y1 - ncy, B);
  xn = x1 + ((dx * c - dy * sn) - dx);
  yn = y1 + ((dx * sn + dy * c) - dy);
}

// Per-tile partials of the rigid FIRE sums over the rings whose first vertex is in the tile:
// [0] v.F, [1] |v|^2, [2] |F|^2 (ring velocities and forces)
__device__ __forceinline__ void rigid_fire_partials(const Lane& L, bool head, double vx, double vy, double Fx,
                                                    double Fy, double* part) {
  const double p0 = wave_sum(head ? vx * Fx + vy * Fy : 0.0);
  const double p1 = wave_sum(head ? vx * vx + vy * vy : 0.0);
  const double p2 = wave_sum(head ? Fx * Fx + Fy * Fy : 0.0);
  if (L.lane == 0) {
    part[L.tile * 4 + 0] = p0;
    part[L.tile * 4 + 1] = p1;
    part[L.tile * 4 + 2] = p2;
  }
}

// Step-kernel epilogue of rigid rings (wave 0, one ring per lane segment): the interaction
// forces' transfer to the ring (calcRigidForceEnergy, DPM2D.cu:2128-2142: torque r x f about
// the centre, moment of inertia sum |r|^2, ring force sum f, ring torque sum (r x f) / I, ring
// energy sum e for vertexVertex), then the second half kick of this step and, with MODE_START,
// the next step's first half: last centre and angle stored, half kick with the next step's
// draw, centre and angle advanced, vertices moved (RigidNVE / RigidLangevin::integrate,
// Simulator.cu:241-252, 316-326).  With MODE_FIRE the half kick takes the system's FIRE step.
template <int MODE, bool VV, bool STORE>
__device__ __forceinline__ void rigid_epilogue(const View& V, const Params& P, const StepArgs& A, const Lane& L,
                                               const Box& B, double x, double y, double fx, double fy, double e,
                                               double cx, double cy, double lx, double ly, double z0, double z1) {
  const Rigid R = *V.rg;
  const double rx = pbx(x - cx, B), ry = pby(y - cy, B);
  const double tq = rx * fy - ry * fx;
  const double I = seg_sum(L.act ? rx * rx + ry * ry : 0.0, L.lane, L.segS, L.segE);
  const double Fx = seg_sum(L.act ? fx : 0.0, L.lane, L.segS, L.segE);
  const double Fy = seg_sum(L.act ? fy : 0.0, L.lane, L.segS, L.segE);
  const double T = seg_sum(L.act ? tq : 0.0, L.lane, L.segS, L.segE) / I;
  double E = 0;
  if constexpr (VV && STORE) E = seg_sum(L.act ? e : 0.0, L.lane, L.segS, L.segE);
  const bool head = L.act && L.lane == L.segS;
  double vx = 0, vy = 0, w = 0;
  if constexpr (MODE != MODE_RIGID) {
    if (L.act) {
      vx = R.pvx[L.r];
      vy = R.pvy[L.r];
      w = R.pw[L.r];
    }
  }
  if constexpr ((MODE & MODE_FIRE) != 0) {
    // the second half kick with the system's FIRE step, then the tile partials of the next
    // iteration's sums (every lane takes part in the wave sums)
    if (L.act) rigid_kick(false, 0.5 * A.fire[L.s].dt, 0.0, Fx, Fy, T, 0.0, 0.0, vx, vy, w);
    rigid_fire_partials(L, head, vx, vy, Fx, Fy, A.part);
  }
  if (!L.act) return;
  if constexpr (STORE) {
    V.fx[L.v] = fx;
    V.fy[L.v] = fy;
    V.ev[L.v] = e;
    R.vtq[L.v] = tq;
    if (head) {
      R.pfx[L.r] = Fx;
      R.pfy[L.r] = Fy;
      R.ptq[L.r] = T;
      R.moi[L.r] = I;
      if constexpr (VV) V.pe[L.r] = E;
    }
  }
  if constexpr (MODE == MODE_RIGID) return;
  if constexpr ((MODE & MODE_FIRE) == 0) {
    rigid_kick(A.rigidLangevin, A.h, P.gamma, Fx, Fy, T, z0, z1, vx, vy, w);
    if constexpr ((MODE & MODE_START) != 0) {
      double n0 = 0, n1 = 0;
      if (A.rigidLangevin)
        gauss_pair(P.seed, (uint32_t)L.s, TAG_THERMAL, A.ctr[0] + (unsigned long long)A.ctrOffT + 1ull,
                   (uint32_t)(L.r - V.sroff[L.s]), n0, n1);
      rigid_kick(A.rigidLangevin, A.h, P.gamma, Fx, Fy, T, n0, n1, vx, vy, w);
      const double ang = V.ang[L.r];
      const double ncx = cx + A.dt * vx, ncy = cy + A.dt * vy, nang = ang + A.dt * w;
      const double dth = nang - ang;
      double xn, yn;
      rigid_move(B, x, y, cx, cy, ncx, ncy, cos(dth), sin(dth), xn, yn);
      A.xout[L.v] = xn;
      A.yout[L.v] = yn;
      if (moved_past(P, B, xn - lx, yn - ly)) {
        atomicOr(&A.flagOut[L.s], 1);
        atomicOr(A.anyOut, 1);
      }
      far_test(P, B, xn - x, yn - y, A.flagOut + L.s);
      if (head) {
        V.ang[L.r] = nang;
        V.cx[L.r] = ncx;
        V.cy[L.r] = ncy;
      }
    }
  }
  if (head) {
    R.pvx[L.r] = vx;
    R.pvy[L.r] = vy;
    R.pw[L.r] = w;
  }
}

}  // namespace dpm
