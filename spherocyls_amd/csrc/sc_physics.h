// Device-side physics shared by the tile and list force kernels: the pair
// force, minimum image, wrapping, cell binning and block reductions.
#pragma once

#include <hip/hip_runtime.h>

#include "sc_internal.h"

namespace sc {

// ---------------------------------------------------------------------------
// pair math
// ---------------------------------------------------------------------------
template <typename T>
struct PairOut {
  T fx, fy, tp, tq, s, t, dx, dy, dist, dV;
};

// Crossed segments (their lines meet inside both): the closest distance is 0
// and stays 0 under small displacements, and D is rounding noise.  The overlap
// energy is continued to negative distance d = -delta, delta the minimal
// translation that uncrosses them: the smallest distance of an endpoint from
// the other segment's line.  That endpoint's segment is pushed back across
// the line; the force is (1 + delta/sigma)/sigma along the push, at the
// endpoint and at its projection on the other segment -- the ordinary contact
// force of the configuration it uncrosses into, so force and energy are
// continuous where the rods uncross.  Fills o as a contact with dist = -delta.
template <typename T>
__device__ __forceinline__ void crossed_contact(T ddx, T ddy, T nxA, T nyA, T nxB, T nyB, T sig,
                                                PairOut<T>& o) {
#pragma clang fp contract(off)
  const T la2 = nxA * nxA + nyA * nyA, lb2 = nxB * nxB + nyB * nyB;
  const T la = sqrt(la2), lb = sqrt(lb2);
  // unit normals of the segments
  const T mAx = -nyA / la, mAy = nxA / la, mBx = -nyB / lb, mBy = nxB / lb;
  // A's endpoints (relative to B's centre) against B's line, and B's against A's
  const T hp = (ddx + nxA) * mBx + (ddy + nyA) * mBy;
  const T hm = (ddx - nxA) * mBx + (ddy - nyA) * mBy;
  const T gp = (-ddx + nxB) * mAx + (-ddy + nyB) * mAy;
  const T gm = (-ddx - nxB) * mAx + (-ddy - nyB) * mAy;
  const T dA = fmin(fabs(hp), fabs(hm)), dB = fmin(fabs(gp), fabs(gm));
  T s, t, ux, uy, delta;
  if (dA <= dB) {  // move A: its nearer endpoint back across B's line
    s = fabs(hp) <= fabs(hm) ? T(1) : T(-1);
    const T h = s > 0 ? hp : hm;
    ux = h > 0 ? -mBx : mBx;
    uy = h > 0 ? -mBy : mBy;
    t = fmin(fmax(((ddx + s * nxA) * nxB + (ddy + s * nyA) * nyB) / lb2, T(-1)), T(1));
    delta = dA;
  } else {  // move B: its nearer endpoint back across A's line (A gets -F_B)
    t = fabs(gp) <= fabs(gm) ? T(1) : T(-1);
    const T gg = t > 0 ? gp : gm;
    ux = gg > 0 ? mAx : -mAx;
    uy = gg > 0 ? mAy : -mAy;
    s = fmin(fmax(((-ddx + t * nxB) * nxA + (-ddy + t * nyB) * nyA) / la2, T(-1)), T(1));
    delta = dB;
  }
  const T dV = (T(1) + delta / sig) / sig;
  const T fx = ux * dV, fy = uy * dV;
  o.fx = fx;
  o.fy = fy;
  o.tp = s * nxA * fy - s * nyA * fx;
  o.tq = t * nyB * fx - t * nxB * fy;
  o.s = s;
  o.t = t;
  o.dist = -delta;
  o.dx = -delta * ux;
  o.dy = -delta * uy;
  o.dV = dV;
}

// Whether two segments intersect: each one's endpoints lie strictly on
// opposite sides of the other's line (cross products, no normalisation).  The
// closest-approach test of crossing (|tu| < 1 and |s| < 1) also fires on noise
// for nearly parallel segments, whose det = a c - b^2 loses its digits to
// cancellation (in FP32 from angles of ~1e-3 down); a crossing is taken only
// when this test confirms it.  For such pairs the endpoints sit a contact
// distance from the other line, far above the rounding of these products.
template <typename T>
__device__ __forceinline__ bool segments_cross(T ddx, T ddy, T nxA, T nyA, T nxB, T nyB) {
#pragma clang fp contract(off)
  const T hp = nxB * (ddy + nyA) - nyB * (ddx + nxA);
  const T hm = nxB * (ddy - nyA) - nyB * (ddx - nxA);
  const T gp = nxA * (nyB - ddy) - nyA * (nxB - ddx);
  const T gm = nxA * (-nyB - ddy) - nyA * (-nxB - ddx);
  return ((hp > T(0) && hm < T(0)) || (hp < T(0) && hm > T(0))) &&
         ((gp > T(0) && gm < T(0)) || (gp < T(0) && gm > T(0)));
}

// Division x / d with a reciprocal that several quotients share.  r =
// reciprocal(d) is the hardware estimate after two Newton steps; the quotient's
// residual is corrected once by fused multiply-adds, which rounds it
// correctly (Markstein) as the compiler's own division sequence does, in 3
// instructions instead of 11 and without its scaling for operands near the
// ends of the exponent range, which lengths and forces do not come near.
// d = 0 gives NaN, also for x != 0: used only where x = 0 then (a disc's
// squared half length), or d > 0.  The pair math is a chain of dependent FP64
// operations (a division is 70 cycles of latency, this 20): 262k particles
// sheared by 100 steps, 7.97 -> 7.59 ms together with root() below.
__device__ __forceinline__ double reciprocal(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
  return fma(fma(-d, r, 1.0), r, r);
}
__device__ __forceinline__ double over(double x, double d, double r) {
  const double q = x * r;
  return fma(fma(-d, q, x), r, q);
}

// sqrt(v) for v > 0 away from the ends of the exponent range, and a reciprocal
// of it for over(): the compiler's sequence without its scaling.
__device__ __forceinline__ double root(double v, double& rinv) {
  const double y = __builtin_amdgcn_rsq(v);
  double g = v * y, h = 0.5 * y;
  const double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  g = fma(fma(-g, g, v), h, g);
  g = fma(fma(-g, g, v), h, g);
  rinv = h + h;
  rinv = fma(fma(-g, rinv, 1.0), rinv, rinv);
  return g;
}

// Segment-segment closest approach and harmonic contact force, following
// calc_force_pair (src/cpp/strain_dynamics.cpp:38-64) term by term.  Returns
// false when |D| >= sigma (or D is NaN).  FP64: no contraction, so the rounding
// matches the reference's x86-64 build.
__device__ __forceinline__ bool pair_contact_f64(double ddx, double ddy, double nxA, double nyA,
                                                 double nxB, double nyB, double Ap, double Aq,
                                                 double sig, PairOut<double>& o) {
#pragma clang fp contract(off)
  double a = Ap * Ap;
  double b = -(nxA * nxB + nyA * nyB);
  double c = Aq * Aq;
  double d = nxA * ddx + nyA * ddy;
  double e = -nxB * ddx - nyB * ddy;
  double det = a * c - b * b;
  double tu = (b * d - a * e) / det;
  double t = fmin(fmax(tu, -1.0), 1.0);
  double s = over(-(b * t + d), a, reciprocal(a));
  double sabs = fabs(s);
  s = fmin(fmax(s, -1.0), 1.0);
  if (sabs > 1.0) t = fmin(fmax(over(-(b * s + e), c, reciprocal(c)), -1.0), 1.0);
  double Dx = ddx + s * nxA - t * nxB;
  double Dy = ddy + s * nyA - t * nyB;
  double d2 = Dx * Dx + Dy * Dy;
  if (!(d2 < sig * sig)) return false;
  o.s = s;
  o.t = t;
  o.dx = Dx;
  o.dy = Dy;
  if (det > 0.0 && fabs(tu) < 1.0 && sabs < 1.0 &&
      segments_cross(ddx, ddy, nxA, nyA, nxB, nyB)) {
    crossed_contact(ddx, ddy, nxA, nyA, nxB, nyB, sig, o);  // crossed segments
    return true;
  }
  if (d2 == 0.0) {  // touching exactly (ends, collinear overlap): no direction
    o.fx = o.fy = o.tp = o.tq = 0.0;
    o.dist = 0.0;
    o.dV = 1.0 / sig;
    return true;
  }
  double rd, rs = reciprocal(sig);
  double dist = root(d2, rd);
  double dV = over(1.0 - over(dist, sig, rs), sig, rs);
  double fx = over(Dx * dV, dist, rd);
  double fy = over(Dy * dV, dist, rd);
  o.fx = fx;
  o.fy = fy;
  o.tp = s * nxA * fy - s * nyA * fx;
  o.tq = t * nyB * fx - t * nxB * fy;
  o.dist = dist;
  o.dV = dV;
  return true;
}

// ---------------------------------------------------------------------------
// two-point contact model
// ---------------------------------------------------------------------------
// Force fields of one contact point from its D vector (harmonic, as above).
template <typename T>
__device__ __forceinline__ bool contact_point(T Dx, T Dy, T s, T t, T nxA, T nyA, T nxB, T nyB,
                                              T sig, bool crossed, T ddx, T ddy, PairOut<T>& o) {
#pragma clang fp contract(off)
  T d2 = Dx * Dx + Dy * Dy;
  if (crossed) {  // as in pair_contact_f64
    crossed_contact(ddx, ddy, nxA, nyA, nxB, nyB, sig, o);
    return true;
  }
  if (!(d2 < sig * sig)) return false;
  o.s = s;
  o.t = t;
  o.dx = Dx;
  o.dy = Dy;
  if (d2 == T(0)) {
    o.fx = o.fy = o.tp = o.tq = T(0);
    o.dist = T(0);
    o.dV = T(1) / sig;
    return true;
  }
  T dist, dV, fx, fy;
  if constexpr (sizeof(T) == sizeof(double)) {
    double rd, rs = reciprocal(sig);
    dist = root(d2, rd);
    dV = over(1.0 - over(dist, sig, rs), sig, rs);
    fx = over(Dx * dV, dist, rd);
    fy = over(Dy * dV, dist, rd);
  } else {
    dist = sqrt(d2);
    dV = (T(1) - dist / sig) / sig;
    fx = Dx * dV / dist;
    fy = Dy * dV / dist;
  }
  o.fx = fx;
  o.fy = fy;
  o.tp = s * nxA * fy - s * nyA * fx;
  o.tq = t * nyB * fx - t * nxB * fy;
  o.dist = dist;
  o.dV = dV;
  return true;
}

// Mixed precision (FP32 pair forces).  The closest-approach parameters s, t
// and the crossing decision stay FP64, in pair_contact_f64's order: they come
// from differences of nearly equal products (det = a c - b^2, b d - a e), which
// in FP32 are noise for nearly parallel rods -- a noise tu in (-1, 1) would
// put the contact anywhere along the overlap, or call the pair crossed.  The
// contact vector D is formed in FP64 as well; its length, the overlap force
// and the torques are FP32.
__device__ __forceinline__ bool pair_contact_mixed(double ddx, double ddy, double nxA, double nyA,
                                                   double nxB, double nyB, double Ap, double Aq,
                                                   double sig, PairOut<float>& o) {
#pragma clang fp contract(off)
  double a = Ap * Ap;
  double b = -(nxA * nxB + nyA * nyB);
  double c = Aq * Aq;
  double d = nxA * ddx + nyA * ddy;
  double e = -nxB * ddx - nyB * ddy;
  double det = a * c - b * b;
  double tu = (b * d - a * e) / det;
  double t = fmin(fmax(tu, -1.0), 1.0);
  double s = -(b * t + d) / a;
  double sabs = fabs(s);
  s = fmin(fmax(s, -1.0), 1.0);
  if (sabs > 1.0) t = fmin(fmax(-(b * s + e) / c, -1.0), 1.0);
  const bool crossed = det > 0.0 && fabs(tu) < 1.0 && sabs < 1.0 &&
                       segments_cross(ddx, ddy, nxA, nyA, nxB, nyB);
  return contact_point<float>((float)(ddx + s * nxA - t * nxB), (float)(ddy + s * nyA - t * nyB),
                              (float)s, (float)t, (float)nxA, (float)nyA, (float)nxB, (float)nyB,
                              (float)sig, crossed, (float)ddx, (float)ddy, o);
}

template <typename T>
__device__ __forceinline__ T clamp1(T v) {
  return fmin(fmax(v, T(-1)), T(1));
}

// Two-point contact model (src/cuda/2point_dynamics.cu:391-546).  Besides the
// closest pair of points (s1, t1), a second pair (s2, t2) -- for nearly parallel
// rods the other end of their overlap -- carries its own harmonic contact when
// it overlaps as well, so two overlapping, nearly aligned rods have no energy
// kink at alignment.  The second pair starts at the opposite end of whichever
// segment fixed the first (s2 = -s1 or t2 = -t1) projected onto the other
// segment; a third candidate from the other segment's matching end replaces it
// when it is closer.  o0 / h0: the closest-point contact; o1 / h1: the second.
// The candidate parameters, every choice between them and the contact vectors
// are FP64; T is the type of each contact's force evaluation (FP32 in mixed
// mode, see pair_contact_mixed).
template <typename T>
__device__ __forceinline__ void pair_contacts_2p(double ddx, double ddy, double nxA, double nyA,
                                                 double nxB, double nyB, double Ap, double Aq,
                                                 double sig, PairOut<T>& o0, bool& h0,
                                                 PairOut<T>& o1, bool& h1) {
#pragma clang fp contract(off)
  const double a = Ap * Ap;
  const double b = -(nxA * nxB + nyA * nyB);
  const double c = Aq * Aq;
  const double d = nxA * ddx + nyA * ddy;
  const double e = -nxB * ddx - nyB * ddy;
  const double det = a * c - b * b;
  double s1, t1, s2, t2, s3, t3;
  bool crossed = false;
  if (det <= 0.0) {  // parallel: the two ends of the overlap
    s1 = clamp1(-(b + d) / a);
    s2 = clamp1(-(d - b) / a);
    if (fabs(s1) == 1.0) t1 = clamp1(-(b * s1 + e) / c);
    else t1 = b < 0.0 ? clamp1(-(b + e) / c) : clamp1(-(e - b) / c);
    if (fabs(s2) == 1.0) t2 = clamp1(-(b * s2 + e) / c);
    else t2 = b < 0.0 ? clamp1(-(e - b) / c) : clamp1(-(b + e) / c);
    s3 = s2;
    t3 = t2;
  } else {
    const double tu = (b * d - a * e) / det;
    const double ra = reciprocal(a), rc = reciprocal(c);
    t1 = clamp1(tu);
    s1 = over(-(b * t1 + d), a, ra);
    const double sarg = fabs(s1);
    s1 = clamp1(s1);
    crossed = fabs(tu) < 1.0 && sarg < 1.0 && segments_cross(ddx, ddy, nxA, nyA, nxB, nyB);
    // The rod whose end (u1 = +-1) fixed the first contact, A if s1 was clamped
    // and else B (whose t1 was): its parameters are u, the other rod's v.  The
    // two cases mirror each other, so both run the same instructions.
    const bool endA = sarg >= 1.0;
    if (endA) t1 = clamp1(over(-(b * s1 + e), c, rc));
    const double u1 = endA ? s1 : t1;
    const double nu = endA ? d : e, du = endA ? a : c, ru = endA ? ra : rc;
    const double nv = endA ? e : d, dv = endA ? c : a, rv = endA ? rc : ra;
    double u2 = -u1;
    double v2 = over(-(b * u2 + nv), dv, rv);
    const bool beyond = fabs(v2) > 1.0;
    v2 = clamp1(v2);
    // one division serves u2 (the second contact beyond v's end) or u3
    double v3 = b < 0.0 ? -u1 : u1;
    const double uq = over(-(b * (beyond ? v2 : v3) + nu), du, ru);
    double u3 = clamp1(uq);
    if (beyond) {
      u2 = u3;
      v3 = v2;
    } else if (fabs(uq) >= 1.0) {
      v3 = clamp1(over(-(b * u3 + nv), dv, rv));
    }
    s2 = endA ? u2 : v2;
    t2 = endA ? v2 : u2;
    s3 = endA ? u3 : v3;
    t3 = endA ? v3 : u3;
  }
  h0 = contact_point<T>(T(ddx + s1 * nxA - t1 * nxB), T(ddy + s1 * nyA - t1 * nyB), T(s1), T(t1),
                        T(nxA), T(nyA), T(nxB), T(nyB), T(sig), crossed, T(ddx), T(ddy), o0);
  h1 = false;
  if (s1 != s2 && t1 != t2) {
    double Dx2 = ddx + s2 * nxA - t2 * nxB;
    double Dy2 = ddy + s2 * nyA - t2 * nyB;
    if (s3 != s1 && s3 != s2) {
      const double Dx3 = ddx + s3 * nxA - t3 * nxB;
      const double Dy3 = ddy + s3 * nyA - t3 * nyB;
      if (Dx3 * Dx3 + Dy3 * Dy3 < Dx2 * Dx2 + Dy2 * Dy2) {
        s2 = s3;
        t2 = t3;
        Dx2 = Dx3;
        Dy2 = Dy3;
      }
    }
    h1 = contact_point<T>(T(Dx2), T(Dy2), T(s2), T(t2), T(nxA), T(nyA), T(nxB), T(nyB), T(sig),
                          false, T(ddx), T(ddy), o1);
  }
}

template <typename T>
__device__ __forceinline__ void widen(const PairOut<T>& a, PairOut<double>& o) {
  o.fx = a.fx; o.fy = a.fy; o.tp = a.tp; o.tq = a.tq; o.s = a.s; o.t = a.t;
  o.dx = a.dx; o.dy = a.dy; o.dist = a.dist; o.dV = a.dV;
}

// Contacts of one pair in the orientation given (A = lower id): the
// closest-point model of the CPU reference, or (TWO_POINT) the two-point model;
// FP64 or mixed (FP32 force evaluation) pair math, FP64 results.  o0 / h0:
// closest-point contact; o1 / h1: the second contact of the two-point model.
template <bool TWO_POINT>
__device__ __forceinline__ void pair_contacts(double ddx, double ddy, double nxA, double nyA,
                                              double nxB, double nyB, double Ap, double Aq,
                                              double sig, bool fp64, PairOut<double>& o0,
                                              bool& h0, PairOut<double>& o1, bool& h1) {
  if (!TWO_POINT) {
    h1 = false;
    if (fp64) {
      h0 = pair_contact_f64(ddx, ddy, nxA, nyA, nxB, nyB, Ap, Aq, sig, o0);
    } else {
      PairOut<float> f0;
      h0 = pair_contact_mixed(ddx, ddy, nxA, nyA, nxB, nyB, Ap, Aq, sig, f0);
      if (h0) widen(f0, o0);
    }
    return;
  }
  if (fp64) {
    pair_contacts_2p<double>(ddx, ddy, nxA, nyA, nxB, nyB, Ap, Aq, sig, o0, h0, o1, h1);
  } else {
    PairOut<float> f0, f1;
    pair_contacts_2p<float>(ddx, ddy, nxA, nyA, nxB, nyB, Ap, Aq, sig, f0, h0, f1, h1);
    if (h0) widen(f0, o0);
    if (h1) widen(f1, o1);
  }
}

// Stress / energy sums of one contact point of pair (A, B) (A = lower id):
// the reference's formulas with their two slips (src/cpp/spherocyl_box.cpp:
// 483-495) and the corrected virial, unnormalised (k_reduce divides).
__device__ __forceinline__ void add_contact_sums(const PairOut<double>& r, double nxA, double nyA,
                                                 double nxB, double nyB, double sig, double* acc) {
#pragma clang fp contract(off)
  double cxa = r.s * nxA - 0.5 * r.dx;
  double cya = r.s * nyA - 0.5 * r.dy;
  double cxb = r.t * nxB + 0.5 * r.dx;
  double cyb_ref = r.t * nxB + 0.5 * r.dy;
  double cyb = r.t * nyB + 0.5 * r.dy;
  acc[kSeE] += r.dV * sig * (1.0 - r.dist / sig);
  acc[kSePxx] += r.fx * cxa - r.fx * cxb - r.fy * cxb;
  acc[kSePyy] += r.fy * cya - r.fy * cyb_ref;
  acc[kSePxy] += r.fy * cxa;
  acc[kSeCPxx] += r.fx * (cxa - cxb);
  acc[kSeCPyy] += r.fy * (cya - cyb);
  acc[kSeCPxy] += r.fy * (cxa - cxb);
  acc[kSeCPyx] += r.fx * (cya - cyb);
}

// Sine and cosine of a rod's angle.  The test makes the library's reduction
// for huge arguments unreachable, so its code, constants and registers leave
// every kernel that moves particles (moving a particle of a one-launch FIRE:
// 3100 -> 1200 cycles); values are the library's.  An angle of 2^20 or more (a
// rod that turned 166 thousand times) first loses its whole turns, by multiples
// of 2 pi held in two words: within 1e-12 up to 1e19, where the angle's own
// last bit is many turns, and finite beyond.
__device__ __forceinline__ void rod_sincos(double x, double* sn, double* cs) {
  double r = x;
  for (int i = 0; i < 24 && !(fabs(r) < 1048576.0); ++i) {
    const double k = rint(r * 0.15915494309189535);
    r = fma(-k, 2.4492935982947064e-16, fma(-k, 6.283185307179586, r));
  }
  if (fabs(r) < 1048576.0) {
    sincos(r, sn, cs);
  } else {  // not finite
    *sn = r - r;
    *cs = 1.0 + *sn;
  }
}

// Minimum image in sheared coordinates (src/cpp/strain_dynamics.cpp:28-29).
__device__ __forceinline__ double min_image(double d, double L) {
#pragma clang fp contract(off)
  return d + L * (double)((d < -0.5 * L) - (d > 0.5 * L));
}

// Wrap rule of find_cells (src/cpp/spherocyl_box.cpp:279-286); bounded so a
// runaway coordinate cannot spin.  Returns false for a non-finite coordinate.
__device__ __forceinline__ bool wrap_coord(double& v, double L) {
  if (v >= 0.0 && v <= L) return true;
  if (!isfinite(v)) return false;
  int guard = 0;
  while (v > L && guard < 8) { v -= L; ++guard; }
  while (v < 0.0 && guard < 16) { v += L; ++guard; }
  if (guard >= 8) v = v - L * floor(v / L);
  return true;
}

__device__ __forceinline__ void wrap_angle(double& p) {
  if (!isfinite(p)) return;
  int guard = 0;
  while (p > kRefPi && guard < 8) { p -= 2 * kRefPi; ++guard; }
  while (p < -kRefPi && guard < 16) { p += 2 * kRefPi; ++guard; }
}

// Column and row of a wrapped position: find_cells' floor(x / w)
// (src/cpp/spherocyl_box.cpp:293-295) as floor(x cols / Lx), one division
// instead of two, clamped so x == L stays in range.  Every kernel that bins a
// particle or looks up its own cell uses this one rule, so a particle's cell
// is the same wherever it is computed.
__device__ __forceinline__ void cell_col_row(double xw, double yw, double Lx, double Ly,
                                             const PackInfo& P, int& col, int& row) {
  col = min(max((int)(xw * ((double)P.cols / Lx)), 0), P.cols - 1);
  row = min(max((int)(yw * ((double)P.rows / Ly)), 0), P.rows - 1);
}

__device__ __forceinline__ int cell_of(double xw, double yw, double Lx, double Ly,
                                      const PackInfo& P) {
  int col, row;
  cell_col_row(xw, yw, Lx, Ly, P, col, row);
  return P.coff + row * P.cols + col;
}

// Bin one particle into bucket buffer (cnt, slot).
__device__ __forceinline__ void bin_into(int g, double xw, double yw, double Lx, double Ly,
                                         const PackInfo& P, int* cnt, int* slot, int* err) {
  const int c = cell_of(xw, yw, Lx, Ly, P);
  int k = atomicAdd(&cnt[c], 1);
  if (k < P.cap) slot[(size_t)c * P.cap + k] = g;
  else atomicOr(err, kErrCellOverflow);
}

// Wavefront-aggregated bucket fill.  Every lane of the wavefront calls it
// (uniform control flow); lane l with c >= 0 puts particle g into bucket c.
// Particles are handled by lanes STRIDE apart (lane 0 of each particle's
// lanes), and storage is sorted by cell, so neighbouring particles often share
// a cell: each run of such lanes with one cell takes its slots with a single
// atomic, issued by the run's first lane, and the lanes of the run take
// consecutive slots from the returned base.  All runs' atomics are issued
// together.  Slot order within a bucket carries no meaning (rows and re-sorts
// order members by particle id).  It pays in the minimiser update, whose
// wavefronts do little besides the binning (about 2.5 particles per cell);
// the Heun passes keep one atomic per particle, which measured no slower there.
template <int STRIDE>
__device__ __forceinline__ void bin_wave(int c, int g, int cap, int* cnt, int* slot, int* err) {
  const int lane = __lane_id();
  const bool act = c >= 0;
  const int cp = __shfl_up(c, STRIDE);  // lanes below STRIDE read their own value
  const bool head = act && (lane < STRIDE || cp != c);
  const unsigned long long actm = __ballot(act), heads = __ballot(head);
  const unsigned long long below = (1ull << lane) - 1ull;  // lanes < lane
  const unsigned long long upto = (2ull << lane) - 1ull;   // lanes <= lane (all for lane 63)
  // first lane of this lane's run (the highest head at or below it)
  const unsigned long long hm = heads & upto;
  const int h = act && hm ? 63 - __clzll((long long)hm) : lane;
  int base = 0;
  if (head) {
    const unsigned long long after = heads & ~upto;  // heads above this lane
    const int end = after ? __ffsll((long long)after) - 1 : 64;
    const unsigned long long span = (end == 64 ? ~0ull : ((1ull << end) - 1ull)) & ~below;
    base = atomicAdd(&cnt[c], __popcll(actm & span));
  }
  base = __shfl(base, h);
  if (act) {
    const int k = base + __popcll(actm & below & ~((1ull << h) - 1ull));
    if (k < cap) slot[(size_t)c * cap + k] = g;
    else atomicOr(err, kErrCellOverflow);
  }
}

// isolated_rotation, src/cpp/strain_dynamics.cpp:174-177: 0.5 (1 - RC cos 2 phi),
// with cos 2 phi taken from the segment vector (nx, ny) = A (cos phi, sin phi)
// the state carries, (nx^2 - ny^2) / A^2, instead of an FP64 cosine (a disc,
// A = 0, has RC = 0).  It differs from cos(2 phi) by rounding only.
__device__ __forceinline__ double iso_rot_seg(double RC, double nx, double ny, double A) {
#pragma clang fp contract(off)
  const double c2 = A > 0.0 ? (nx * nx - ny * ny) / (A * A) : 1.0;
  return 0.5 * (1 - RC * c2);
}

// Force of partner q on particle i (i's data in registers), accumulated into
// (Fx, Fy, Tq) and, for the lower-id side of the pair, into the stress/energy
// sums.  The pair is evaluated in the reference's orientation (lower particle
// id first, src/cpp/spherocyl_box.cpp:514-520) so both sides agree bitwise.
template <bool SUMS, bool TWO_POINT>
__device__ __forceinline__ void pair_into(double xi, double yi, double nxi, double nyi, double Ri,
                                          double Ai, int idi, double xq, double yq, double nxq,
                                          double nyq, double Rq, double Aq, int idq, double Lx,
                                          double Ly, double gam, bool fp64, bool do_se,
                                          double& Fx, double& Fy, double& Tq, double* acc) {
#pragma clang fp contract(off)
  const bool iP = idi < idq;
  double ddx = min_image(iP ? xi - xq : xq - xi, Lx);
  double ddy = min_image(iP ? yi - yq : yq - yi, Ly);
  ddx += gam * ddy;
  const double sig = Ri + Rq;
  const double nxA = iP ? nxi : nxq, nyA = iP ? nyi : nyq;
  const double nxB = iP ? nxq : nxi, nyB = iP ? nyq : nyi;
  const double Ap = iP ? Ai : Aq, Aqq = iP ? Aq : Ai;
  PairOut<double> r0, r1;
  bool h0, h1;
  pair_contacts<TWO_POINT>(ddx, ddy, nxA, nyA, nxB, nyB, Ap, Aqq, sig, fp64, r0, h0, r1, h1);
  if (h0) {
    if (iP) {
      Fx += r0.fx;
      Fy += r0.fy;
      Tq += r0.tp;
      if (SUMS && do_se) {
        add_contact_sums(r0, nxA, nyA, nxB, nyB, sig, acc);
        acc[kSeNc] += 1.0;
      }
    } else {
      Fx -= r0.fx;
      Fy -= r0.fy;
      Tq += r0.tq;
    }
  }
  if (TWO_POINT && h1) {
    if (iP) {
      Fx += r1.fx;
      Fy += r1.fy;
      Tq += r1.tp;
      if (SUMS && do_se) add_contact_sums(r1, nxA, nyA, nxB, nyB, sig, acc);
    } else {
      Fx -= r1.fx;
      Fy -= r1.fy;
      Tq += r1.tq;
    }
  }
}

// What a minimiser does after a force pass, from its packing's sums: the FIRE
// step (velocity mixing or retreat, time step and mixing factor, convergence)
// or the gradient-descent stop test.  Cheap enough that every wavefront that
// moves particles takes it for itself.
struct MinStep {
  double dt_old, dt, alpha, npos;  // FIRE: time step before and after, mixing factor, uphill count
  double c_keep, c_force;          // FIRE: velocity = c_keep v + c_force g (mix), or a retreat
  double frms;                     // set where it can end the run (or with `residual`)
  int mix, prec;
  int end;                         // 0: go on, 1: converged, 2: FIRE at max_iter
};

// What the step depends on besides the sums.
struct MinState {
  double dt, alpha, npos;
  int step, prec;
};
__device__ __forceinline__ MinState min_state(const PackScal& S) {
  return MinState{S.fire_dt, S.fire_alpha, S.fire_npos, S.step, S.prec};
}

// S: the state the force pass evaluated; R2, Pw, G, V: FIRE's sums; E: the
// gradient descent's energy sum.  residual: frms is wanted in any case.
__device__ __forceinline__ MinStep minimiser_step(const FireParams& fp, bool do_fire, int n,
                                                  double inv_2n, const MinState& S, double R2,
                                                  double Pw, double G, double V, double E,
                                                  bool residual) {
#pragma clang fp contract(off)
  MinStep m;
  const bool last = S.step >= (int)fp.max_iter;
  m.dt_old = m.dt = S.dt;
  m.alpha = S.alpha;
  m.npos = S.npos;
  m.c_keep = m.c_force = m.frms = 0.0;
  m.mix = m.end = 0;
  m.prec = S.prec;
  if (do_fire) {
    // Selects, not branches: every step takes this path and waits for it.
    const bool up = Pw >= 0;
    const double root = sqrt(V / G);  // NaN for G = 0, not used then
    const double npos = S.npos + 1;
    const bool grow = npos > fp.n_min;
    const double dt_up = grow ? fmin(S.dt * fp.f_inc, fp.dt_max) : S.dt;
    const double alpha_up = grow ? S.alpha * fp.f_alpha : S.alpha;
    m.mix = up ? 1 : 0;
    m.c_keep = up ? 1.0 - S.alpha : 0.0;
    m.c_force = up && G > 0 ? S.alpha * root : 0.0;
    m.npos = up ? npos : 0.0;
    m.dt = up ? dt_up : S.dt * fp.f_dec;
    m.alpha = up ? alpha_up : fp.alpha0;
    // Convergence is judged on FP64 pair forces only: a packing still on FP32
    // pair math whose residual falls below max(switch_frms, ftol) moves to FP64
    // and keeps iterating.  The root is taken only where F_rms may be below a
    // limit (its square times 3 N, with room for rounding and underflow).
    const bool fp32 = m.prec == kFP32;
    const double lim = fp32 ? fmax(fp.switch_frms, fp.ftol) : fp.ftol;
    if (residual || last || R2 <= lim * lim * (3.0 * n) * (1.0 + 1e-9) + 1e-300) {
      m.frms = sqrt(R2 / (3.0 * n));
      if (!fp32 && m.frms < fp.ftol) m.end = 1;
      else if (last) m.end = 2;
      else if (fp32 && m.frms < lim) m.prec = kFP64;
    }
  } else {
    // gradient-descent passes always record energy: E / (2N)
    if (residual) m.frms = sqrt(R2 / (3.0 * n));
    if (E * inv_2n <= fp.emin || last) m.end = 1;
  }
  return m;
}

// The state after that step.
__device__ __forceinline__ MinState after(const MinState& S, const MinStep& m) {
  return m.end ? S : MinState{m.dt, m.alpha, m.npos, S.step + 1, m.prec};
}

// The scalars after that step (the storing thread).
__device__ __forceinline__ void advance(PackScal& S1, const PackScal& S0, const MinStep& m,
                                        bool do_fire) {
  S1 = S0;
  if (m.end) {
    S1.frms = m.frms;
    S1.converged = m.end;
    S1.iters = S0.step;
    return;
  }
  S1.step = S0.step + 1;
  if (!do_fire) return;
  S1.fire_dt = m.dt;
  S1.fire_alpha = m.alpha;
  S1.fire_npos = m.npos;
  S1.prec = m.prec;
  // read by the update kernel when k_reduce took the decision
  S1.fire_mix = m.mix;
  S1.fire_c_keep = m.c_keep;
  S1.fire_c_force = m.c_force;
  S1.fire_dt_old = m.dt_old;
  S1.fire_dt_new = m.dt;
}

// ---------------------------------------------------------------------------
// block reduction helpers (fixed order -> deterministic)
// ---------------------------------------------------------------------------
// Sum over the wavefront's 64 lanes, valid in lane 63.  Data-parallel-primitive
// moves (rows of 16 lanes, then the row broadcasts) cost VALU issue only; the
// same tree by shuffles is six LDS round trips.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, ROWS, 0xf, false);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1
  v = dpp_add<0x112, 0xf>(v);  // row_shr:2
  v = dpp_add<0x114, 0xf>(v);  // row_shr:4
  v = dpp_add<0x118, 0xf>(v);  // row_shr:8
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Sums over the L lanes (1, 2, 4 or 8, aligned) that share a particle, in all of
// them, as the tree lane ^ 4, ^ 2, ^ 1.  Data-parallel-primitive moves instead
// of shuffles, which are LDS round trips: lanes four apart by row shifts (a
// half row's lower bank takes the upper one's values and the other way), then
// quad permutes.
__device__ __forceinline__ int dpp_xor4(int v) {
  const int up = __builtin_amdgcn_update_dpp(v, v, 0x104, 0xf, 0x5, false);   // row_shl:4
  return __builtin_amdgcn_update_dpp(up, v, 0x114, 0xf, 0xa, false);          // row_shr:4
}
template <int CTRL>
__device__ __forceinline__ int dpp_quad(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}
__device__ __forceinline__ void group_sum(double (&v)[3], int L) {
  auto join = [](int lo, int hi) {
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
  };
  if (L >= 8)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const long long u = __double_as_longlong(v[i]);
      v[i] += join(dpp_xor4((int)u), dpp_xor4((int)(u >> 32)));
    }
  if (L >= 4)  // lanes 2 3 0 1
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const long long u = __double_as_longlong(v[i]);
      v[i] += join(dpp_quad<0x4e>((int)u), dpp_quad<0x4e>((int)(u >> 32)));
    }
  if (L >= 2)  // lanes 1 0 3 2
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const long long u = __double_as_longlong(v[i]);
      v[i] += join(dpp_quad<0xb1>((int)u), dpp_quad<0xb1>((int)(u >> 32)));
    }
}

// The value in lane `lane`, as a scalar.
__device__ __forceinline__ double lane_value(double v, int lane) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)u, lane);
  const int hi = __builtin_amdgcn_readlane((int)(u >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Sum of v over the lanes with this lane's last two bits, valid in lanes 12-15
// of every row of 16.
__device__ __forceinline__ double quad_sum(double v) {
  v = dpp_add<0x114, 0xf>(v);  // row_shr:4
  v = dpp_add<0x118, 0xf>(v);  // row_shr:8
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  return v;
}
// Sums of four values over the wavefront, value i in lanes 12 + i (mod 16): two
// exchanges within quads leave each lane with one value, so the rest is a
// single tree instead of four.
__device__ __forceinline__ double four_sums(double a, double b, double c, double d) {
  auto quad = [](double v, bool two) {
    const long long u = __double_as_longlong(v);
    const int lo = two ? dpp_quad<0x4e>((int)u) : dpp_quad<0xb1>((int)u);
    const int hi = two ? dpp_quad<0x4e>((int)(u >> 32)) : dpp_quad<0xb1>((int)(u >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
  };
  const bool odd = threadIdx.x & 1, high = threadIdx.x & 2;
  const double ab = (odd ? b : a) + quad(odd ? a : b, false);
  const double cd = (odd ? d : c) + quad(odd ? c : d, false);
  return quad_sum((high ? cd : ab) + quad(high ? ab : cd, true));
}

// OR of v over the wavefront, valid in lane 63.
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long dpp_or(unsigned long long v) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWS, 0xf, false);
  return v | ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo;
}
__device__ __forceinline__ unsigned long long wave_or(unsigned long long v) {
  v = dpp_or<0x111, 0xf>(v);
  v = dpp_or<0x112, 0xf>(v);
  v = dpp_or<0x114, 0xf>(v);
  v = dpp_or<0x118, 0xf>(v);
  v = dpp_or<0x142, 0xa>(v);
  return dpp_or<0x143, 0xc>(v);
}

// Sums of v over the workgroup in wavefront order, in s_red[0 .. NV) for every
// thread.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* s_red, int nthr) {
  const int tid = threadIdx.x;
  const int w = tid >> 6, nw = nthr >> 6;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const double x = wave_sum(v[i]);
    if ((tid & 63) == 63) s_red[w * NV + i] = x;
  }
  if (nw > 1) {
    __syncthreads();
    if (tid < NV) {
      double x = 0;
      for (int k = 0; k < nw; ++k) x += s_red[k * NV + tid];
      s_red[tid] = x;  // each slot tid is read (k = 0) before this write by the same thread
    }
  }
  __syncthreads();
}

}  // namespace sc
