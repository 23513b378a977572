// Pair arithmetic of the NBody mobility operator, shared by the gfx950 kernels
// and by the host-side arithmetic self-check (lm_selftest_pair_block_host).
//
// Geometry is in units of the hydrodynamic radius a.  Position records are
// (x, y, z, b): for open boundaries z is the coordinate and b = 1; for the
// bottom wall z is the clamped height max(z, a)/a and b = clamp(z/a, 0, 1) is
// the damping factor of Usabiaga et al. 2017 (App. 1).
//
// The four 3x3 blocks follow solvers/NBody/extra/hydrodynamicKernels.cuh:
//   open RPY       UF :41-57,143-150   WT :63-86,152-159   UT/WF :89-118,161-173
//   wall terms     UF :187-249  WT :253-282  UT :287-319,416-431  WF :324-359
//   damping/clamp  :362-390
// The wall corrections are regrouped into vector form (fewer operations per
// pair than the reference's entry-by-entry 3x3 application):
//   UF: c = f1 v + f2 e (e.v) + f3 v_z e + z^ (f4 (e.v) + f5 v_z)
//   WT: c = g1 v + g2 e (e.v) + g4 p (e_y, -e_x, 0) + z^ g3 (e.v),  p = e_y v_x - e_x v_y
//   WF: c = (k3 e_y (e.v) - (k1 e_z + k4) v_y + (k1 + k2) e_y v_z,
//            (k1 e_z + k4) v_x - k3 e_x (e.v) - (k1 + k2) e_x v_z,  -k1 p)
//   UT: same factors with R' = (-d_x, -d_y, R_z) and h = h_i
// with R = (d_x, d_y, h_i + h_j), e = R/|R|.  The regrouping is exact algebra;
// the CPU oracle (explicit reference matrices) checks it.
#pragma once
#include <hip/hip_runtime.h>

namespace lm {

enum BlockBits : int { kUF = 1, kUT = 2, kWT = 4, kWF = 8 };

template <class R>
struct Vec3 {
  R x, y, z;
};

template <class R>
struct PairAcc {
  Vec3<R> uf, ut, wt, wf;
};

template <class R>
__host__ __device__ inline void acc_zero(PairAcc<R>& a) {
  a.uf = {R(0), R(0), R(0)};
  a.ut = {R(0), R(0), R(0)};
  a.wt = {R(0), R(0), R(0)};
  a.wf = {R(0), R(0), R(0)};
}

// Marks the branch it is placed in as one that stays a branch: an opaque
// statement, so the compiler does not evaluate that branch's arithmetic for
// every lane and select afterwards.  For the self-pair terms (r == 0), which
// are rare: off the diagonal tiles only coincident distinct particles take them.
__host__ __device__ inline void lm_rare_path() { __asm__ __volatile__(""); }

__host__ __device__ inline float lm_rsqrt(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rsqf(x);
#else
  return 1.0f / __builtin_sqrtf(x);
#endif
}
// FP64: hardware estimate refined by one Newton step, y (1 + h/2) with
// h = 1 - x y^2 (relative error 1.5 e0^2 for an estimate error e0).  No
// special-value handling: x = 0 only occurs for self pairs, whose
// coefficients are replaced by the overlap branch.
__host__ __device__ inline double lm_rsqrt(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double y = __builtin_amdgcn_rsq(x);
  const double h = __builtin_fma(-x * y, y, 1.0);
  return __builtin_fma(0.5 * y, h, y);
#else
  return 1.0 / __builtin_sqrt(x);
#endif
}
__host__ __device__ inline float lm_rcp(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcpf(x);
#else
  return 1.0f / x;
#endif
}
// FP64: hardware estimate refined by two Newton steps y (2 - x y) (relative
// error e0^4 for an estimate error e0).  Callers pass finite x > 0.
__host__ __device__ inline double lm_rcp(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  double y = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, y, 1.0);
  y = __builtin_fma(y, e, y);
  e = __builtin_fma(-x, y, 1.0);
  return __builtin_fma(y, e, y);
#else
  return 1.0 / x;
#endif
}
__host__ __device__ inline float lm_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__host__ __device__ inline double lm_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
__host__ __device__ inline float lm_sqrt(float x) { return __builtin_sqrtf(x); }
__host__ __device__ inline double lm_sqrt(double x) { return __builtin_sqrt(x); }

// Open-boundary RPY coefficients for r2 = |d|^2 (scaled units).
//   fuf, guf : f and g/r^2 of M_UF
//   fwt, gwt : f and g/r^2 of M_WT
//   c        : coupling coefficient of U = c (T x d), W = c (F x d)
// Far field (r >= 2) uses rsqrt; the overlap branch (r < 2, including the
// self pair r = 0) is the regularised RPY of hydrodynamicKernels.cuh:51-55,
// :73-84, :97-100.  It is a divergent branch so that waves with no near pair
// skip it.  For r = 0 the far-field values are infinite; they are overwritten
// (never combined) by the overlap branch.
template <class R>
struct RpyCoef {
  R fuf, guf, fwt, gwt, c;
};

// Far-field (r >= 2) coefficients from ir = 1/r.
template <class R, int BLK>
__host__ __device__ inline void rpy_far(R ir, RpyCoef<R>& k) {
  const R ir2 = ir * ir;
  const R ir3 = ir * ir2;
  if (BLK & kUF) {
    k.fuf = ir * (R(0.75) + R(0.5) * ir2);
    k.guf = ir3 * (R(0.75) - R(1.5) * ir2);
  }
  if (BLK & kWT) {
    k.fwt = R(-0.5) * ir3;
    k.gwt = R(1.5) * ir3 * ir2;
  }
  if (BLK & (kUT | kWF)) k.c = ir3;
}

// Overlap (r < 2, including the self pair r = 0) coefficients; r and 1/r come
// from the rsqrt already computed (no sqrt, no division).
template <class R, int BLK>
__host__ __device__ inline void rpy_near(R r2, R ir, RpyCoef<R>& k) {
  const R r = r2 > R(0) ? r2 * ir : R(0);
  const R ir_n = r2 > R(0) ? ir : R(0);
  if (BLK & kUF) {
    k.fuf = R(1) - R(0.28125) * r;
    k.guf = R(0.09375) * ir_n;
  }
  if (BLK & kWT) {
    k.fwt = R(1) - R(0.84375) * r + R(0.078125) * r * r * r;
    k.gwt = r > R(0) ? (R(0.28125) * ir_n - R(0.046875) * r) : R(0);
  }
  if (BLK & (kUT | kWF)) k.c = R(0.5) * (R(1) - R(0.375) * r);
}

// Replace k by the overlap coefficients when r2 < 4, by selects (no branch).
template <class R, int BLK>
__host__ __device__ inline void rpy_near_select(R r2, R ir, RpyCoef<R>& k) {
  RpyCoef<R> n = k;
  rpy_near<R, BLK>(r2, ir, n);
  const bool is_near = r2 < R(4);
  if (BLK & kUF) {
    k.fuf = is_near ? n.fuf : k.fuf;
    k.guf = is_near ? n.guf : k.guf;
  }
  if (BLK & kWT) {
    k.fwt = is_near ? n.fwt : k.fwt;
    k.gwt = is_near ? n.gwt : k.gwt;
  }
  if (BLK & (kUT | kWF)) k.c = is_near ? n.c : k.c;
}

template <class R, int BLK>
__host__ __device__ inline void rpy_coeffs(R r2, R& fuf, R& guf, R& fwt, R& gwt, R& c) {
  const R ir = lm_rsqrt(r2);
  RpyCoef<R> k{};
  rpy_far<R, BLK>(ir, k);
  if (__builtin_expect(r2 < R(4), 0)) {
#if defined(__HIP_DEVICE_COMPILE__)
    // An opaque statement keeps this a branch: speculating it (if-conversion)
    // would put the overlap arithmetic on every pair.
    __asm__ __volatile__("");
#endif
    rpy_near<R, BLK>(r2, ir, k);
  }
  fuf = k.fuf;
  guf = k.guf;
  fwt = k.fwt;
  gwt = k.gwt;
  c = k.c;
}

// Open-boundary UF coefficients times 4/3, so that the far field costs one
// operation less: fuf = 1/r + (2/3)/r^3, guf = 1/r^3 - 2/r^5 (4/3 of
// rpy_far's); the caller scales its sums by 3/4.
template <class R>
__host__ __device__ inline void rpy_far_uf34(R ir, RpyCoef<R>& k) {
  const R ir2 = ir * ir;
  const R ir3 = ir * ir2;
  k.fuf = lm_fma(R(2.0 / 3.0), ir3, ir);
  k.guf = lm_fma(R(-2) * ir2, ir3, ir3);
}

// rpy_near_select for the 4/3-scaled coefficients
template <class R>
__host__ __device__ inline void rpy_near_select_uf34(R r2, R ir, RpyCoef<R>& k) {
  RpyCoef<R> n = k;
  rpy_near<R, kUF>(r2, ir, n);
  const bool is_near = r2 < R(4);
  k.fuf = is_near ? n.fuf * R(4.0 / 3.0) : k.fuf;
  k.guf = is_near ? n.guf * R(4.0 / 3.0) : k.guf;
}

// Open-boundary contribution of one source (f = force, t = torque) to one
// target with given coefficients, added into a (dimensionless; the caller
// applies t0, rt0, r0).
template <class R, int BLK>
__host__ __device__ inline void open_accumulate(R dx, R dy, R dz, R fx, R fy, R fz, R tx, R ty,
                                                R tz, const RpyCoef<R>& k, PairAcc<R>& a) {
  const R fuf = k.fuf, guf = k.guf, fwt = k.fwt, gwt = k.gwt, c = k.c;
  // Accumulate as two FMAs per component: acc = fma(f, v, acc); acc = fma(s, d, acc).
  if (BLK & kUF) {
    const R s = guf * (dx * fx + dy * fy + dz * fz);
    a.uf.x = lm_fma(s, dx, lm_fma(fuf, fx, a.uf.x));
    a.uf.y = lm_fma(s, dy, lm_fma(fuf, fy, a.uf.y));
    a.uf.z = lm_fma(s, dz, lm_fma(fuf, fz, a.uf.z));
  }
  if (BLK & kWT) {
    const R s = gwt * (dx * tx + dy * ty + dz * tz);
    a.wt.x = lm_fma(s, dx, lm_fma(fwt, tx, a.wt.x));
    a.wt.y = lm_fma(s, dy, lm_fma(fwt, ty, a.wt.y));
    a.wt.z = lm_fma(s, dz, lm_fma(fwt, tz, a.wt.z));
  }
  if (BLK & (kUT | kWF)) {  // v x (c d)
    const R cdx = c * dx, cdy = c * dy, cdz = c * dz;
    if (BLK & kUT) {  // c (T x d)
      a.ut.x = lm_fma(ty, cdz, lm_fma(-tz, cdy, a.ut.x));
      a.ut.y = lm_fma(tz, cdx, lm_fma(-tx, cdz, a.ut.y));
      a.ut.z = lm_fma(tx, cdy, lm_fma(-ty, cdx, a.ut.z));
    }
    if (BLK & kWF) {  // c (F x d)
      a.wf.x = lm_fma(fy, cdz, lm_fma(-fz, cdy, a.wf.x));
      a.wf.y = lm_fma(fz, cdx, lm_fma(-fx, cdz, a.wf.y));
      a.wf.z = lm_fma(fx, cdy, lm_fma(-fy, cdx, a.wf.z));
    }
  }
}

template <class R, int BLK>
__host__ __device__ inline void open_pair(R dx, R dy, R dz, R fx, R fy, R fz, R tx, R ty, R tz,
                                          PairAcc<R>& a) {
  const R r2 = dx * dx + dy * dy + dz * dz;
  RpyCoef<R> k{};
  rpy_coeffs<R, BLK>(r2, k.fuf, k.guf, k.fwt, k.gwt, k.c);
  open_accumulate<R, BLK>(dx, dy, dz, fx, fy, fz, tx, ty, tz, k, a);
}

// ---- one pair in symmetric units, and in both directions ----------------------
// Units in which the grand mobility matrix needs no factors between its blocks:
//   U = (3/4) t0 [ UF' F + UT (T / a) ],   W = rt0 [ WF F + WT (T / a) ]
// with UF' = 4/3 UF (t0 = 1/(6 pi eta a), rt0 = 1/(8 pi eta a^2); the angular
// self mobility r0 = rt0 / a).  The damping of the bottom wall multiplies every
// block by b_i b_j, so the caller scales the forces and torques of j by b_j
// and the sums of i by b_i; no pair carries a factor of its own.  U and W of a
// particle are one accumulator each.
//
// Image system of the bottom wall (Swan & Brady, hydrodynamicKernels.cuh:187-359):
// R = (d_x, d_y, h_i + h_j), e = R/|R|, u = 1/|R|^2, q = (e_y, -e_x, 0),
// h = h_j/R_z (h_i/R_z where marked):
//   UF:  M v = f1 v + (f2 (e.v) + f3 v_z) e + z^ (f4 (e.v) + f5 v_z), with t1 = 5 e_z^2 - 1,
//        hq = h (1 - h) e_z^2 and
//        f1 = -(3 (1 + 2 hq) + 2 (1 - 3 e_z^2) u + 2 t1 u^2) / (4 |R|)
//        f2 = -(3 (1 - 6 hq) + 6 t1 u + 10 (1 - 7 e_z^2) u^2) / (4 |R|)
//        f3 = e_z (3 h (1 - 6 (1 - h) e_z^2) + 6 t1 u + 10 (2 - 7 e_z^2) u^2) / (2 |R|)
//        f4 = e_z (3 h - 10 u^2) / (2 |R|)
//        f5 = -(3 h^2 e_z^2 + 3 e_z^2 u + (2 - 15 e_z^2) u^2) / |R|
//   WT:  M v = g1 v + g2 (e.v) e + g3 (e.v) z^ + g4 (q.v) q, with
//        g1 = (1 - 6 e_z^2) u / (2 |R|), g2 = -3 u / (2 |R|), g3 = 3 e_z u / |R|, g4 = 3 u / |R|
//   WF:  B v = q (k3 (e.v) + (k1 + k2) v_z) + kz (z^ x v) - k1 (q.v) z^
//   UT:  C v = k3 (q.v) e - kz (z^ x v) + k1 v_z q + gam (q.v) z^ (h = h_i),
//        gam = -(k1 + k2 + 2 k3 e_z), with k1 = u, k2 = 2 u (6 h e_z^2 + (1 - 10 e_z^2) u),
//        k3 = -2 e_z u (3 h - 5 u), kz = e_z u (1 - 2 h + 2 u).
// Self pairs (r = 0, h_i = h_j) have their own forms (B1-B3, :190-202, :256-261,
// :290-294, :327-331).
//
// The grand mobility matrix is symmetric: blockwise M_ji = M_ij^T, with UF and
// WT transposing into themselves and the cross blocks swapping,
// M_UT(ji) = M_WF(ij)^T and M_WF(ji) = M_UT(ij)^T.  So the coefficients of the
// pair (i <- j) also give what j receives from i:
//   UF^T v = f1 v + (f2 (e.v) + f4 v_z) e + z^ (f3 (e.v) + f5 v_z)   (f3, f4 swap)
//   WT^T v = g1 v + (g2 (e.v) + g3 v_z) e + g4 (q.v) q
//   B^T v = (k3 e + (k1 + k2) z^) (q.v) - kz (z^ x v) - k1 v_z q
//   C^T v = (k3 (e.v) + gam v_z) q + kz (z^ x v) + k1 (q.v) z^
// and the open parts: UF, WT symmetric; c (v x d) transposes to -c (v x d).
// The polynomials in u are evaluated in Horner form and the open part and the
// image terms of a block are merged into one set of coefficients (dot products
// with v = F or T of the other particle, c_v = d_y v_x - d_x v_y = |R| (q.v)):
//   UF:  x, y: A v + (G (d.v) + Q/|R|) d,  z: (A + F5) v_z + G (d.v) d_z + Q e_z + F4 (e.v)
//        with A = fuf + F1, G = guf, Q = F2 (e.v) + F3 v_z; F3 and F4 swap for j.
//   WT:  x: Aw v_x + (Gw (d.v) + G2 (e.v)/|R|) d_x + G4 c_v d_y,  y: ... - G4 c_v d_x,
//        z: Aw v_z + Gw (d.v) d_z + (g2 e_z + g3) (e.v); for j, G2 (e.v) + G3 v_z
//        takes the place of G2 (e.v) and of the z coefficient.
//   WF, UT and their transposes: x, y from (v_y, -v_x) and (d_x, d_y), z from c_v;
//        their d terms join those of UF and WT.  With p = h e_z^2, R3 = 1/|R|^3:
//        K3 = k3/|R| = R3 e_z (10 u - 6 h), K12 = (k1 + k2)/|R| = R3 (1 + u (2 - 20 e_z^2) + 12 p).

// Geometry of a pair: separation d, heights' sum and the inverses.
template <class R>
struct PairGeo {
  R dx, dy, dz, r2, ir, Rz, R2, iR, iRz;
};
template <class R, bool WALL>
__host__ __device__ inline void pair_distances(R xi, R yi, R hi, R xj, R yj, R hj, PairGeo<R>& g) {
  g.dx = xi - xj;
  g.dy = yi - yj;
  g.dz = hi - hj;
  const R xy = lm_fma(g.dy, g.dy, g.dx * g.dx);
  g.r2 = lm_fma(g.dz, g.dz, xy);
  if (WALL) {
    g.Rz = hi + hj;
    g.R2 = lm_fma(g.Rz, g.Rz, xy);
  }
}
template <class R, bool WALL>
__host__ __device__ inline void pair_inverses(PairGeo<R>& g) {
  g.ir = lm_rsqrt(g.r2);
  if (WALL) {
    g.iR = lm_rsqrt(g.R2);
    g.iRz = lm_rcp(g.Rz);
  }
}

// Open coefficients in these units: far field (r >= 2) and overlap.
template <class R, int BLK>
__host__ __device__ inline void rpy_unit_far(R ir, RpyCoef<R>& k) {
  const R ir2 = ir * ir;
  const R ir3 = ir * ir2;
  const R ir5 = ir3 * ir2;
  if (BLK & kUF) {
    k.fuf = lm_fma(R(2.0 / 3.0), ir3, ir);
    k.guf = lm_fma(R(-2), ir5, ir3);
  }
  if (BLK & kWT) {
    k.fwt = R(-0.5) * ir3;
    k.gwt = R(1.5) * ir5;
  }
  if (BLK & (kUT | kWF)) k.c = ir3;
}
template <class R, int BLK>
__host__ __device__ inline void rpy_unit_near(R r2, R ir, RpyCoef<R>& k) {
  rpy_near<R, BLK>(r2, ir, k);
  if (BLK & kUF) {
    k.fuf *= R(4.0 / 3.0);
    k.guf *= R(4.0 / 3.0);
  }
}
// The overlap values where r < 2, by selects.
template <class R, int BLK>
__host__ __device__ inline void rpy_unit_near_select(R r2, R ir, RpyCoef<R>& k) {
  RpyCoef<R> n = k;
  rpy_unit_near<R, BLK>(r2, ir, n);
  const bool is_near = r2 < R(4);
  k.fuf = is_near ? n.fuf : k.fuf;
  k.guf = is_near ? n.guf : k.guf;
  k.fwt = is_near ? n.fwt : k.fwt;
  k.gwt = is_near ? n.gwt : k.gwt;
  k.c = is_near ? n.c : k.c;
}
// Both, the overlap in a branch that stays a branch.
template <class R, int BLK>
__host__ __device__ inline void rpy_unit(R r2, R ir, RpyCoef<R>& k) {
  k = RpyCoef<R>{};
  rpy_unit_far<R, BLK>(ir, k);
  if (__builtin_expect(r2 < R(4), 0)) {
    lm_rare_path();
    rpy_unit_near<R, BLK>(r2, ir, k);
  }
}

// Open boundaries: u, w of i from (Fj, Tj) and (kToJ) su, sw of j from (Fi, Ti).
template <class R, int BLK, bool kToJ>
__host__ __device__ inline void open_unit(R dx, R dy, R dz, const RpyCoef<R>& k, const Vec3<R>& Fj,
                                          const Vec3<R>& Tj, const Vec3<R>& Fi, const Vec3<R>& Ti,
                                          Vec3<R>& u, Vec3<R>& w, Vec3<R>& su, Vec3<R>& sw) {
  if (BLK & kUF) {
    const R s = k.guf * (dx * Fj.x + dy * Fj.y + dz * Fj.z);
    u.x = lm_fma(s, dx, lm_fma(k.fuf, Fj.x, u.x));
    u.y = lm_fma(s, dy, lm_fma(k.fuf, Fj.y, u.y));
    u.z = lm_fma(s, dz, lm_fma(k.fuf, Fj.z, u.z));
    if (kToJ) {
      const R ss = k.guf * (dx * Fi.x + dy * Fi.y + dz * Fi.z);
      su.x = lm_fma(ss, dx, lm_fma(k.fuf, Fi.x, su.x));
      su.y = lm_fma(ss, dy, lm_fma(k.fuf, Fi.y, su.y));
      su.z = lm_fma(ss, dz, lm_fma(k.fuf, Fi.z, su.z));
    }
  }
  if (BLK & kWT) {
    const R s = k.gwt * (dx * Tj.x + dy * Tj.y + dz * Tj.z);
    w.x = lm_fma(s, dx, lm_fma(k.fwt, Tj.x, w.x));
    w.y = lm_fma(s, dy, lm_fma(k.fwt, Tj.y, w.y));
    w.z = lm_fma(s, dz, lm_fma(k.fwt, Tj.z, w.z));
    if (kToJ) {
      const R ss = k.gwt * (dx * Ti.x + dy * Ti.y + dz * Ti.z);
      sw.x = lm_fma(ss, dx, lm_fma(k.fwt, Ti.x, sw.x));
      sw.y = lm_fma(ss, dy, lm_fma(k.fwt, Ti.y, sw.y));
      sw.z = lm_fma(ss, dz, lm_fma(k.fwt, Ti.z, sw.z));
    }
  }
  if (BLK & (kUT | kWF)) {  // v x (c d) to i, -v x (c d) to j
    const R cx = k.c * dx, cy = k.c * dy, cz = k.c * dz;
    if (BLK & kUT) {
      u.x = lm_fma(Tj.y, cz, lm_fma(-Tj.z, cy, u.x));
      u.y = lm_fma(Tj.z, cx, lm_fma(-Tj.x, cz, u.y));
      u.z = lm_fma(Tj.x, cy, lm_fma(-Tj.y, cx, u.z));
      if (kToJ) {
        su.x = lm_fma(-Ti.y, cz, lm_fma(Ti.z, cy, su.x));
        su.y = lm_fma(-Ti.z, cx, lm_fma(Ti.x, cz, su.y));
        su.z = lm_fma(-Ti.x, cy, lm_fma(Ti.y, cx, su.z));
      }
    }
    if (BLK & kWF) {
      w.x = lm_fma(Fj.y, cz, lm_fma(-Fj.z, cy, w.x));
      w.y = lm_fma(Fj.z, cx, lm_fma(-Fj.x, cz, w.y));
      w.z = lm_fma(Fj.x, cy, lm_fma(-Fj.y, cx, w.z));
      if (kToJ) {
        sw.x = lm_fma(-Fi.y, cz, lm_fma(Fi.z, cy, sw.x));
        sw.y = lm_fma(-Fi.z, cx, lm_fma(Fi.x, cz, sw.y));
        sw.z = lm_fma(-Fi.x, cy, lm_fma(Fi.y, cx, sw.z));
      }
    }
  }
}

// The UF image coefficients F1..F5 (4/3 of f1..f5) from hw = h_j/R_z, hu =
// 1 - hw, p = hw e_z^2.
template <class R>
struct WallUF {
  R F1, F2, F3, F4, F5;
};
template <class R>
__host__ __device__ inline WallUF<R> wall_uf_coefs(R hw, R hu, R p, R ez, R ez2, R u, R iR) {
  WallUF<R> w;
  const R hq = hu * p;
  const R tw = hw + hw;
  const R eR = ez * iR;
  w.F1 = iR * lm_fma(u, lm_fma(u, lm_fma(R(-10.0 / 3.0), ez2, R(2.0 / 3.0)),
                               lm_fma(R(2), ez2, R(-2.0 / 3.0))),
                     lm_fma(R(-2), hq, R(-1)));
  w.F2 = iR * lm_fma(u, lm_fma(u, lm_fma(R(70.0 / 3.0), ez2, R(-10.0 / 3.0)),
                               lm_fma(R(-10), ez2, R(2))),
                     lm_fma(R(6), hq, R(-1)));
  w.F3 = eR * lm_fma(u, lm_fma(u, lm_fma(R(-140.0 / 3.0), ez2, R(40.0 / 3.0)),
                               lm_fma(R(20), ez2, R(-4))),
                     lm_fma(R(-12), hq, tw));
  w.F4 = eR * lm_fma(R(-20.0 / 3.0) * u, u, tw);
  w.F5 = iR * lm_fma(u, lm_fma(u, lm_fma(R(20), ez2, R(-8.0 / 3.0)), R(-4) * ez2),
                     R(4) * (hq - p));
  return w;
}

// Bottom wall, r > 0: u, w of i from (Fj, Tj) and (kToJ) su, sw of j from (Fi, Ti).
template <class R, int BLK, bool kToJ>
__host__ __device__ inline void wall_unit(const PairGeo<R>& g, R hj, const RpyCoef<R>& k,
                                          const Vec3<R>& Fj, const Vec3<R>& Tj, const Vec3<R>& Fi,
                                          const Vec3<R>& Ti, Vec3<R>& u, Vec3<R>& w, Vec3<R>& su,
                                          Vec3<R>& sw) {
  constexpr bool kCross = (BLK & (kUT | kWF)) != 0;
  const R dx = g.dx, dy = g.dy, dz = g.dz, iR = g.iR;
  const R U = iR * iR;  // u of the comment above
  const R ez = g.Rz * iR;
  const R ez2 = ez * ez;
  const R hw = hj * g.iRz;
  const R hu = R(1) - hw;
  const R p = hw * ez2;
  const R R3 = U * iR;
  const R R3ez = R3 * ez;
  // projections of the source's force and torque, and of the target's
  const R pF = dx * Fj.x + dy * Fj.y, pFi = kToJ ? dx * Fi.x + dy * Fi.y : R(0);
  const R eF = lm_fma(pF, iR, ez * Fj.z), eFi = kToJ ? lm_fma(pFi, iR, ez * Fi.z) : R(0);
  const R cT = dy * Tj.x - dx * Tj.y, cTi = kToJ ? dy * Ti.x - dx * Ti.y : R(0);
  // factors of d (U) and of d and (d_y, -d_x) (W), summed over the blocks
  R Sd = R(0), Sdj = R(0), Sw = R(0), Swj = R(0), Pw = R(0), Pwj = R(0);
  if (BLK & kUF) {
    const WallUF<R> f = wall_uf_coefs<R>(hw, hu, p, ez, ez2, U, iR);
    const R A = k.fuf + f.F1;
    const R A5 = A + f.F5;
    const R GdF = k.guf * lm_fma(dz, Fj.z, pF);
    const R Q = lm_fma(f.F2, eF, f.F3 * Fj.z);
    Sd = lm_fma(Q, iR, GdF);
    u.x = lm_fma(A, Fj.x, u.x);
    u.y = lm_fma(A, Fj.y, u.y);
    u.z = lm_fma(f.F4, eF, lm_fma(Q, ez, lm_fma(GdF, dz, lm_fma(A5, Fj.z, u.z))));
    if (kToJ) {  // F3 and F4 swap
      const R GdFi = k.guf * lm_fma(dz, Fi.z, pFi);
      const R Qi = lm_fma(f.F2, eFi, f.F4 * Fi.z);
      Sdj = lm_fma(Qi, iR, GdFi);
      su.x = lm_fma(A, Fi.x, su.x);
      su.y = lm_fma(A, Fi.y, su.y);
      su.z = lm_fma(f.F3, eFi, lm_fma(Qi, ez, lm_fma(GdFi, dz, lm_fma(A5, Fi.z, su.z))));
    }
  }
  if (BLK & kWT) {
    const R pT = dx * Tj.x + dy * Tj.y, pTi = kToJ ? dx * Ti.x + dy * Ti.y : R(0);
    const R Aw = lm_fma(R3, lm_fma(R(-3), ez2, R(0.5)), k.fwt);
    const R G2 = R(-1.5) * R3;
    const R G23 = R(1.5) * R3ez;  // g2 e_z + g3
    const R G4 = R(3) * R3 * U;
    const R eT = lm_fma(pT, iR, ez * Tj.z);
    const R GdT = k.gwt * lm_fma(dz, Tj.z, pT);
    Sw = lm_fma(G2 * iR, eT, GdT);
    Pw = G4 * cT;
    w.x = lm_fma(Aw, Tj.x, w.x);
    w.y = lm_fma(Aw, Tj.y, w.y);
    w.z = lm_fma(G23, eT, lm_fma(GdT, dz, lm_fma(Aw, Tj.z, w.z)));
    if (kToJ) {
      const R eTi = lm_fma(pTi, iR, ez * Ti.z);
      const R SS = lm_fma(G2, eTi, (G23 + G23) * Ti.z);
      const R GdTi = k.gwt * lm_fma(dz, Ti.z, pTi);
      Swj = lm_fma(SS, iR, GdTi);
      Pwj = G4 * cTi;
      sw.x = lm_fma(Aw, Ti.x, sw.x);
      sw.y = lm_fma(Aw, Ti.y, sw.y);
      sw.z = lm_fma(SS, ez, lm_fma(GdTi, dz, lm_fma(Aw, Ti.z, sw.z)));
    }
  }
  if (kCross) {
    // suffix w: h = h_j (WF to i, UT to j), suffix u: h = h_i (UT to i, WF to j)
    const R e6 = R(-6) * R3ez, e10 = R(10) * U * R3ez;
    const R K3w = lm_fma(hw, e6, e10), K3u = lm_fma(hu, e6, e10);
    const R t = lm_fma(U, lm_fma(R(-20), ez2, R(2)), R(1));
    const R K12w = R3 * lm_fma(R(12), p, t), K12u = R3 * lm_fma(R(12), ez2 - p, t);
    const R ezu = ez * U;
    const R v = hw - hu;
    const R kzw = ezu * lm_fma(R(2), U, -v), kzu = ezu * lm_fma(R(2), U, v);
    const R c = k.c;
    const R Cz = c - R3;
    const R Cw = lm_fma(c, dz, -kzw), Cu = lm_fma(c, dz, kzu);
    const R KCw = K12w - c;
    const R Zu = lm_fma(-K3u, ez, c - K12u);
    if (BLK & kWF) {
      Pw += lm_fma(K3w, eF, KCw * Fj.z);
      w.x = lm_fma(Fj.y, Cw, w.x);
      w.y = lm_fma(-Fj.x, Cw, w.y);
      w.z = lm_fma(Cz, dy * Fj.x - dx * Fj.y, w.z);
      if (kToJ) {
        Pwj += lm_fma(K3u, eFi, lm_fma(-K3u, ez, Zu) * Fi.z);
        sw.x = lm_fma(-Fi.y, Cu, sw.x);
        sw.y = lm_fma(Fi.x, Cu, sw.y);
        sw.z = lm_fma(-Cz, dy * Fi.x - dx * Fi.y, sw.z);
      }
    }
    if (BLK & kUT) {
      const R n = -Cz * Tj.z;
      Sd = lm_fma(K3u * iR, cT, Sd);
      u.x = lm_fma(dy, n, lm_fma(Tj.y, Cu, u.x));
      u.y = lm_fma(-dx, n, lm_fma(-Tj.x, Cu, u.y));
      u.z = lm_fma(Zu, cT, u.z);
      if (kToJ) {
        const R ni = Cz * Ti.z;
        Sdj = lm_fma(K3w * iR, cTi, Sdj);
        su.x = lm_fma(dy, ni, lm_fma(-Ti.y, Cw, su.x));
        su.y = lm_fma(-dx, ni, lm_fma(Ti.x, Cw, su.y));
        su.z = lm_fma(lm_fma(K3w, ez, KCw), cTi, su.z);
      }
    }
  }
  if (BLK & (kUF | kUT)) {
    u.x = lm_fma(Sd, dx, u.x);
    u.y = lm_fma(Sd, dy, u.y);
    if (kToJ) {
      su.x = lm_fma(Sdj, dx, su.x);
      su.y = lm_fma(Sdj, dy, su.y);
    }
  }
  if (BLK & kWT) {
    w.x = lm_fma(Sw, dx, w.x);
    w.y = lm_fma(Sw, dy, w.y);
    if (kToJ) {
      sw.x = lm_fma(Swj, dx, sw.x);
      sw.y = lm_fma(Swj, dy, sw.y);
    }
  }
  if (BLK & (kWT | kWF)) {
    w.x = lm_fma(Pw, dy, w.x);
    w.y = lm_fma(-Pw, dx, w.y);
    if (kToJ) {
      sw.x = lm_fma(Pwj, dy, sw.x);
      sw.y = lm_fma(-Pwj, dx, sw.y);
    }
  }
}

// Bottom wall, self pair (r = 0, h_i = h_j): Swan & Brady B1-B3 and the open
// self terms; each block equals its transpose's counterpart, so j gets the
// same forms.
template <class R, int BLK, bool kToJ>
__host__ __device__ inline void wall_self_unit(R hj, const Vec3<R>& Fj, const Vec3<R>& Tj,
                                               const Vec3<R>& Fi, const Vec3<R>& Ti, Vec3<R>& u,
                                               Vec3<R>& w, Vec3<R>& su, Vec3<R>& sw) {
  const R ih = R(1) / hj;
  const R ih2 = ih * ih;
  const R ih3 = ih2 * ih;
  if (BLK & kUF) {
    const R ih5 = ih3 * ih2;
    const R cp = R(4.0 / 3.0) * (R(1) - R(0.0625) * (R(9) * ih - R(2) * ih3 + ih5));
    const R cz = R(4.0 / 3.0) * (R(1) - R(0.125) * (R(9) * ih - R(4) * ih3 + ih5));
    u.x += cp * Fj.x;
    u.y += cp * Fj.y;
    u.z += cz * Fj.z;
    if (kToJ) {
      su.x += cp * Fi.x;
      su.y += cp * Fi.y;
      su.z += cz * Fi.z;
    }
  }
  if (BLK & kWT) {
    const R cp = R(1) - R(0.3125) * ih3;
    const R cz = R(1) - R(0.125) * ih3;
    w.x += cp * Tj.x;
    w.y += cp * Tj.y;
    w.z += cz * Tj.z;
    if (kToJ) {
      sw.x += cp * Ti.x;
      sw.y += cp * Ti.y;
      sw.z += cz * Ti.z;
    }
  }
  const R c4 = R(0.125) * ih3 * ih;
  if (BLK & kWF) {  // (-c4 v_y, c4 v_x, 0)
    w.x -= c4 * Fj.y;
    w.y += c4 * Fj.x;
    if (kToJ) {
      sw.x -= c4 * Fi.y;
      sw.y += c4 * Fi.x;
    }
  }
  if (BLK & kUT) {  // (c4 v_y, -c4 v_x, 0)
    u.x += c4 * Tj.y;
    u.y -= c4 * Tj.x;
    if (kToJ) {
      su.x += c4 * Ti.y;
      su.y -= c4 * Ti.x;
    }
  }
}

// One pair, everything after its geometry.
template <class R, bool WALL, int BLK, bool kToJ>
__host__ __device__ inline void pair_unit(const PairGeo<R>& g, R hj, const Vec3<R>& Fj,
                                          const Vec3<R>& Tj, const Vec3<R>& Fi, const Vec3<R>& Ti,
                                          Vec3<R>& u, Vec3<R>& w, Vec3<R>& su, Vec3<R>& sw) {
  RpyCoef<R> k;
  rpy_unit<R, BLK>(g.r2, g.ir, k);
  if constexpr (!WALL) {
    open_unit<R, BLK, kToJ>(g.dx, g.dy, g.dz, k, Fj, Tj, Fi, Ti, u, w, su, sw);
  } else {
    if (g.r2 != R(0)) {
      wall_unit<R, BLK, kToJ>(g, hj, k, Fj, Tj, Fi, Ti, u, w, su, sw);
    } else {
      lm_rare_path();
      wall_self_unit<R, BLK, kToJ>(hj, Fj, Tj, Fi, Ti, u, w, su, sw);
    }
  }
}

// Open boundaries, both directions of every block, in the order of operations
// that plain Lanczos products over open systems keep: the target accumulates
// M_ij [F_j; T_j] into a; the source sums are in units of t0 (su: UF part +
// kut * UT part, kut = rt0/t0) and r0 (sw: WT part + kwf * WF part, kwf = rt0/r0).
template <class R, int BLK>
__host__ __device__ inline void open_both(R dx, R dy, R dz, R fuf, R guf, R fwt, R gwt, R c,
                                          const Vec3<R>& Fj, const Vec3<R>& Tj,
                                          const Vec3<R>& Fi, const Vec3<R>& Ti, R kut, R kwf,
                                          PairAcc<R>& a, Vec3<R>& su, Vec3<R>& sw) {
  if (BLK & kUF) {
    const R s = guf * (dx * Fj.x + dy * Fj.y + dz * Fj.z);
    a.uf.x = lm_fma(s, dx, lm_fma(fuf, Fj.x, a.uf.x));
    a.uf.y = lm_fma(s, dy, lm_fma(fuf, Fj.y, a.uf.y));
    a.uf.z = lm_fma(s, dz, lm_fma(fuf, Fj.z, a.uf.z));
    const R ss = guf * (dx * Fi.x + dy * Fi.y + dz * Fi.z);
    su.x = lm_fma(ss, dx, lm_fma(fuf, Fi.x, su.x));
    su.y = lm_fma(ss, dy, lm_fma(fuf, Fi.y, su.y));
    su.z = lm_fma(ss, dz, lm_fma(fuf, Fi.z, su.z));
  }
  if (BLK & kWT) {
    const R s = gwt * (dx * Tj.x + dy * Tj.y + dz * Tj.z);
    a.wt.x = lm_fma(s, dx, lm_fma(fwt, Tj.x, a.wt.x));
    a.wt.y = lm_fma(s, dy, lm_fma(fwt, Tj.y, a.wt.y));
    a.wt.z = lm_fma(s, dz, lm_fma(fwt, Tj.z, a.wt.z));
    const R ss = gwt * (dx * Ti.x + dy * Ti.y + dz * Ti.z);
    sw.x = lm_fma(ss, dx, lm_fma(fwt, Ti.x, sw.x));
    sw.y = lm_fma(ss, dy, lm_fma(fwt, Ti.y, sw.y));
    sw.z = lm_fma(ss, dz, lm_fma(fwt, Ti.z, sw.z));
  }
  // cross blocks: v x (c d), with the source side's factors -kut, -kwf on
  // the target's own torque and force (fixed over the source loop)
  const R cdx = c * dx, cdy = c * dy, cdz = c * dz;
  if (BLK & kUT) {  // c (T_j x d) to i; -c (T_i x d) to j, in units of t0
    a.ut.x = lm_fma(Tj.y, cdz, lm_fma(-Tj.z, cdy, a.ut.x));
    a.ut.y = lm_fma(Tj.z, cdx, lm_fma(-Tj.x, cdz, a.ut.y));
    a.ut.z = lm_fma(Tj.x, cdy, lm_fma(-Tj.y, cdx, a.ut.z));
    const R kx = -kut * Ti.x, ky = -kut * Ti.y, kz = -kut * Ti.z;
    su.x = lm_fma(ky, cdz, lm_fma(-kz, cdy, su.x));
    su.y = lm_fma(kz, cdx, lm_fma(-kx, cdz, su.y));
    su.z = lm_fma(kx, cdy, lm_fma(-ky, cdx, su.z));
  }
  if (BLK & kWF) {  // c (F_j x d) to i; -c (F_i x d) to j, in units of r0
    a.wf.x = lm_fma(Fj.y, cdz, lm_fma(-Fj.z, cdy, a.wf.x));
    a.wf.y = lm_fma(Fj.z, cdx, lm_fma(-Fj.x, cdz, a.wf.y));
    a.wf.z = lm_fma(Fj.x, cdy, lm_fma(-Fj.y, cdx, a.wf.z));
    const R kx = -kwf * Fi.x, ky = -kwf * Fi.y, kz = -kwf * Fi.z;
    sw.x = lm_fma(ky, cdz, lm_fma(-kz, cdy, sw.x));
    sw.y = lm_fma(kz, cdx, lm_fma(-kx, cdz, sw.y));
    sw.z = lm_fma(kx, cdy, lm_fma(-ky, cdx, sw.z));
  }
}

// One open pair in both directions in that order.
template <class R, int BLK>
__host__ __device__ inline void open_pair_both(R dx, R dy, R dz, const Vec3<R>& Fj,
                                               const Vec3<R>& Tj, const Vec3<R>& Fi,
                                               const Vec3<R>& Ti, R kut, R kwf, PairAcc<R>& a,
                                               Vec3<R>& su, Vec3<R>& sw) {
  constexpr bool kCross = (BLK & (kUT | kWF)) != 0;
  const R r2 = dx * dx + dy * dy + dz * dz;
  R fuf, guf, fwt, gwt, c;
  rpy_coeffs<R, BLK | (kCross ? (kUT | kWF) : 0)>(r2, fuf, guf, fwt, gwt, c);
  open_both<R, BLK>(dx, dy, dz, fuf, guf, fwt, gwt, c, Fj, Tj, Fi, Ti, kut, kwf, a, su, sw);
}

// Dimensionless column of the coupling blocks (units t0, rt0, rt0, r0) of target
// record pi and source record pj (x, y, z, b): velocities of i for the force f
// or the torque t of j.  toJ: what j receives from f or t of i instead.
template <class R, bool WALL, bool toJ>
__host__ __device__ inline void block_column(const R* pi, const R* pj, const Vec3<R>& f,
                                             const Vec3<R>& t, R* out6) {
  constexpr int all = kUF | kUT | kWT | kWF;
  const Vec3<R> zero = {R(0), R(0), R(0)};
  Vec3<R> u = zero, w = zero, su = zero, sw = zero, u2 = zero, w2 = zero, su2 = zero, sw2 = zero;
  PairGeo<R> g;
  pair_distances<R, WALL>(pi[0], pi[1], pi[2], pj[0], pj[1], pj[2], g);
  pair_inverses<R, WALL>(g);
  if (toJ) {
    pair_unit<R, WALL, all, true>(g, pj[2], zero, zero, f, zero, u, w, su, sw);
    pair_unit<R, WALL, all, true>(g, pj[2], zero, zero, zero, t, u2, w2, su2, sw2);
  } else {
    pair_unit<R, WALL, all, true>(g, pj[2], f, zero, zero, zero, su, sw, u, w);
    pair_unit<R, WALL, all, true>(g, pj[2], zero, t, zero, zero, su2, sw2, u2, w2);
  }
  const R b = WALL ? pi[3] * pj[3] : R(1);
  const R q = R(0.75) * b;  // UF' is 4/3 of UF
  out6[0] = q * su.x + b * su2.x;
  out6[1] = q * su.y + b * su2.y;
  out6[2] = q * su.z + b * su2.z;
  out6[3] = b * (sw.x + sw2.x);
  out6[4] = b * (sw.y + sw2.y);
  out6[5] = b * (sw.z + sw2.z);
}

// ---- translational block (UF) split into a per-pair part and a per-vector part
// for products with several force vectors at once, in the units above.  For
// one pair
//   U += a0 F + cd (d.F) d + (e.F) g + F_z h
// holds the open RPY part (a0 = fuf, cd = guf) and, for the wall, the image
// terms: a0 += F1, g = F2 e + F4 z^, h = F3 e + F5 z^; self pairs (r = 0) have
// e = g = 0 and a0 = cp, h = (0, 0, cz - cp).
template <class R>
struct UFCoef {
  R a0, cd, dx, dy, dz, ex, ey, ez, gx, gy, gz, hx, hy, hz;
};

// Open boundaries: coefficients from d and the RPY coefficients (e, g, h unused).
template <class R>
__host__ __device__ inline void uf_apply_open(const UFCoef<R>& k, R fx, R fy, R fz, Vec3<R>& u) {
  const R s = k.cd * (k.dx * fx + k.dy * fy + k.dz * fz);
  u.x = lm_fma(s, k.dx, lm_fma(k.a0, fx, u.x));
  u.y = lm_fma(s, k.dy, lm_fma(k.a0, fy, u.y));
  u.z = lm_fma(s, k.dz, lm_fma(k.a0, fz, u.z));
}

template <class R>
__host__ __device__ inline void uf_apply_wall(const UFCoef<R>& k, R fx, R fy, R fz, Vec3<R>& u) {
  const R s = k.cd * (k.dx * fx + k.dy * fy + k.dz * fz);
  const R ev = k.ex * fx + k.ey * fy + k.ez * fz;
  u.x = lm_fma(fz, k.hx, lm_fma(ev, k.gx, lm_fma(s, k.dx, lm_fma(k.a0, fx, u.x))));
  u.y = lm_fma(fz, k.hy, lm_fma(ev, k.gy, lm_fma(s, k.dy, lm_fma(k.a0, fy, u.y))));
  u.z = lm_fma(fz, k.hz, lm_fma(ev, k.gz, lm_fma(s, k.dz, lm_fma(k.a0, fz, u.z))));
}

// Wall UF coefficients of a target at (xi, yi, hi) and a source at (xj, yj, hj);
// the caller applies the damping b_i b_j.
template <class R>
__host__ __device__ inline void uf_coef_wall(R xi, R yi, R hi, R xj, R yj, R hj, UFCoef<R>& k) {
  PairGeo<R> q;
  pair_distances<R, true>(xi, yi, hi, xj, yj, hj, q);
  pair_inverses<R, true>(q);
  RpyCoef<R> c;
  rpy_unit<R, kUF>(q.r2, q.ir, c);
  k.dx = q.dx;
  k.dy = q.dy;
  k.dz = q.dz;
  k.cd = c.guf;
  if (q.r2 != R(0)) {
    const R ex = q.dx * q.iR, ey = q.dy * q.iR, ez = q.Rz * q.iR;
    const R ez2 = ez * ez;
    const R hw = hj * q.iRz;
    const WallUF<R> f = wall_uf_coefs<R>(hw, R(1) - hw, hw * ez2, ez, ez2, q.iR * q.iR, q.iR);
    k.a0 = c.fuf + f.F1;
    k.ex = ex;
    k.ey = ey;
    k.ez = ez;
    k.gx = f.F2 * ex;
    k.gy = f.F2 * ey;
    k.gz = lm_fma(f.F2, ez, f.F4);
    k.hx = f.F3 * ex;
    k.hy = f.F3 * ey;
    k.hz = lm_fma(f.F3, ez, f.F5);
  } else {
    // self (Swan & Brady B1), as in wall_self_unit
    lm_rare_path();
    const R ih = R(1) / hj;
    const R ih3 = ih * ih * ih;
    const R ih5 = ih3 * ih * ih;
    const R cp = R(4.0 / 3.0) * (R(1) - R(0.0625) * (R(9) * ih - R(2) * ih3 + ih5));
    const R cz = R(4.0 / 3.0) * (R(1) - R(0.125) * (R(9) * ih - R(4) * ih3 + ih5));
    k.a0 = cp;
    k.cd = R(0);
    k.ex = k.ey = k.ez = R(0);
    k.gx = k.gy = k.gz = R(0);
    k.hx = k.hy = R(0);
    k.hz = cz - cp;
  }
}

}  // namespace lm
