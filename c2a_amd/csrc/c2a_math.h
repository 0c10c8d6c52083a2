// c2a_math.h -- FP64 geometry kernels shared by the HIP device code and the
// host-side builder / API layer.
//
// Every routine evaluates its expressions in a fixed order and the whole
// library is compiled with -ffp-contract=off, so host and device produce the
// same bits.  Reference citations name the EwhaGlab/C2A file:line whose
// semantics each routine implements (PQP routines are cited at their C2A
// call sites; PQP itself is not vendored).
#pragma once

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
// Forced inlining: the CCD kernel is one persistent loop, and an outlined
// call in it costs a scratch-resident frame and register save/restore.
#define C2A_HD __host__ __device__ inline __attribute__((always_inline))
#else
#define C2A_HD inline
#endif

namespace c2a {

struct V3 {
  double x[3];
};

C2A_HD double dot3(const double* a, const double* b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }
C2A_HD void sub3(double* r, const double* a, const double* b) {
  r[0] = a[0] - b[0]; r[1] = a[1] - b[1]; r[2] = a[2] - b[2];
}
C2A_HD void add3(double* r, const double* a, const double* b) {
  r[0] = a[0] + b[0]; r[1] = a[1] + b[1]; r[2] = a[2] + b[2];
}
C2A_HD void cross3(double* r, const double* a, const double* b) {
  double r0 = a[1] * b[2] - a[2] * b[1];
  double r1 = a[2] * b[0] - a[0] * b[2];
  double r2 = a[0] * b[1] - a[1] * b[0];
  r[0] = r0; r[1] = r1; r[2] = r2;
}
C2A_HD void neg3(double* r, const double* a) { r[0] = a[0] * -1; r[1] = a[1] * -1; r[2] = a[2] * -1; }
// r = a + b*s
C2A_HD void axpy3(double* r, const double* a, const double* b, double s) {
  r[0] = a[0] + b[0] * s; r[1] = a[1] + b[1] * s; r[2] = a[2] + b[2] * s;
}
C2A_HD double len3(const double* a) { return sqrt(dot3(a, a)); }
C2A_HD double dist2_3(const double* a, const double* b) {
  double d0 = a[0] - b[0], d1 = a[1] - b[1], d2 = a[2] - b[2];
  return d0 * d0 + d1 * d1 + d2 * d2;
}
// multiply by the reciprocal length; no zero guard (a zero vector gives NaN)
C2A_HD void normalize3(double* v) {
  double d = 1.0 / sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  v[0] *= d; v[1] *= d; v[2] *= d;
}
// Matrices are row-major double[9].
C2A_HD void mxv(double* r, const double* M, const double* v) {
  double t0 = M[0] * v[0] + M[1] * v[1] + M[2] * v[2];
  double t1 = M[3] * v[0] + M[4] * v[1] + M[5] * v[2];
  double t2 = M[6] * v[0] + M[7] * v[1] + M[8] * v[2];
  r[0] = t0; r[1] = t1; r[2] = t2;
}
C2A_HD void mtxv(double* r, const double* M, const double* v) {
  double t0 = M[0] * v[0] + M[3] * v[1] + M[6] * v[2];
  double t1 = M[1] * v[0] + M[4] * v[1] + M[7] * v[2];
  double t2 = M[2] * v[0] + M[5] * v[1] + M[8] * v[2];
  r[0] = t0; r[1] = t1; r[2] = t2;
}
C2A_HD void mxvpv(double* r, const double* M, const double* v, const double* w) {
  double t0 = M[0] * v[0] + M[1] * v[1] + M[2] * v[2] + w[0];
  double t1 = M[3] * v[0] + M[4] * v[1] + M[5] * v[2] + w[1];
  double t2 = M[6] * v[0] + M[7] * v[1] + M[8] * v[2] + w[2];
  r[0] = t0; r[1] = t1; r[2] = t2;
}
// R = A B
C2A_HD void mxm(double* R, const double* A, const double* B) {
  double t[9];
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++)
      t[3 * i + j] = A[3 * i + 0] * B[j] + A[3 * i + 1] * B[3 + j] + A[3 * i + 2] * B[6 + j];
  for (int i = 0; i < 9; i++) R[i] = t[i];
}
// R = A^T B
C2A_HD void mtxm(double* R, const double* A, const double* B) {
  double t[9];
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++)
      t[3 * i + j] = A[i] * B[j] + A[3 + i] * B[3 + j] + A[6 + i] * B[6 + j];
  for (int i = 0; i < 9; i++) R[i] = t[i];
}

// ---------------------------------------------------------------------------
// sin/cos of the interpolation angle.  Cody-Waite reduction by pi/2 (three
// 33-bit parts, exact products for |k| < 2^20) and Taylor polynomials on
// |r| <= pi/4 (sin through r^17, cos through r^18; truncation < 1e-19).
// Identical arithmetic on host and device, so poses integrated on the GPU
// match host-side checks bit for bit.
// ---------------------------------------------------------------------------
C2A_HD void sincos_ca(double x, double* s, double* c) {
  double k = rint(x * 0.6366197723675814);
  double r = x - k * 1.5707963267341256;
  r = r - k * 6.077100506303966e-11;
  r = r - k * 2.0222662487959506e-21;
  double r2 = r * r;
  double ps = 2.8114572543455207632e-15;
  ps = ps * r2 + -7.6471637318198164759e-13;
  ps = ps * r2 + 1.6059043836821614599e-10;
  ps = ps * r2 + -2.5052108385441718775e-08;
  ps = ps * r2 + 2.7557319223985890653e-06;
  ps = ps * r2 + -1.9841269841269841270e-04;
  ps = ps * r2 + 8.3333333333333333333e-03;
  ps = ps * r2 + -1.6666666666666666667e-01;
  double sv = r + (r * r2) * ps;
  double pc = 1.5619206968586225796e-16;
  pc = pc * r2 + -4.7794773323873852974e-14;
  pc = pc * r2 + 1.1470745597729724714e-11;
  pc = pc * r2 + -2.0876756987868098979e-09;
  pc = pc * r2 + 2.7557319223985890653e-07;
  pc = pc * r2 + -2.4801587301587301587e-05;
  pc = pc * r2 + 1.3888888888888888889e-03;
  pc = pc * r2 + -4.1666666666666666667e-02;
  double cv = (1.0 - 0.5 * r2) - (r2 * r2) * pc;
  long q = ((long)k) & 3;
  if (q == 0) { *s = sv; *c = cv; }
  else if (q == 1) { *s = cv; *c = -sv; }
  else if (q == 2) { *s = -sv; *c = -cv; }
  else { *s = -cv; *c = sv; }
}

// ---------------------------------------------------------------------------
// Rotation conventions (LinearMath.h): quaternions (x, y, z, w).
// ---------------------------------------------------------------------------
// Matrix3x3::Quaternion_ (LinearMath.h:759-793)
C2A_HD void quat_from_matrix(const double* v, double* q) {
  double trace = v[0] + v[4] + v[8];
  if (trace > 0.0) {
    double s = sqrt(trace + 1.0);
    q[3] = s * 0.5;
    s = 0.5 / s;
    q[0] = (v[7] - v[5]) * s;
    q[1] = (v[2] - v[6]) * s;
    q[2] = (v[3] - v[1]) * s;
  } else {
    int i = v[0] < v[4] ? (v[4] < v[8] ? 2 : 1) : (v[0] < v[8] ? 2 : 0);
    int j = (i + 1) % 3, k = (i + 2) % 3;
    double s = sqrt(v[i * 3 + i] - v[j * 3 + j] - v[k * 3 + k] + 1.0);
    q[i] = s * 0.5;
    s = 0.5 / s;
    q[3] = (v[k * 3 + j] - v[j * 3 + k]) * s;
    q[j] = (v[j * 3 + i] + v[i * 3 + j]) * s;
    q[k] = (v[k * 3 + i] + v[i * 3 + k]) * s;
  }
}
// Matrix3x3::Set_Value(const Quaternion&) (LinearMath.h:809-831)
C2A_HD void matrix_from_quat(const double* q, double* R) {
  double d = q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
  double s = 2.0 / d;
  double xs = q[0] * s, ys = q[1] * s, zs = q[2] * s;
  double wx = q[3] * xs, wy = q[3] * ys, wz = q[3] * zs;
  double xx = q[0] * xs, xy = q[0] * ys, xz = q[0] * zs;
  double yy = q[1] * ys, yz = q[1] * zs, zz = q[2] * zs;
  R[0] = 1.0 - (yy + zz); R[1] = xy - wz; R[2] = xz + wy;
  R[3] = xy + wz; R[4] = 1.0 - (xx + zz); R[5] = yz - wx;
  R[6] = xz - wy; R[7] = yz + wx; R[8] = 1.0 - (xx + yy);
}
// Hamilton product (LinearMath.h:1018-1025)
C2A_HD void quat_mul(const double* a, const double* b, double* r) {
  double x = a[3] * b[0] + a[0] * b[3] + a[1] * b[2] - a[2] * b[1];
  double y = a[3] * b[1] + a[1] * b[3] + a[2] * b[0] - a[0] * b[2];
  double z = a[3] * b[2] + a[2] * b[3] + a[0] * b[1] - a[1] * b[0];
  double w = a[3] * b[3] - a[0] * b[0] - a[1] * b[1] - a[2] * b[2];
  r[0] = x; r[1] = y; r[2] = z; r[3] = w;
}

// Linear motion of one object over t in [0,1] (CInterpMotion_Linear).
struct Motion {
  double R0[9], T0[3];
  double q0[4];
  double cv[3];
  double axis[3];
  double angVel;
  double pad;
  // The axis the motion bounds cross with world-frame directions: `axis`
  // itself (the reference, InterpMotion.cpp:838-845, 784-791) or, in strict
  // mode, the world-frame axis R0 * axis (q(t) = q0 * q_rel(t) turns about
  // the body-frame `axis`, i.e. about R0 * axis in world coordinates).
  double bax[3];
};

// CInterpMotion_Linear ctor + velocity() + LinearAngularVelocity
// (InterpMotion.cpp:148-168, 486-491, 228-270).  Host only (acos).
inline void motion_init(Motion* m, const double* R0, const double* T0, const double* R1,
                        const double* T1, bool strict = false) {
  for (int i = 0; i < 9; i++) m->R0[i] = R0[i];
  for (int i = 0; i < 3; i++) m->T0[i] = T0[i];
  sub3(m->cv, T1, T0);
  double qs[4], qt[4], qc[4], qr[4];
  quat_from_matrix(R0, qs);
  quat_from_matrix(R1, qt);
  for (int i = 0; i < 4; i++) m->q0[i] = qs[i];
  qc[0] = -qs[0]; qc[1] = -qs[1]; qc[2] = -qs[2]; qc[3] = qs[3];
  quat_mul(qc, qt, qr);
  double s = 1 < qr[3] ? 1 : qr[3];
  double sign = s < 0 ? -1 : 1;
  double a = (fabs(s - 1) <= 1e-40 || fabs(s + 1) <= 1e-40)
                 ? (2 * sign)
                 : (sign * acos(2 * s * s - 1) / sqrt(1 - s * s));
  double tg[3] = {a * qr[0], a * qr[1], a * qr[2]};
  m->angVel = len3(tg);
  double len = tg[0] * tg[0] + tg[1] * tg[1] + tg[2] * tg[2];
  if (len < (double)0.00000001f) {
    m->axis[0] = 1.0; m->axis[1] = 0.0; m->axis[2] = 0.0;
  } else {
    double inv = 1.0 / sqrt(len);
    m->axis[0] = tg[0] * inv; m->axis[1] = tg[1] * inv; m->axis[2] = tg[2] * inv;
  }
  m->pad = 0.0;
  if (strict) mxv(m->bax, m->R0, m->axis);
  else for (int i = 0; i < 3; i++) m->bax[i] = m->axis[i];
}

// CInterpMotion_Linear::integrate (InterpMotion.cpp:516-568): pose at t
// (t clamped to 1); q (optional) receives the quaternion (x,y,z,w).
C2A_HD void motion_integrate(const Motion& m, double t, double* R, double* T, double* q_out) {
  double dt = t;
  if (dt > 1) dt = 1;
  T[0] = m.T0[0] + dt * m.cv[0];
  T[1] = m.T0[1] + dt * m.cv[1];
  T[2] = m.T0[2] + dt * m.cv[2];
  double ang = 0.5 * m.angVel * dt;
  double sa, ca;
  sincos_ca(ang, &sa, &ca);
  double drt[4] = {sa * m.axis[0], sa * m.axis[1], sa * m.axis[2], ca};
  double q[4];
  quat_mul(m.q0, drt, q);
  matrix_from_quat(q, R);
  if (q_out) { q_out[0] = q[0]; q_out[1] = q[1]; q_out[2] = q[2]; q_out[3] = q[3]; }
}

// Admissible time a tested leaf pair contributes to mint.  Reference: only
// an improving leaf (dTri <= distance, C2A.cpp:1150) contributes, and a
// touching one (dTri == 0: zero-length normalise, NaN) does not.  Strict:
// every tested leaf contributes, a touching one with 0.
C2A_HD double leaf_time(double dTri, double mleaf, int strict) {
  return (strict && dTri == 0.0) ? 0.0 : mleaf;
}

// computeTOC_MotionBound (InterpMotion.cpp:831-881); N is normalised in place.
C2A_HD double motion_bound(const Motion& m, double angR, double* N) {
  double cr[3];
  normalize3(N);
  cross3(cr, m.bax, N);
  double w = angR * len3(cr) * m.angVel;
  double v = dot3(m.cv, N);
  if (v < 0) v = 0;
  double path = v + w;
  if (path <= 0) path = 1e-30;
  return path;
}

// computeTOC(d, r1, S) leaf bound (InterpMotion.cpp:746-828); S normalised in place.
C2A_HD double motion_bound_leaf(const Motion& m, double angR, double* S) {
  normalize3(S);
  double w, v;
  if (m.angVel == 0) {
    w = 0;
    v = dot3(m.cv, S);
    if (v < 0) v = 0;
  } else {
    double cwc[3] = {m.bax[0] * m.angVel, m.bax[1] * m.angVel, m.bax[2] * m.angVel};
    double cr[3];
    cross3(cr, cwc, S);
    w = angR * len3(cr);
    v = dot3(m.cv, S);
    if (v < 0) v = 0;
  }
  double path = w + v;
  if (path == 0) path = 1e-30;
  return path;
}

// ---------------------------------------------------------------------------
// RSS rectangle distance (C2A_RectDist.h:44-934).  A = [0,a0]x[0,a1] in its
// own frame, B = Tab + Rab*[0,b0]x[0,b1].  Returns the distance and S = Q-P
// (A's frame); S is not written when the rectangles overlap.
// ---------------------------------------------------------------------------
C2A_HD void clampd(double& v, double lo, double hi) {
  if (v < lo) v = lo;
  else if (v > hi) v = hi;
}
// Lumelsky segment parameters (C2A_RectDist.h:81-111)
C2A_HD void seg_params(double& t, double& u, double a, double b, double AB, double AT, double BT) {
  double denom = 1 - AB * AB;
  if (denom == 0) t = 0;
  else {
    t = (AT - BT * AB) / denom;
    clampd(t, 0, a);
  }
  u = t * AB - BT;
  if (u < 0) {
    u = 0;
    t = AT;
    clampd(t, 0, a);
  } else if (u > b) {
    u = b;
    t = u * AB + AT;
    clampd(t, 0, a);
  }
}
// InsideVoronoi (C2A_RectDist.h:123-154), without branches.  The clamps by
// min / max and the two ordered compares decide as the reference's nested
// ifs do, a NaN included (every comparison with it is false).
C2A_HD bool voronoi(double a, double b, double AnB, double AnT, double AB, double AT, double BT) {
  const double u0 = -AnT / AnB;
  const double u = __builtin_fmin(__builtin_fmax(u0, 0.0), b);
  const double t0 = u * AB + AT;
  const double t = __builtin_fmin(__builtin_fmax(t0, 0.0), a);
  const double v = t * AB - BT;
  const bool in = AnB > 0 ? v > (u + 1e-7) : v < (u - 1e-7);
  return in & !(fabs(AnB) < 1e-7) & (u0 == u0) & (t0 == t0);
}

// True when any active lane of the wavefront holds p (host: the lane itself).
C2A_HD bool wave_any(bool p) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __ballot(p) != 0;
#else
  return p;
#endif
}

// One class of the rectangle distance's edge pairs: A's two edges along one
// of its axes against B's two edges along one of its own.  f marks the fixed
// axis of an edge, t the one it runs along.
struct EdgeClass {
  double at, af, bt, bf;       // sides
  double ABtt, ABtf, ABft;     // direction cosines [A axis][B axis]
  double aABff, aABft, bABff, bABtf;   // ... times af (aAB) or bf (bAB)
  double Tat, Taf, Tbt, Tbf;   // Tab on A's axes, Tba on B's
};
// Which of two corner coordinates' tests holds for the reference's lo / hi
// pair: first when x < y, else the second.
C2A_HD bool sel(bool first, bool x, bool y) {
  return (first & x) | (!first & y);
}

// Corner coordinates of a rectangle against the other one's slab [0, m]:
// below 0, above m.
struct Side {
  bool lo, hi;
};
C2A_HD Side side(double x, double m) {
  Side r;
  r.lo = x < 0;
  r.hi = x > m;
  return r;
}

// The winning edge pair of a lane.
struct EdgeWin {
  int w;           // 4 * class + case, -1 none
  double AT, BT;   // segment parameters
};

#if defined(__clang__)   // lane masks are combined without branches on purpose
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wbitwise-instead-of-logical"
#endif
// The four cases of a class in the reference's order: both edges at their
// far side, A's far and B's near, A's near and B's far, both near.  Each lane
// takes its own next case that passes the extent pre-test, so a wavefront
// makes as many turns as its busiest lane has such cases (one or two, mostly)
// instead of one per case, and the two Voronoi tests of a turn run side by
// side.  x1, y1 / z1, w1: A's corners at B's near / far edge order (the
// reference's lo / hi and ulo / uhi), o1 whether x1 < y1; x2 .. o2 the same for B's
// corners.  first: class 0, whose far-far sums the reference associates
// differently.
C2A_HD void edge_class(EdgeWin& g, int cls, const EdgeClass& e, bool o1, Side x1, Side y1, Side z1,
                       Side w1, bool o2, Side x2, Side y2, Side z2, Side w2) {
  bool c0 = sel(o1, w1.hi, z1.hi) & sel(o2, w2.hi, z2.hi);   // uhi1 > bf, uhi2 > af
  bool c1 = sel(o1, z1.lo, w1.lo) & sel(o2, y2.hi, x2.hi);   // ulo1 < 0, hi2 > af
  bool c2 = sel(o1, y1.hi, x1.hi) & sel(o2, z2.lo, w2.lo);   // hi1 > bf, ulo2 < 0
  bool c3 = sel(o1, x1.lo, y1.lo) & sel(o2, x2.lo, y2.lo);   // lo1 < 0, lo2 < 0
  bool open = g.w < 0;
  c0 = c0 & open;
  c1 = c1 & open;
  c2 = c2 & open;
  c3 = c3 & open;
  if (!wave_any(c0 | c1 | c2 | c3)) return;
  const double q1 = e.aABft - e.Tbt, w1v = -e.Tat - e.bABtf;
  const double n1hh = cls == 0 ? e.aABff - e.bf - e.Tbf : e.aABff - e.Tbf - e.bf;
  const double n1hl = e.Tbf - e.aABff, n1lh = -e.Tbf - e.bf;
  const double n2hh = cls == 0 ? e.Taf + e.bABff - e.af : e.Taf - e.af + e.bABff;
  const double n2hl = e.Taf - e.af, n2lh = -e.Taf - e.bABff;
  do {
    const bool p0 = c0, p1 = c1 & !c0, p2 = c2 & !c0 & !c1, p3 = c3 & !c0 & !c1 & !c2;
    const bool ah = p0 | p1, bh = p0 | p2;
    // the far / near shortcuts past a Voronoi test
    const bool s1 = (p0 & sel(o1, z1.hi, w1.hi)) | (p1 & sel(o1, w1.lo, z1.lo)) |
                    (p2 & sel(o1, x1.hi, y1.hi)) | (p3 & sel(o1, y1.lo, x1.lo));
    const bool s2 = (p0 & sel(o2, z2.hi, w2.hi)) | (p1 & sel(o2, x2.hi, y2.hi)) |
                    (p2 & sel(o2, w2.lo, z2.lo)) | (p3 & sel(o2, y2.lo, x2.lo));
    const double AT = ah ? q1 : -e.Tbt, BT = bh ? w1v : -e.Tat;
    const double n1 = ah ? (bh ? n1hh : n1hl) : (bh ? n1lh : e.Tbf);
    const double n2 = ah ? (bh ? n2hh : n2hl) : (bh ? n2lh : -e.Taf);
    const bool v1 = voronoi(e.bt, e.at, bh ? e.ABtf : -e.ABtf, n1, e.ABtt, AT, BT);
    const bool v2 = voronoi(e.at, e.bt, ah ? e.ABft : -e.ABft, n2, e.ABtt, -BT, -AT);
    const bool ok = (p0 | p1 | p2 | p3) & (s1 | v1) & (s2 | v2);
    if (ok) {
      g.w = 4 * cls + (ah ? 0 : 2) + (bh ? 0 : 1);
      g.AT = -BT;
      g.BT = -AT;
    }
    c0 = false;
    c1 = c1 & !p1 & !ok;
    c2 = c2 & !p2 & !ok;
    c3 = c3 & !p3 & !ok;
  } while (wave_any(c1 | c2 | c3));
}
#if defined(__clang__)
#pragma clang diagnostic pop
#endif

// The 16 edge-pair cases are decided in the reference's order; the first one
// whose extent pre-test and two Voronoi tests hold gives the closest points.
// All pre-tests come from 40 comparisons of corner coordinates, kept as lane
// masks.  What bounds it is the instruction stream of the one wavefront per
// SIMD (FP64 divisions above all): 64 random pairs of a knot pair take 6,400
// cycles on MI355X; trying the 16 cases one after another for the whole
// wavefront took 15,300.
C2A_HD double rect_dist(const double* Rab, const double* Tab, const double* a, const double* b,
                        double* S) {
  const double AB00 = Rab[0], AB01 = Rab[1], AB10 = Rab[3], AB11 = Rab[4];
  const double aAB00 = a[0] * AB00, aAB01 = a[0] * AB01;
  const double aAB10 = a[1] * AB10, aAB11 = a[1] * AB11;
  const double bAB00 = b[0] * AB00, bAB10 = b[0] * AB10;
  const double bAB01 = b[1] * AB01, bAB11 = b[1] * AB11;
  double Tba[3];
  mtxv(Tba, Rab, Tab);
  // corner coordinates of A in B's frame and of B in A's frame
  const double ALLx = -Tba[0];
  const double ALUx = ALLx + aAB10;
  const double AULx = ALLx + aAB00;
  const double AUUx = ALUx + aAB00;
  const double BLLx = Tab[0];
  const double BLUx = BLLx + bAB01;
  const double BULx = BLLx + bAB00;
  const double BUUx = BLUx + bAB00;
  const double ALLy = -Tba[1];
  const double ALUy = ALLy + aAB11;
  const double AULy = ALLy + aAB01;
  const double AUUy = ALUy + aAB01;
  const double BLLy = Tab[1];
  const double BLUy = BLLy + bAB11;
  const double BULy = BLLy + bAB10;
  const double BUUy = BLUy + bAB10;

  EdgeWin g;
  g.w = -1;
  g.AT = g.BT = 0.0;
  {
    const Side all = side(ALLx, b[0]), alu = side(ALUx, b[0]), aul = side(AULx, b[0]),
               auu = side(AUUx, b[0]);
    const Side ally = side(ALLy, b[1]), aluy = side(ALUy, b[1]), auly = side(AULy, b[1]),
               auuy = side(AUUy, b[1]);
    const Side bll = side(BLLx, a[0]), blu = side(BLUx, a[0]), bul = side(BULx, a[0]),
               buu = side(BUUx, a[0]);
    const Side blly = side(BLLy, a[1]), bluy = side(BLUy, a[1]), buly = side(BULy, a[1]),
               buuy = side(BUUy, a[1]);
    // A's 1-axis edges against B's 1-axis, then 0-axis edges; A's 0-axis edges likewise
    const EdgeClass e0 = {a[1], a[0], b[1], b[0], AB11, AB10, AB01, aAB00, aAB01,
                          bAB00, bAB10, Tab[1], Tab[0], Tba[1], Tba[0]};
    edge_class(g, 0, e0, ALLx < ALUx, all, alu, aul, auu, BLLx < BLUx, bll, blu, bul, buu);
    const EdgeClass e1 = {a[1], a[0], b[0], b[1], AB10, AB11, AB00, aAB01, aAB00,
                          bAB01, bAB11, Tab[1], Tab[0], Tba[0], Tba[1]};
    edge_class(g, 1, e1, ALLy < ALUy, ally, aluy, auly, auuy, BLLx < BULx, bll, bul, blu, buu);
    const EdgeClass e2 = {a[0], a[1], b[1], b[0], AB01, AB00, AB11, aAB10, aAB11,
                          bAB10, bAB00, Tab[0], Tab[1], Tba[1], Tba[0]};
    edge_class(g, 2, e2, ALLx < AULx, all, aul, alu, auu, BLLy < BLUy, blly, bluy, buly, buuy);
    const EdgeClass e3 = {a[0], a[1], b[0], b[1], AB00, AB01, AB10, aAB11, aAB10,
                          bAB11, bAB01, Tab[0], Tab[1], Tba[0], Tba[1]};
    edge_class(g, 3, e3, ALLy < AULy, ally, auly, aluy, auuy, BLLy < BULy, blly, buly, bluy, buuy);
  }
  if (g.w >= 0) {
    // P on A's edge, Q = Tab + (B's fixed side) + (B's edge) * u
    const bool a1 = g.w < 8, b1 = (g.w & 4) == 0;   // the edges run along the 1-axes
    const bool ah = (g.w & 2) == 0, bh = (g.w & 1) == 0;
    double t, u;
    seg_params(t, u, a1 ? a[1] : a[0], b1 ? b[1] : b[0],
               a1 ? (b1 ? AB11 : AB10) : (b1 ? AB01 : AB00), g.AT, g.BT);
    const double lf = b1 ? b[0] : b[1], p = ah ? (a1 ? a[0] : a[1]) : 0.0;
    double Q[3];
    for (int i = 0; i < 3; i++) {
      const double cv = b1 ? Rab[3 * i + 1] : Rab[3 * i], cf = b1 ? Rab[3 * i] : Rab[3 * i + 1];
      Q[i] = (bh ? Tab[i] + cf * lf : Tab[i]) + cv * u;
    }
    S[0] = Q[0] - (a1 ? p : t);
    S[1] = Q[1] - (a1 ? t : p);
    S[2] = Q[2] - 0;
    return sqrt(dot3(S, S));
  }

  // face-normal separation (C2A_RectDist.h:855-933)
  double sep1, sep2;
  if (Tab[2] > 0.0) {
    sep1 = Tab[2];
    if (Rab[6] < 0.0) sep1 += b[0] * Rab[6];
    if (Rab[7] < 0.0) sep1 += b[1] * Rab[7];
  } else {
    sep1 = -Tab[2];
    if (Rab[6] > 0.0) sep1 -= b[0] * Rab[6];
    if (Rab[7] > 0.0) sep1 -= b[1] * Rab[7];
  }
  if (Tba[2] < 0) {
    sep2 = -Tba[2];
    if (Rab[2] < 0.0) sep2 += a[0] * Rab[2];
    if (Rab[5] < 0.0) sep2 += a[1] * Rab[5];
  } else {
    sep2 = Tba[2];
    if (Rab[2] > 0.0) sep2 -= a[0] * Rab[2];
    if (Rab[5] > 0.0) sep2 -= a[1] * Rab[5];
  }
  if (sep1 >= sep2 && sep1 >= 0) {
    S[0] = 0.0 - 0.0;
    S[1] = 0.0 - 0.0;
    S[2] = ((Tab[2] > 0.0) ? sep1 : -sep1) - 0.0;
  }
  if (sep2 >= sep1 && sep2 >= 0) {
    double P[3];
    if (Tba[2] < 0) {
      P[0] = Rab[2] * sep2 + Tab[0];
      P[1] = Rab[5] * sep2 + Tab[1];
      P[2] = Rab[8] * sep2 + Tab[2];
    } else {
      P[0] = -Rab[2] * sep2 + Tab[0];
      P[1] = -Rab[5] * sep2 + Tab[1];
      P[2] = -Rab[8] * sep2 + Tab[2];
    }
    S[0] = Tab[0] - P[0]; S[1] = Tab[1] - P[1]; S[2] = Tab[2] - P[2];
  }
  double sep = (sep1 > sep2 ? sep1 : sep2);
  return (sep > 0 ? sep : 0);
}

// ---------------------------------------------------------------------------
// Triangle-triangle distance (C2A.cpp:59-405 restating PQP TriDist).
// Feature codes: type 0 vertex, 1 edge, 2 face; -1 unset.
// ---------------------------------------------------------------------------
C2A_HD void seg_points(double* VEC, double* X, double* Y, const double* P, const double* A,
                       const double* Q, const double* B) {
  double T[3], TMP[3];
  sub3(T, Q, P);
  double AA = dot3(A, A), BB = dot3(B, B), AB = dot3(A, B);
  double AT = dot3(A, T), BT = dot3(B, T);
  double denom = AA * BB - AB * AB;
  double t = (AT * BB - BT * AB) / denom;
  if ((t < 0) || isnan(t)) t = 0;
  else if (t > 1) t = 1;
  double u = (t * AB - BT) / BB;
  if ((u <= 0) || isnan(u)) {
    Y[0] = Q[0]; Y[1] = Q[1]; Y[2] = Q[2];
    t = AT / AA;
    if ((t <= 0) || isnan(t)) {
      X[0] = P[0]; X[1] = P[1]; X[2] = P[2];
      sub3(VEC, Q, P);
    } else if (t >= 1) {
      add3(X, P, A);
      sub3(VEC, Q, X);
    } else {
      axpy3(X, P, A, t);
      cross3(TMP, T, A);
      cross3(VEC, A, TMP);
    }
  } else if (u >= 1) {
    add3(Y, Q, B);
    t = (AB + AT) / AA;
    if ((t <= 0) || isnan(t)) {
      X[0] = P[0]; X[1] = P[1]; X[2] = P[2];
      sub3(VEC, Y, P);
    } else if (t >= 1) {
      add3(X, P, A);
      sub3(VEC, Y, X);
    } else {
      axpy3(X, P, A, t);
      sub3(T, Y, P);
      cross3(TMP, T, A);
      cross3(VEC, A, TMP);
    }
  } else {
    axpy3(Y, Q, B, u);
    if ((t <= 0) || isnan(t)) {
      X[0] = P[0]; X[1] = P[1]; X[2] = P[2];
      cross3(TMP, T, B);
      cross3(VEC, B, TMP);
    } else if (t >= 1) {
      add3(X, P, A);
      sub3(T, Q, X);
      cross3(TMP, T, B);
      cross3(VEC, B, TMP);
    } else {
      axpy3(X, P, A, t);
      cross3(VEC, A, B);
      if (dot3(VEC, T) < 0) { VEC[0] = VEC[0] * -1; VEC[1] = VEC[1] * -1; VEC[2] = VEC[2] * -1; }
    }
  }
}

// vertex of triangle `tt` closest to the face of `ts` (or -1)
C2A_HD int tri_vertex_face(const double* ts, const double* sv, const double* tt, double* Nrm,
                           double& Nl, double* proj, int& disjoint) {
  double V[3], Z[3];
  cross3(Nrm, sv + 0, sv + 3);
  Nl = dot3(Nrm, Nrm);
  if (!(Nl > 1e-15)) return -1;
  sub3(V, ts, tt + 0); proj[0] = dot3(V, Nrm);
  sub3(V, ts, tt + 3); proj[1] = dot3(V, Nrm);
  sub3(V, ts, tt + 6); proj[2] = dot3(V, Nrm);
  int point = -1;
  if ((proj[0] > 0) && (proj[1] > 0) && (proj[2] > 0)) {
    point = (proj[0] < proj[1]) ? 0 : 1;
    if (proj[2] < proj[point]) point = 2;
  } else if ((proj[0] < 0) && (proj[1] < 0) && (proj[2] < 0)) {
    point = (proj[0] > proj[1]) ? 0 : 1;
    if (proj[2] > proj[point]) point = 2;
  }
  if (point < 0) return -1;
  disjoint = 1;
  for (int e = 0; e < 3; e++) {
    sub3(V, tt + 3 * point, ts + 3 * e);
    cross3(Z, Nrm, sv + 3 * e);
    if (!(dot3(V, Z) > 0)) return -1;
  }
  return point;
}

// S, T: 3 vertices each (9 doubles).  P, Q: closest points.
C2A_HD double tri_dist(double* P, double* Q, const double* S, const double* T, int* feat) {
  double Sv[9], Tv[9], VEC[3], V[3], Z[3], minP[3], minQ[3];
  int ta = -1, fa = -1, tb = -1, fb = -1;
  sub3(Sv + 0, S + 3, S + 0); sub3(Sv + 3, S + 6, S + 3); sub3(Sv + 6, S + 0, S + 6);
  sub3(Tv + 0, T + 3, T + 0); sub3(Tv + 3, T + 6, T + 3); sub3(Tv + 6, T + 0, T + 6);
  int shown_disjoint = 0;
  double mindd = dist2_3(S, T) + 1;
  double result = -1;
  bool done = false;
  for (int i = 0; i < 3 && !done; i++) {
    for (int j = 0; j < 3; j++) {
      seg_points(VEC, P, Q, S + 3 * i, Sv + 3 * i, T + 3 * j, Tv + 3 * j);
      sub3(V, Q, P);
      double dd = dot3(V, V);
      if (dd <= mindd) {
        minP[0] = P[0]; minP[1] = P[1]; minP[2] = P[2];
        minQ[0] = Q[0]; minQ[1] = Q[1]; minQ[2] = Q[2];
        mindd = dd;
        ta = 1; fa = i; tb = 1; fb = j;
        sub3(Z, S + 3 * ((i + 2) % 3), P);
        double a = dot3(Z, VEC);
        sub3(Z, T + 3 * ((j + 2) % 3), Q);
        double b = dot3(Z, VEC);
        if ((a <= 0) && (b >= 0)) { result = sqrt(dd); done = true; break; }
        double p = dot3(V, VEC);
        if (a < 0) a = 0;
        if (b > 0) b = 0;
        if ((p - a + b) > 0) shown_disjoint = 1;
      }
    }
  }
  if (!done) {
    double Nrm[3], Nl, proj[3];
    int pt = tri_vertex_face(S, Sv, T, Nrm, Nl, proj, shown_disjoint);
    if (pt >= 0) {
      ta = 2; fa = -1; tb = 0; fb = pt;
      axpy3(P, T + 3 * pt, Nrm, proj[pt] / Nl);
      Q[0] = T[3 * pt]; Q[1] = T[3 * pt + 1]; Q[2] = T[3 * pt + 2];
      result = sqrt(dist2_3(P, Q));
    } else {
      pt = tri_vertex_face(T, Tv, S, Nrm, Nl, proj, shown_disjoint);
      if (pt >= 0) {
        ta = 0; fa = pt; tb = 2; fb = -1;
        P[0] = S[3 * pt]; P[1] = S[3 * pt + 1]; P[2] = S[3 * pt + 2];
        axpy3(Q, S + 3 * pt, Nrm, proj[pt] / Nl);
        result = sqrt(dist2_3(P, Q));
      } else if (shown_disjoint) {
        P[0] = minP[0]; P[1] = minP[1]; P[2] = minP[2];
        Q[0] = minQ[0]; Q[1] = minQ[1]; Q[2] = minQ[2];
        result = sqrt(mindd);
      } else {
        result = 0;
      }
    }
  }
  if (feat) { feat[0] = ta; feat[1] = fa; feat[2] = tb; feat[3] = fb; }
  return result;
}

// C2A_TriDistance: triangle 2 mapped into model 1's frame by (R, T)
C2A_HD double tri_distance(const double* R, const double* T, const double* t1, const double* t2,
                           double* p, double* q, int* feat) {
  double b[9];
  mxvpv(b + 0, R, t2 + 0, T);
  mxvpv(b + 3, R, t2 + 3, T);
  mxvpv(b + 6, R, t2 + 6, T);
  return tri_dist(p, q, t1, b, feat);
}

// PQP's TriContact (declared at C2A_PQP.cpp:441, called by CollideRecurse
// :831; PQP itself is not vendored): the separating-axis test over the two
// face normals, the nine edge-edge cross products and the six in-plane edge
// normals, vertices taken relative to P1.  1 when the projections overlap
// on every axis (touching counts as contact).
C2A_HD bool project6(const double* ax, const double* p1, const double* p2, const double* p3,
                     const double* q1, const double* q2, const double* q3) {
  const double P1 = dot3(ax, p1), P2 = dot3(ax, p2), P3 = dot3(ax, p3);
  const double Q1 = dot3(ax, q1), Q2 = dot3(ax, q2), Q3 = dot3(ax, q3);
  double mx1 = P1 > P2 ? P1 : P2, mn1 = P1 < P2 ? P1 : P2;
  mx1 = mx1 > P3 ? mx1 : P3;
  mn1 = mn1 < P3 ? mn1 : P3;
  double mx2 = Q1 > Q2 ? Q1 : Q2, mn2 = Q1 < Q2 ? Q1 : Q2;
  mx2 = mx2 > Q3 ? mx2 : Q3;
  mn2 = mn2 < Q3 ? mn2 : Q3;
  return !(mn1 > mx2) && !(mn2 > mx1);
}

C2A_HD bool tri_contact(const double* P1, const double* P2, const double* P3, const double* Q1,
                        const double* Q2, const double* Q3) {
  const double p1[3] = {0.0, 0.0, 0.0};
  double p2[3], p3[3], q1[3], q2[3], q3[3];
  double e[3][3], f[3][3], n1[3], m1[3], g[3][3], h[3][3], ef[3];
  sub3(p2, P2, P1);
  sub3(p3, P3, P1);
  sub3(q1, Q1, P1);
  sub3(q2, Q2, P1);
  sub3(q3, Q3, P1);
  sub3(e[0], p2, p1);
  sub3(e[1], p3, p2);
  sub3(e[2], p1, p3);
  sub3(f[0], q2, q1);
  sub3(f[1], q3, q2);
  sub3(f[2], q1, q3);
  cross3(n1, e[0], e[1]);
  cross3(m1, f[0], f[1]);
  for (int i = 0; i < 3; i++) {
    cross3(g[i], e[i], n1);
    cross3(h[i], f[i], m1);
  }
  if (!project6(n1, p1, p2, p3, q1, q2, q3)) return false;
  if (!project6(m1, p1, p2, p3, q1, q2, q3)) return false;
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) {
      cross3(ef, e[i], f[j]);
      if (!project6(ef, p1, p2, p3, q1, q2, q3)) return false;
    }
  for (int i = 0; i < 3; i++) {
    if (!project6(g[i], p1, p2, p3, q1, q2, q3)) return false;
    if (!project6(h[i], p1, p2, p3, q1, q2, q3)) return false;
  }
  return true;
}

}  // namespace c2a
