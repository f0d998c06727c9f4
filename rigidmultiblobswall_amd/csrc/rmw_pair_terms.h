// Pair terms of the wall-corrected RPY blob mobility (Rotne-Prager-Yamakawa
// tensor plus the Swan-Brady single-wall image correction), written once as
// host/device templates over the real type T (float or double).
//
// Reference math: mobility/mobility_numba.py
//   UF  :200-276  (RPY :209-234, wall :241-276)
//   UT  :614-679  (wall in the transposed source/target role, :646-679)
//   WF  :1004-1065
//   WT  :1256-1321
//
// The reference forms the 3x3 block M_ij element by element and multiplies
// it by the source vector.  Here each block is decomposed into a few scalar
// coefficients times dyads built from d = r_i - r_j, the image vector
// R = (d_x, d_y, z_i + z_j) and z-hat, so that the product M_ij v costs
// ~16-20 operations per right-hand side and the geometry part is shared by
// k right-hand sides and by the four blocks of the grand mobility:
//
//   UF v = (A + f1) v + Bc (d.v) d + [f2 (e.v) + f3 v_z] e + [f4 (e.v) + f5 v_z] z
//   WF v = c (v x d) - [F1 (v x e) + (F2 v_z + F3 (e.v)) (z x e) + F4 (v x z)]
//   UT v = c (v x d) - [F1 (e' x v) + (F2 z + F3 e') ((z x e').v) + F4 (z x v)]
//   WT v = (A + G1) v + Bc (d.v) d + G2 (e.v) e + G3 (e.v) z + G4 ((z x e).v)(z x e)
//
// with e = R/|R| and e' = (-R_x, -R_y, R_z)/|R| (UT's image seen from the
// source).  All lengths are in units of the blob radius a; the 1/(8 pi eta
// a^p) normalisations are folded into the source vectors by the caller.
// Self pairs (i == j in the central box) are handled by the caller.
#pragma once

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define RMW_HD __host__ __device__ __forceinline__
#else
#include <cmath>
#define RMW_HD inline
#endif

namespace rmw {

template <typename T> struct Vec3 { T x, y, z; };

// Boundary of the fluid (the `domain` options of the reference):
//   wall          RPY + Swan-Brady image (mobility_numba.py:123-287, ...)
//   no wall       RPY alone (:12-120, 440-545, 832-936, 1077-1186)
//   in plane      the wall blocks projected on x-y, P M P with
//                 P = diag(1, 1, 0) (:291-437, 690-830); the caller
//                 projects sources and outputs
//   free surface  RPY(d) + RPY(R) D, D = diag(1, 1, -1) (:1770-1938); UF only
enum : int { kDomWall = 0, kDomNoWall = 1, kDomInPlane = 2, kDomFreeSurface = 3 };
RMW_HD bool dom_has_wall(int dom) { return dom == kDomWall || dom == kDomInPlane; }

// Reciprocal square root.  FP32 on the device uses the hardware v_rsq_f32
// (about 1 ulp).  FP64 on the device refines the hardware estimate v_rsq_f64
// (relative error eps <= 5.3e-8 = 2^-24.2, measured on gfx950 over 4M
// arguments in [1e-7, 1e7]) by one third-order step of Newton's iteration
// for y^-2 = x: with e = 1 - x y^2, x^-1/2 = y (1 - e)^-1/2
// = y (1 + e/2 + 3 e^2/8 + O(e^3)), so the error falls to ~(5/16) eps^3
// plus the rounding of the step (measured: <= 1.39e-16 relative, against
// 1.66e-16 for 1/sqrt(x) with both operations rounded) in 5 FP64 operations
// instead of the ~25 of a correctly rounded sqrt and division.
RMW_HD float rsq(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rsqf(x);
#else
  return 1.0f / std::sqrt(x);
#endif
}
RMW_HD double rsq(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-(x * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
#else
  return 1.0 / std::sqrt(x);
#endif
}

RMW_HD float rcp(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcpf(x);
#else
  return 1.0f / x;
#endif
}
RMW_HD double rcp(double x) { return 1.0 / x; }

// Fused multiply-add a*b + c (single rounding on the device and the host).
RMW_HD float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
RMW_HD double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }

// The smaller of x and a constant; a NaN x gives the constant.
RMW_HD float min_(float x, float c) { return __builtin_fminf(x, c); }
RMW_HD double min_(double x, double c) { return __builtin_fmin(x, c); }

// min(|d|, 2).  Blobs at one point and non-finite positions (|d| = NaN) must give
// non-finite results in every block: FP32 keeps the NaN here (gfx950 has such a
// minimum, at the price of the other), FP64 adds it where no other factor has it
// (nan_of, an FMA; a minimum that keeps it would be a compare and selects).
RMW_HD float clamp_2(float r)
{
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_elementwise_minimum(r, 2.0f);
#else
  return r > 2.0f ? 2.0f : r;
#endif
}
RMW_HD double clamp_2(double r) { return min_(r, 2.0); }
RMW_HD float nan_of(float, float c) { return c; }
RMW_HD double nan_of(double r, double c) { return __builtin_fma(0.0, r, c); }

// ---------------------------------------------------------------------------
// Shared geometry of one (target, source) pair.
// ---------------------------------------------------------------------------
template <typename T> struct Geom {
  T dx, dy, dz;   // d = r_i - r_j (units of a)
  T Rz;           // z_i + z_j
  T r2, invr, r;  // |d|^2, 1/|d|, |d|
  T ic, rm;       // min(1/|d|, 1/2) and min(|d|, 2): see "overlapping blobs"
  T invR;         // 1/|R|
};

// Overlapping blobs.  Every RPY coefficient has a far form (|d| > 2) and an
// overlap form that meet at |d| = 2.  Instead of evaluating both and
// selecting, the far form is taken at |d| clamped from below at 2 (through
// ic = min(1/|d|, 1/2)) and the overlap form's difference from its value at
// 2 is added through rm = min(|d|, 2).  The constants are chosen so that the
// added polynomial is exactly 0 in binary arithmetic at rm = 2, so far pairs
// get the far form bit for bit.  On gfx950 a compare and each select take
// two issue cycles against one for an FMA: the two minima replace three
// compares and five selects of the four blocks (UF 2 selects and 1 compare).

template <typename T>
RMW_HD Geom<T> make_geom(T dx, T dy, T dz, T zi, T zj)
{
  Geom<T> g;
  g.dx = dx; g.dy = dy; g.dz = dz;
  g.Rz = zi + zj;
  T p2 = dx * dx + dy * dy;
  g.r2 = p2 + dz * dz;
  g.invr = rsq(g.r2);
  g.r = g.r2 * g.invr;
  g.ic = min_(g.invr, T(0.5));
  g.rm = clamp_2(g.r);
  T R2 = p2 + g.Rz * g.Rz;
  g.invR = rsq(R2);
  return g;
}

// make_geom of a pair that may not be taken (on = false): then 1/|d| =
// 1/|R| = 0 and |d| = 3 (the far-field branches), which makes every
// coefficient of every block and boundary exactly zero, so the pair adds +-0
// to both of its blobs without a select per output.  d and the heights must
// be finite; a taken pair gets the same values as make_geom.
template <typename T>
RMW_HD Geom<T> make_geom_on(T dx, T dy, T dz, T zi, T zj, bool on)
{
  Geom<T> g;
  g.dx = dx; g.dy = dy; g.dz = dz;
  g.Rz = zi + zj;
  T p2 = dx * dx + dy * dy;
  g.r2 = p2 + dz * dz;
  const T ir = rsq(g.r2);
  g.invr = on ? ir : T(0);
  g.r = on ? g.r2 * ir : T(3);
  g.ic = min_(g.invr, T(0.5));
  g.rm = clamp_2(g.r);
  T R2 = p2 + g.Rz * g.Rz;
  const T iR = rsq(R2);
  g.invR = on ? iR : T(0);
  return g;
}

// ---------------------------------------------------------------------------
// UF: translation from force.   mobility_numba.py:209-276
// ---------------------------------------------------------------------------
template <typename T> struct CoefUF {
  T s;      // A + f1 (coefficient of v)
  T s5;     // s + f5 (coefficient of v_z in the z row)
  T Bc;     // coefficient of (d.v) d
  T g2;     // f2 / |R|^2  -> coefficient of (R.v) R
  T g3;     // f3 / |R|    -> coefficient of v_z R
  T g4;     // f4 / |R|    -> coefficient of (R.v) z
};

// RPY translational coefficients A I + B r r^T (units of a):
//   far      A = (1 + 2/(3 r^2))/r,  B = (1 - 2/r^2)/r^3
//   overlap  A = 4/3 - 3 r/8,        B = 1/(8 r)
// With ic and rm, A = ic + 2 ic^3/3 + (3/4 - 3 rm/8) and B = (1 - 2 ic^2)
// ic^2 / r.  Returned is A - sub: above a wall far pairs lose most of A to
// the image's 1/|R|, and taking that off ic first (sub = 1/|R|) leaves the
// difference free of the rounding of A.
template <typename T>
RMW_HD void rpy_tt(T invr, T ic, T rm, T sub, T& A, T& B)
{
  const T w = ic * ic;
  A = fma_(T(2.0 / 3.0), w * ic, (ic - sub) + fma_(T(-0.375), rm, T(0.75)));
  B = fma_(T(-2), w, T(1)) * w * invr;
}

template <typename T>
RMW_HD CoefUF<T> coef_uf(const Geom<T>& g, T zi, T zj, int dom = kDomWall)
{
  const T one = T(1);
  CoefUF<T> c;
  T A;
  rpy_tt(g.invr, g.ic, g.rm, dom_has_wall(dom) ? g.invR : T(0), A, c.Bc);
  if (dom == kDomNoWall) {
    c.s = A; c.s5 = A; c.g2 = T(0); c.g3 = T(0); c.g4 = T(0);
    return c;
  }
  if (dom == kDomFreeSurface) {
    // + RPY(R) D v = A_R (v - 2 v_z z) + B_R R (R.v) - 2 B_R R_z v_z R
    T AR, BR;
    rpy_tt(g.invR, min_(g.invR, T(0.5)), min_(one / g.invR, T(2)), T(0), AR, BR);
    c.s = A + AR; c.s5 = A - AR; c.g2 = BR; c.g3 = T(-2) * BR * g.Rz; c.g4 = T(0);
    return c;
  }

  // Swan-Brady wall correction (mobility_numba.py:254-264) regrouped as
  // polynomials in w = 1/|R|^2 with E = e_z^2 = R_z^2 w.  With
  // h_hat = z_j/R_z the h_hat factors combine into division-free monomials:
  //   h_hat (1-h_hat) e_z^2 = z_i z_j w,  h_hat e_z / |R| = z_j w,
  //   (1-h_hat) e_z^2 = z_i R_z w,        h_hat^2 e_z^2 = z_j^2 w,
  // giving, with q = 1/|R|, zz = z_i z_j, b = R_z w,
  // P = -6 zz - 2 + 10 E + w (10/3 - 70 E/3) and m = (10/3) b w,
  //   f1 = -q [1 + w (2 zz + 2/3 - 2E) + w^2 (10E/3 - 2/3)]
  //   f2 = -q [1 + w P]
  //   f3 = 2 w [z_j + b P + m]
  //   f4 = 2 w [z_j - m]
  //   f5 = -4 q w [z_j^2 + E + w (2/3 - 5E)]
  T q = g.invR;
  T w = q * q;
  T b = g.Rz * w;
  T E = g.Rz * b;
  T zz = zi * zj;
  T t1 = fma_(T(2), zz, fma_(T(-2), E, T(2.0 / 3.0)));
  T t2 = fma_(T(10.0 / 3.0), E, T(-2.0 / 3.0));
  T qw = q * w;
  c.s = fma_(-qw, fma_(w, t2, t1), A);                     // RPY's A + f1, the -q of f1 taken off above
  T t3 = fma_(T(-6), zz, fma_(T(10), E, T(-2)));
  T t4 = fma_(T(-70.0 / 3.0), E, T(10.0 / 3.0));
  T P = fma_(w, t4, t3);
  c.g2 = -qw * fma_(w, P, one);                            // f2 w
  T c2 = qw + qw;
  T m = T(10.0 / 3.0) * b * w;
  c.g3 = c2 * fma_(b, P, zj + m);                          // f3 q
  c.g4 = c2 * (zj - m);                                    // f4 q
  T t7 = fma_(T(-5), E, T(2.0 / 3.0));
  T t8 = fma_(zj, zj, E);
  c.s5 = fma_(T(-2) * c2, fma_(w, t7, t8), c.s);           // + f5
  return c;
}

// The products below come in two forms: M v, and (ADD) acc + M v with acc
// entering the FMA chain, which saves the separate add of every component.
template <bool ADD, typename T>
RMW_HD T fma_or_mul(T a, T b, T acc) { return ADD ? fma_(a, b, acc) : a * b; }

template <bool ADD = false, typename T>
RMW_HD Vec3<T> apply_uf(const Geom<T>& g, const CoefUF<T>& c, T vx, T vy, T vz, const Vec3<T>& acc = Vec3<T>{})
{
  T p = fma_(g.dx, vx, g.dy * vy);
  T dv = fma_(g.dz, vz, p);        // d.v
  T Rv = fma_(g.Rz, vz, p);        // R.v
  T ge = fma_(c.g2, Rv, c.g3 * vz);  // coefficient of R
  T q = c.Bc * dv;                 // coefficient of d
  T qe = q + ge;                   // x and y rows share d_x = R_x, d_y = R_y
  Vec3<T> u;
  u.x = fma_(c.s, vx, fma_or_mul<ADD>(qe, g.dx, acc.x));
  u.y = fma_(c.s, vy, fma_or_mul<ADD>(qe, g.dy, acc.y));
  u.z = fma_(c.s5, vz, fma_(q, g.dz, fma_(ge, g.Rz, fma_or_mul<ADD>(c.g4, Rv, acc.z))));
  return u;
}

// Transposed block: UF_ij^T v, which is UF_ji v (the mobility is symmetric),
// so one evaluation of a pair serves both of its blobs.  The coefficients of
// v_z R and (R.v) z trade places.
template <bool ADD = false, typename T>
RMW_HD Vec3<T> apply_uf_t(const Geom<T>& g, const CoefUF<T>& c, T vx, T vy, T vz, const Vec3<T>& acc = Vec3<T>{})
{
  T p = fma_(g.dx, vx, g.dy * vy);
  T dv = fma_(g.dz, vz, p);
  T Rv = fma_(g.Rz, vz, p);
  T ge = fma_(c.g2, Rv, c.g4 * vz);
  T q = c.Bc * dv;
  T qe = q + ge;
  Vec3<T> u;
  u.x = fma_(c.s, vx, fma_or_mul<ADD>(qe, g.dx, acc.x));
  u.y = fma_(c.s, vy, fma_or_mul<ADD>(qe, g.dy, acc.y));
  u.z = fma_(c.s5, vz, fma_(q, g.dz, fma_(ge, g.Rz, fma_or_mul<ADD>(c.g3, Rv, acc.z))));
  return u;
}

// ---------------------------------------------------------------------------
// Wall coefficients shared by UT and WF (mobility_numba.py:659-665 and
// :1046-1052), for a given h_hat.  Returned pre-divided by powers of |R| so
// that they multiply R rather than e.
// ---------------------------------------------------------------------------
template <typename T> struct CoefRot {
  T c;    // RPY antisymmetric coefficient (1/r^3 far, (1 - 3r/8)/2 near)
  T F1r;  // F1 / |R|
  T F2r;  // F2 / |R|
  T F3r2; // F3 / |R|^2
  T F4;   // F4
};

// RPY: c = 1/r^3 far, (1 - 3r/8)/2 overlapping: ic^3 + (3/8 - 3 rm/16).
// Wall, for h = h_hat R_z, with q = 1/|R|, w = q^2, b = R_z w:
//   F1 = w,  F4 = -2 w q (h - b),  F3 = -2 w q B,  F2 = 2 w^2 (1 + 2 R_z B),
//   B = 3 h - 5 b   (h_hat e_z^2 = h b and h_hat e_z = h q: no division).
template <typename T>
RMW_HD CoefRot<T> coef_rot(const Geom<T>& g, T hnum, int dom = kDomWall)
{
  CoefRot<T> c;
  c.c = fma_(g.ic * g.ic, g.ic, fma_(T(-0.1875), g.rm, nan_of(g.r, T(0.375))));
  if (!dom_has_wall(dom)) {
    c.F1r = T(0); c.F2r = T(0); c.F3r2 = T(0); c.F4 = T(0);
    return c;
  }
  T q = g.invR;
  T w = q * q;
  T b = g.Rz * w;
  T qw = q * w;
  T c2 = qw + qw;
  T c2w = c2 * w;
  T B = fma_(T(-5), b, T(3) * hnum);
  c.F1r = qw;
  c.F3r2 = -c2w * B;
  c.F2r = fma_(T(-2) * g.Rz, c.F3r2, c2w);
  c.F4 = c2 * (b - hnum);
  return c;
}

// WF v = c (v x d) - [F1 (v x e) + (F2 v_z + F3 (e.v)) (z x e) + F4 (v x z)]:
//   x =  G v_y + (h - k v_z) d_y,   y = -G v_x - (h - k v_z) d_x,
//   z =  k (v_x d_y - v_y d_x)
// with G = c d_z - F1 R_z/|R| - F4, k = c - F1/|R| and
// h = F2 v_z/|R| + F3 (R.v)/|R|^2.
template <bool ADD = false, typename T>
RMW_HD Vec3<T> apply_wf(const Geom<T>& g, const CoefRot<T>& c, T vx, T vy, T vz, const Vec3<T>& acc = Vec3<T>{})
{
  T Rv = fma_(g.dx, vx, fma_(g.dy, vy, g.Rz * vz));
  T G = fma_(c.c, g.dz, -fma_(c.F1r, g.Rz, c.F4));
  T k = c.c - c.F1r;
  T h = fma_(c.F3r2, Rv, (c.F2r - k) * vz);
  T zc = fma_(vx, g.dy, -(vy * g.dx));       // (v x d)_z = (v x R)_z
  Vec3<T> w;
  w.x = fma_(G, vy, fma_or_mul<ADD>(h, g.dy, acc.x));
  w.y = fma_(-G, vx, fma_or_mul<ADD>(-h, g.dx, acc.y));
  w.z = fma_or_mul<ADD>(k, zc, acc.z);
  return w;
}

// UT v = c (v x d) - [F1 (e' x v) + (F2 z + F3 e') ((z x e').v) + F4 (z x v)],
// e' = (-d_x, -d_y, R_z)/|R|, coefficients built with h_hat = z_i / R_z:
//   x =  G v_y - k d_y v_z + m d_x,   y = -G v_x + k d_x v_z + m d_y,
//   z = (k - F2/|R|) q - m R_z
// with G = c d_z + F1 R_z/|R| + F4, k = c - F1/|R|, q = d_y v_x - d_x v_y
// (= |R| (z x e').v) and m = F3 q/|R|^2.
template <bool ADD = false, typename T>
RMW_HD Vec3<T> apply_ut(const Geom<T>& g, const CoefRot<T>& c, T vx, T vy, T vz, const Vec3<T>& acc = Vec3<T>{})
{
  T q = fma_(g.dy, vx, -(g.dx * vy));
  T m = c.F3r2 * q;
  T G = fma_(c.c, g.dz, fma_(c.F1r, g.Rz, c.F4));
  T k = c.c - c.F1r;
  T kv = k * vz;
  Vec3<T> u;
  u.x = fma_(G, vy, fma_(m, g.dx, fma_or_mul<ADD>(-kv, g.dy, acc.x)));
  u.y = fma_(-G, vx, fma_(m, g.dy, fma_or_mul<ADD>(kv, g.dx, acc.y)));
  u.z = fma_(k - c.F2r, q, fma_or_mul<ADD>(-m, g.Rz, acc.z));
  return u;
}

// Transposes of the rotational couplings, read off the component forms
// above.  Reciprocity gives UT_ji = WF_ij^T and WF_ji = UT_ij^T, so with
// the coefficients of the pair (i, j) these are the blocks of (j, i).
// WF_ij^T v, with G and k of WF, q = d_y v_x - d_x v_y and m = F3 q/|R|^2:
//   x = m d_x - G v_y + k d_y v_z,   y = m d_y + G v_x - k d_x v_z,
//   z = (F2/|R| + F3 R_z/|R|^2 - k) q
template <bool ADD = false, typename T>
RMW_HD Vec3<T> apply_wf_t(const Geom<T>& g, const CoefRot<T>& c, T vx, T vy, T vz, const Vec3<T>& acc = Vec3<T>{})
{
  T q = fma_(g.dy, vx, -(g.dx * vy));
  T m = c.F3r2 * q;
  T G = fma_(c.c, g.dz, -fma_(c.F1r, g.Rz, c.F4));
  T k = c.c - c.F1r;
  T kv = k * vz;
  Vec3<T> w;
  w.x = fma_(-G, vy, fma_(m, g.dx, fma_or_mul<ADD>(kv, g.dy, acc.x)));
  w.y = fma_(G, vx, fma_(m, g.dy, fma_or_mul<ADD>(-kv, g.dx, acc.y)));
  w.z = fma_or_mul<ADD>(fma_(c.F3r2, g.Rz, c.F2r - k), q, acc.z);
  return w;
}

// UT_ij^T v, with G and k of UT, p = d_x v_x + d_y v_y, q as above and
// K = k - F2/|R| - F3 R_z/|R|^2:
//   x =  F3 d_y p/|R|^2 - G v_y + K d_y v_z
//   y = -F3 d_x p/|R|^2 + G v_x - K d_x v_z
//   z = -k q
template <bool ADD = false, typename T>
RMW_HD Vec3<T> apply_ut_t(const Geom<T>& g, const CoefRot<T>& c, T vx, T vy, T vz, const Vec3<T>& acc = Vec3<T>{})
{
  T p = fma_(g.dx, vx, g.dy * vy);
  T q = fma_(g.dy, vx, -(g.dx * vy));
  T G = fma_(c.c, g.dz, fma_(c.F1r, g.Rz, c.F4));
  T k = c.c - c.F1r;
  T K = k - fma_(c.F3r2, g.Rz, c.F2r);
  T m = fma_(c.F3r2, p, K * vz);
  Vec3<T> u;
  u.x = fma_(-G, vy, fma_or_mul<ADD>(m, g.dy, acc.x));
  u.y = fma_(G, vx, fma_or_mul<ADD>(-m, g.dx, acc.y));
  u.z = fma_or_mul<ADD>(-k, q, acc.z);
  return u;
}

// ---------------------------------------------------------------------------
// WT: rotation from torque.  mobility_numba.py:1256-1321
// ---------------------------------------------------------------------------
template <typename T> struct CoefWT {
  T s;    // A + G1
  T Bc;   // coefficient of (d.v) d
  T G2r;  // G2 / |R|^2 -> (R.v) R
  T G3r;  // G3 / |R|   -> (R.v) z
  T G4r;  // G4 / |R|^2 -> ((z x R).v)(z x R)
};

// RPY:  far      A = -1/(2 r^3),                  B = 3/(2 r^5)
//       overlap  A = 1 - 27 r/32 + 5 r^3/64,      B = 9/(32 r) - 3 r/64
// A = -ic^3/2 + (17/16 + rm (-27/32 + 5 rm^2/64)),
// B = (3 ic^4/2 + (3/16 - 3 rm^2/64)) / r.
// Wall, with q = 1/|R|, w = q^2: G1 = (1 - 6 e_z^2) q^3/2, G2 = -3 q^3/2,
// G3 = 3 q^3 e_z, G4 = 3 q^3.
template <typename T>
RMW_HD CoefWT<T> coef_wt(const Geom<T>& g, int dom = kDomWall)
{
  CoefWT<T> c;
  T w2 = g.ic * g.ic;
  T m2 = g.rm * g.rm;
  T A = fma_(T(-0.5) * w2, g.ic, fma_(fma_(T(0.078125), m2, T(-0.84375)), g.rm, T(1.0625)));
  c.Bc = fma_(T(1.5) * w2, w2, fma_(T(-0.046875), m2, T(0.1875))) * g.invr;
  if (!dom_has_wall(dom)) {
    c.s = A; c.G2r = T(0); c.G3r = T(0); c.G4r = T(0);
    return c;
  }
  T q = g.invR;
  T w = q * q;
  T b = g.Rz * w;
  T qw = q * w;
  c.s = fma_(qw, fma_(T(-3) * g.Rz, b, T(0.5)), A);
  c.G4r = T(3) * qw * w;
  c.G2r = T(-0.5) * c.G4r;
  c.G3r = T(3) * qw * b;
  return c;
}

template <bool ADD = false, typename T>
RMW_HD Vec3<T> apply_wt(const Geom<T>& g, const CoefWT<T>& c, T vx, T vy, T vz, const Vec3<T>& acc = Vec3<T>{})
{
  T p = fma_(g.dx, vx, g.dy * vy);
  T dv = fma_(g.dz, vz, p);
  T Rv = fma_(g.Rz, vz, p);
  T zt = fma_(g.dx, vy, -(g.dy * vx));   // (z x R).v
  T q = c.Bc * dv;
  T ge = c.G2r * Rv;
  T qe = q + ge;
  T gz = c.G4r * zt;
  Vec3<T> w;
  w.x = fma_(c.s, vx, fma_(qe, g.dx, fma_or_mul<ADD>(-gz, g.dy, acc.x)));
  w.y = fma_(c.s, vy, fma_(qe, g.dy, fma_or_mul<ADD>(gz, g.dx, acc.y)));
  w.z = fma_(c.s, vz, fma_(q, g.dz, fma_(ge, g.Rz, fma_or_mul<ADD>(c.G3r, Rv, acc.z))));
  return w;
}

// WT_ij^T v = WT_ji v: the (R.v) z term becomes v_z R.
template <bool ADD = false, typename T>
RMW_HD Vec3<T> apply_wt_t(const Geom<T>& g, const CoefWT<T>& c, T vx, T vy, T vz, const Vec3<T>& acc = Vec3<T>{})
{
  T p = fma_(g.dx, vx, g.dy * vy);
  T dv = fma_(g.dz, vz, p);
  T Rv = fma_(g.Rz, vz, p);
  T zt = fma_(g.dx, vy, -(g.dy * vx));
  T q = c.Bc * dv;
  T ge = fma_(c.G2r, Rv, c.G3r * vz);
  T qe = q + ge;
  T gz = c.G4r * zt;
  Vec3<T> w;
  w.x = fma_(c.s, vx, fma_(qe, g.dx, fma_or_mul<ADD>(-gz, g.dy, acc.x)));
  w.y = fma_(c.s, vy, fma_(qe, g.dy, fma_or_mul<ADD>(gz, g.dx, acc.y)));
  w.z = fma_(c.s, vz, fma_(q, g.dz, fma_or_mul<ADD>(ge, g.Rz, acc.z)));
  return w;
}

// ---------------------------------------------------------------------------
// Explicit 3x3 blocks, m[r][c] = e_r . B e_c, of the four dyadic forms above
// (read off apply_uf / apply_ut / apply_wf / apply_wt at the unit vectors).
// A kernel that applies one pair's blocks to several right-hand sides forms
// them once and then spends 9 FMAs per block, side and right-hand side
// (the transposed blocks are the same entries read by columns).
// ---------------------------------------------------------------------------
template <typename T> struct Mat3 { T m[3][3]; };

template <typename T>
RMW_HD Mat3<T> mat_uf(const Geom<T>& g, const CoefUF<T>& c)
{
  Mat3<T> M;
  const T P = c.Bc + c.g2;
  const T h = fma_(c.Bc, g.dz, c.g2 * g.Rz);
  const T a3 = h + c.g3, b3 = h + c.g4;
  const T Pdx = P * g.dx;
  M.m[0][0] = fma_(Pdx, g.dx, c.s);
  M.m[0][1] = Pdx * g.dy;
  M.m[0][2] = a3 * g.dx;
  M.m[1][0] = M.m[0][1];
  M.m[1][1] = fma_(P * g.dy, g.dy, c.s);
  M.m[1][2] = a3 * g.dy;
  M.m[2][0] = b3 * g.dx;
  M.m[2][1] = b3 * g.dy;
  M.m[2][2] = fma_(c.Bc * g.dz, g.dz, fma_(fma_(c.g2, g.Rz, c.g3 + c.g4), g.Rz, c.s5));
  return M;
}

// UT (coefficients of coef_rot(g, z_i)); m[2][2] = 0.
template <typename T>
RMW_HD Mat3<T> mat_ut(const Geom<T>& g, const CoefRot<T>& c)
{
  Mat3<T> M;
  const T G = fma_(c.c, g.dz, fma_(c.F1r, g.Rz, c.F4));
  const T K = c.c - c.F1r - fma_(c.F3r2, g.Rz, c.F2r);
  const T cf = c.c - c.F1r;
  const T Fx = c.F3r2 * g.dx;
  M.m[0][0] = Fx * g.dy;
  M.m[0][1] = fma_(-Fx, g.dx, G);
  M.m[0][2] = -cf * g.dy;
  M.m[1][0] = fma_(c.F3r2 * g.dy, g.dy, -G);
  M.m[1][1] = -M.m[0][0];
  M.m[1][2] = cf * g.dx;
  M.m[2][0] = K * g.dy;
  M.m[2][1] = -K * g.dx;
  M.m[2][2] = T(0);
  return M;
}

// WF (coefficients of coef_rot(g, z_j)); m[2][2] = 0.
template <typename T>
RMW_HD Mat3<T> mat_wf(const Geom<T>& g, const CoefRot<T>& c)
{
  Mat3<T> M;
  const T G = fma_(c.c, g.dz, -fma_(c.F1r, g.Rz, c.F4));
  const T K = c.c - c.F1r - fma_(c.F3r2, g.Rz, c.F2r);
  const T cf = c.c - c.F1r;
  const T Fx = c.F3r2 * g.dx;
  M.m[0][0] = Fx * g.dy;
  M.m[0][1] = fma_(c.F3r2 * g.dy, g.dy, G);
  M.m[0][2] = -K * g.dy;
  M.m[1][0] = -fma_(Fx, g.dx, G);
  M.m[1][1] = -M.m[0][0];
  M.m[1][2] = K * g.dx;
  M.m[2][0] = cf * g.dy;
  M.m[2][1] = -cf * g.dx;
  M.m[2][2] = T(0);
  return M;
}

template <typename T>
RMW_HD Mat3<T> mat_wt(const Geom<T>& g, const CoefWT<T>& c)
{
  Mat3<T> M;
  const T P = c.Bc + c.G2r;
  const T h = fma_(c.Bc, g.dz, c.G2r * g.Rz);
  const T h3 = h + c.G3r;
  const T dxy = g.dx * g.dy;
  M.m[0][0] = fma_(P * g.dx, g.dx, fma_(c.G4r * g.dy, g.dy, c.s));
  M.m[0][1] = (P - c.G4r) * dxy;
  M.m[0][2] = h * g.dx;
  M.m[1][0] = M.m[0][1];
  M.m[1][1] = fma_(P * g.dy, g.dy, fma_(c.G4r * g.dx, g.dx, c.s));
  M.m[1][2] = h * g.dy;
  M.m[2][0] = h3 * g.dx;
  M.m[2][1] = h3 * g.dy;
  M.m[2][2] = fma_(c.Bc * g.dz, g.dz, fma_(fma_(c.G2r, g.Rz, c.G3r), g.Rz, c.s));
  return M;
}

// ---------------------------------------------------------------------------
// Blobs of different radii (target radius a, source radius b), lengths in
// absolute units, normalisation 1/(8 pi eta) folded in by the caller.
// mobility_numba.py:1479-1658.  The self pair (d = 0) needs no special
// case: it falls in the inner RPY regime.
//
//   RPY:  C1 I + C2 d d^T with, for r = |d| and s = a^2 + b^2,
//         r > a + b:     C1 = (1 + s/(3r^2))/r,  C2 = (1 - s/r^2)/r^3
//         r > |b - a|:   C1 = 4/(3ab) [(a + b)/2 - ((b-a)^2 + 3r^2)^2/(32 r^3)]
//                        C2 = 4/(3ab) (3/32) ((b-a)^2 - r^2)^2 / r^5
//         otherwise:     C1 = 4/(3 max(a, b)),   C2 = 0
//   wall: -S D v with D = diag(1, 1, -1), R = (d_x, d_y, x3 + y3) (x3, y3 the
//         target and source heights), rho = |R| and
//         S = alpha I + beta R R^T + g1 R z^T + g2 z R^T + delta z z^T,
//   the image Stokeslet, its doublets weighted by ca = 2a^2/3, cb = 2b^2/3
//   and the quadrupole weighted by cab = 2a^2 b^2/3 collected per dyad.
//   free surface (mobility_numba.py:1941-2093): + (C1' I + C2' R R^T) D v,
//         the RPY coefficients of the three regimes evaluated at rho, i.e.
//         S = -(C1' I + C2' R R^T) in the wall's form.
// ---------------------------------------------------------------------------
enum : int { kRadiiUnbounded = 0, kRadiiWall = 1, kRadiiFreeSurface = 2 };

template <typename T> struct CoefRadii {
  T C1, C2;                 // RPY
  T al, be, g1, g2, de;     // wall (or image) dyads
};

// RPY coefficients C1, C2 of radii a, b at squared distance r2.
template <typename T>
RMW_HD void rpy_radii(T r2, T a, T b, T inva, T invb, T& C1, T& C2)
{
  const T invr = rsq(r2);
  const T r = r2 > T(0) ? r2 * invr : T(0);
  const T w = invr * invr;
  const T s = a * a + b * b;
  const T C1_far = fma_(s * w, T(1.0 / 3.0), T(1)) * invr;
  const T C2_far = fma_(-s, w, T(1)) * w * invr;
  const T dab = b - a;
  const T dab2 = dab * dab;
  const T k1 = T(4.0 / 3.0) * inva * invb;
  const T t = fma_(T(3), r2, dab2);
  const T invr3 = w * invr;
  const T C1_mid = k1 * (T(0.5) * (a + b) - T(1.0 / 32.0) * t * t * invr3);
  const T u = dab2 - r2;
  const T C2_mid = k1 * T(3.0 / 32.0) * u * u * invr3 * w;
  const T C1_in = T(4.0 / 3.0) * (inva < invb ? inva : invb);
  const bool far = r > a + b;
  const bool mid = r > (dab < T(0) ? -dab : dab);
  C1 = far ? C1_far : (mid ? C1_mid : C1_in);
  C2 = far ? C2_far : (mid ? C2_mid : T(0));
}

// bnd: kRadiiUnbounded, kRadiiWall or kRadiiFreeSurface.
template <typename T>
RMW_HD CoefRadii<T> coef_radii(T dx, T dy, T dz, T Rz, T x3, T y3, T a, T b, T inva, T invb, int bnd)
{
  CoefRadii<T> c;
  const T r2 = dx * dx + dy * dy + dz * dz;
  rpy_radii(r2, a, b, inva, invb, c.C1, c.C2);
  if (bnd == kRadiiWall) {
    // powers of w = 1/rho^2 gathered per dyad (Horner), q = 1/rho:
    //   alpha = q [1 + w (s/3 + 2 x3 y3 + w (-3 m R_z - cab + 5 cab R_z^2 w))]
    //   beta  = q^3 [1 - w (s + 6 x3 y3 - w (15 m R_z + 5 cab - 35 cab R_z^2 w))]
    //   g1 = q^3 [x3 (t - 2) + z],  g2 = q^3 [y3 (-t - 2) + z],
    //   t = 3 (ca - cb) w,  z = 10 cab R_z w^2
    //   delta = -q [2 + w (ca + cb + 2 cab w)],  m = ca y3 + cb x3
    const T a2 = a * a, b2 = b * b, s = a2 + b2;
    const T rho2 = fma_(dx, dx, fma_(dy, dy, Rz * Rz));
    const T q = rsq(rho2);
    const T w = q * q;
    const T q3 = q * w;
    const T ca = T(2.0 / 3.0) * a2, cb = T(2.0 / 3.0) * b2, cab = ca * b2;
    const T xy = x3 * y3;
    const T mR = fma_(ca, y3, cb * x3) * Rz;
    const T cz = cab * Rz * w;               // cab R_z w
    const T cR = cz * Rz;
    c.al = q * fma_(w, fma_(w, fma_(T(5), cR, fma_(T(-3), mR, -cab)), fma_(T(2), xy, T(1.0 / 3.0) * s)), T(1));
    c.be = q3 * fma_(w, fma_(w, fma_(T(-35), cR, fma_(T(15), mR, T(5) * cab)), fma_(T(-6), xy, -s)), T(1));
    const T t = T(3) * (ca - cb) * w;
    const T z = T(10) * cz * w;
    c.g1 = q3 * fma_(x3, t - T(2), z);
    c.g2 = q3 * fma_(y3, -t - T(2), z);
    c.de = -q * fma_(w, fma_(T(2) * cab, w, ca + cb), T(2));
  } else if (bnd == kRadiiFreeSurface) {
    T I1, I2;
    rpy_radii(dx * dx + dy * dy + Rz * Rz, a, b, inva, invb, I1, I2);
    c.al = -I1;
    c.be = -I2;
    c.g1 = c.g2 = c.de = T(0);
  } else {
    c.al = c.be = c.g1 = c.g2 = c.de = T(0);
  }
  return c;
}

template <typename T, bool ADD = false>
RMW_HD Vec3<T> apply_radii(T dx, T dy, T dz, T Rz, const CoefRadii<T>& c, T vx, T vy, T vz,
                           const Vec3<T>& acc = Vec3<T>{})
{
  const T p = fma_(dx, vx, dy * vy);
  const T dv = fma_(dz, vz, p);
  const T Rv = fma_(-Rz, vz, p);          // R . D v
  const T h = fma_(c.be, Rv, -c.g1 * vz);   // coefficient of -R
  const T q = c.C2 * dv;
  const T k = c.C1 - c.al, e = q - h;
  Vec3<T> u;
  u.x = fma_(k, vx, fma_or_mul<ADD>(e, dx, acc.x));
  u.y = fma_(k, vy, fma_or_mul<ADD>(e, dy, acc.y));
  u.z = fma_(c.C1 + c.al + c.de, vz, fma_(q, dz, fma_(-h, Rz, fma_or_mul<ADD>(-c.g2, Rv, acc.z))));
  return u;
}

// M_ij^T v (the coefficients as computed for the ordered pair (i, j)).
template <typename T>
RMW_HD Vec3<T> apply_radii_t(T dx, T dy, T dz, T Rz, const CoefRadii<T>& c, T vx, T vy, T vz)
{
  const T p = fma_(dx, vx, dy * vy);
  const T dv = fma_(dz, vz, p);
  const T Rv = fma_(Rz, vz, p);           // R . v
  const T h = fma_(c.be, Rv, c.g2 * vz);    // coefficient of -D R
  const T q = c.C2 * dv;
  const T k = c.C1 - c.al, e = q - h;
  Vec3<T> u;
  u.x = fma_(k, vx, e * dx);
  u.y = fma_(k, vy, e * dy);
  u.z = fma_(c.C1 + c.al + c.de, vz, fma_(q, dz, fma_(h, Rz, c.g1 * Rv)));
  return u;
}

// ---------------------------------------------------------------------------
// Self blocks (i == j, central box), mobility_numba.py:202-208 + 245-252,
// :653-657, :1040-1044, :1291-1297.  h = z_i / a (effective height).
// ---------------------------------------------------------------------------
template <typename T>
RMW_HD Vec3<T> self_uf(T h, T vx, T vy, T vz)
{
  T ih = T(1) / h;
  T ih3 = ih * ih * ih;
  T ih5 = ih3 * ih * ih;
  T pxy = T(4) / T(3) - (T(9) * ih - T(2) * ih3 + ih5) / T(12);
  T pz = T(4) / T(3) - (T(9) * ih - T(4) * ih3 + ih5) / T(6);
  return Vec3<T>{pxy * vx, pxy * vy, pz * vz};
}

// UT self: M_xy = +h^-4/8, M_yx = -h^-4/8.
template <typename T>
RMW_HD Vec3<T> self_ut(T h, T vx, T vy, T vz)
{
  T ih = T(1) / h;
  T c = T(0.125) * ih * ih * ih * ih;
  return Vec3<T>{c * vy, -c * vx, T(0)};
}

// WF self: M_xy = -h^-4/8, M_yx = +h^-4/8.
template <typename T>
RMW_HD Vec3<T> self_wf(T h, T vx, T vy, T vz)
{
  T ih = T(1) / h;
  T c = T(0.125) * ih * ih * ih * ih;
  return Vec3<T>{-c * vy, c * vx, T(0)};
}

template <typename T>
RMW_HD Vec3<T> self_wt(T h, T vx, T vy, T vz)
{
  T ih = T(1) / h;
  T ih3 = ih * ih * ih;
  T pxy = T(1) - T(0.3125) * ih3;
  T pz = T(1) - T(0.125) * ih3;
  return Vec3<T>{pxy * vx, pxy * vy, pz * vz};
}

// Self terms of every domain (same units as the wall ones): no wall, the
// bare RPY self mobility (4/3 I, 0, 0, I); free surface, 4/3 I plus the
// image RPY(R) D at R = (0, 0, 2h); in plane, the wall terms (the caller
// projects).
template <typename T>
RMW_HD Vec3<T> self_uf_dom(int dom, T h, T vx, T vy, T vz)
{
  const T s = T(4) / T(3);
  if (dom == kDomNoWall) return Vec3<T>{s * vx, s * vy, s * vz};
  if (dom == kDomFreeSurface) {
    const T R = h + h;
    T AR, BR;
    rpy_tt(T(1) / R, min_(T(1) / R, T(0.5)), min_(R, T(2)), T(0), AR, BR);
    return Vec3<T>{(s + AR) * vx, (s + AR) * vy, (s - AR - R * R * BR) * vz};
  }
  return self_uf(h, vx, vy, vz);
}
template <typename T>
RMW_HD Vec3<T> self_ut_dom(int dom, T h, T vx, T vy, T vz)
{
  return dom_has_wall(dom) ? self_ut(h, vx, vy, vz) : Vec3<T>{T(0), T(0), T(0)};
}
template <typename T>
RMW_HD Vec3<T> self_wf_dom(int dom, T h, T vx, T vy, T vz)
{
  return dom_has_wall(dom) ? self_wf(h, vx, vy, vz) : Vec3<T>{T(0), T(0), T(0)};
}
template <typename T>
RMW_HD Vec3<T> self_wt_dom(int dom, T h, T vx, T vy, T vz)
{
  return dom_has_wall(dom) ? self_wt(h, vx, vy, vz) : Vec3<T>{vx, vy, vz};
}

}  // namespace rmw
