// Device code shared by the wall-RPY product kernels: blob staging, the block
// masks, one pair's evaluation for one target (ordered kernels) or for both
// of its blobs (symmetric kernels), the symmetric kernels' parameters and
// the last step of every product (self term, damping, scaling).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "rmw_internal.h"
#include "rmw_pair_terms.h"
#include "rmw_tile_pairs.h"
#include "rmw_accum.h"

namespace rmw {

constexpr int kBlock = 256;  // targets per workgroup = sources per LDS tile
enum : int { kUF = 1, kUT = 2, kWF = 4, kWT = 8 };

// ---------------------------------------------------------------------------
// Blob staging: scaled position (x/a, y/a, z_eff/a) with z_eff = max(z, a)
// (shift_heights, mobility.py:52-64) and damping B = min(z/a, 1)
// (damping_matrix_B, mobility.py:67-84) when a wall bounds the fluid; the
// no-wall and free-surface products take the heights as they are
// (mobility.py:1119-1129, 1390-1406).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void scale_blob(double x, double y, double z, double a, double inva, double& X, double& Y,
                                           double& Z, double& B, int dom)
{
  // the scaled coordinates are rounded here: were the product fused into a
  // later difference, blobs at one position would not be at distance 0
#pragma clang fp contract(off)
  const bool wall = dom_has_wall(dom);
  const double ze = wall && z <= a ? a : z;
  X = x * inva;
  Y = y * inva;
  Z = ze * inva;
  B = wall && z < a ? z * inva : 1.0;
}

__device__ __forceinline__ void load_blob(const double* __restrict__ r, int64_t g, double a, double inva,
                                          double& X, double& Y, double& Z, double& B, int dom)
{
  scale_blob(r[3 * g], r[3 * g + 1], r[3 * g + 2], a, inva, X, Y, Z, B, dom);
}

// A blob's position and its K forces and torques as they lie in memory:
// loaded ahead of their use, scaled when they are staged.
template <int K, bool NF, bool NT>
struct RawBlob {
  double r[3];
  double f[NF ? K : 1][3], t[NT ? K : 1][3];
  __device__ __forceinline__ void load(const double* __restrict__ rr, const double* __restrict__ ff,
                                       const double* __restrict__ tt, int64_t stride, int64_t g)
  {
#pragma unroll
    for (int c = 0; c < 3; ++c) r[c] = rr[3 * g + c];
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if constexpr (NF) f[k][c] = ff[k * stride + 3 * g + c];
        if constexpr (NT) t[k][c] = tt[k * stride + 3 * g + c];
      }
  }
};

template <int K, int ACC>
__device__ __forceinline__ void flush_all(Acc<ACC> (&u)[K][3], Acc<ACC> (&w)[K][3])
{
#pragma unroll
  for (int k = 0; k < K; ++k)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      u[k][c].flush();
      w[k][c].flush();
    }
}

template <int MASK> struct BlockTraits {
  static constexpr bool HU = (MASK & (kUF | kUT)) != 0;  // writes velocity
  static constexpr bool HW = (MASK & (kWF | kWT)) != 0;  // writes omega
  static constexpr bool NF = (MASK & (kUF | kWF)) != 0;  // reads force
  static constexpr bool NT = (MASK & (kUT | kWT)) != 0;  // reads torque
  static constexpr int OC = 3 * ((HU ? 1 : 0) + (HW ? 1 : 0));
};

template <typename T> struct V4;
template <> struct V4<float> { using type = float4; };
template <> struct V4<double> { using type = double4; };

// One (target, source) pair for all blocks of MASK and all K right-hand
// sides.  sf(k) and st(k) give the scaled force and torque of the source
// (anything with members x, y, z); `skip` drops the pair (the self pair of
// the central box).
template <int MASK, int K, int ACC, typename T, int DOM, typename SF, typename ST>
__device__ __forceinline__ void pair_eval(T dx, T dy, T dz, T zi, T zj, SF&& sf, ST&& st, bool skip,
                                          Acc<ACC> (&u)[K][3], Acc<ACC> (&w)[K][3])
{
  using BT = BlockTraits<MASK>;
  Geom<T> g = make_geom(dx, dy, dz, zi, zj);
  CoefUF<T> cuf;
  CoefRot<T> cut, cwf;
  CoefWT<T> cwt;
  if constexpr ((MASK & kUF) != 0) cuf = coef_uf(g, zi, zj, DOM);
  if constexpr ((MASK & kUT) != 0) cut = coef_rot(g, zi, DOM);
  if constexpr ((MASK & kWF) != 0) cwf = coef_rot(g, zj, DOM);
  if constexpr ((MASK & kWT) != 0) cwt = coef_wt(g, DOM);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    constexpr bool UF = (MASK & kUF) != 0, UT = (MASK & kUT) != 0, WF = (MASK & kWF) != 0, WT = (MASK & kWT) != 0;
    Vec3<T> uu{}, ww{}, fv, tv;
    if constexpr (BT::NF) { const auto q = sf(k); fv = Vec3<T>{q.x, q.y, q.z}; }
    if constexpr (BT::NT) { const auto q = st(k); tv = Vec3<T>{q.x, q.y, q.z}; }
    // each block's product is seeded with the one before it
    if constexpr (UF) uu = apply_uf(g, cuf, fv.x, fv.y, fv.z);
    if constexpr (UT) uu = apply_ut<UF>(g, cut, tv.x, tv.y, tv.z, uu);
    if constexpr (WF) ww = apply_wf(g, cwf, fv.x, fv.y, fv.z);
    if constexpr (WT) ww = apply_wt<WF>(g, cwt, tv.x, tv.y, tv.z, ww);
    if constexpr (BT::HU) {
      u[k][0].add(skip ? T(0) : uu.x);
      u[k][1].add(skip ? T(0) : uu.y);
      u[k][2].add(skip ? T(0) : uu.z);
    }
    if constexpr (BT::HW) {
      w[k][0].add(skip ? T(0) : ww.x);
      w[k][1].add(skip ? T(0) : ww.y);
      w[k][2].add(skip ? T(0) : ww.z);
    }
  }
}

struct MutSys {
  int64_t b0, n, n_t;   // first blob, blobs, tiles of kBlock
  int64_t item0;        // first work item
  int64_t pi0, pj0;     // first target-side / source-side slot
  int64_t t0;           // tiles of the systems before
};

// Source-side sums over one source's images: in the pair's type where the
// mode sums images so anyway, in FP64 for the FP32 modes that do not.
template <int ACC, typename R>
using ImageSum = typename std::conditional<ACC == RMW_PREC_F32_F64ACC || ACC == RMW_PREC_F32_KAHAN, double, R>::type;

struct MutParams {
  const double* r;
  const double* f;          // K right-hand sides rhs_stride apart, or null
  const double* t;
  int64_t rhs_stride;
  double a, inva, c1, c2;
  double* part_i;           // [slot][K][kBlock][OC]
  double* part_j;
  const MutSys* table;      // nullptr -> single
  MutSys single;
  int nsys;
  int64_t n_items, chunk_blocks;   // work item: a run of chunk_blocks 64-source blocks
  int periodic;             // bit d set when L_d > 0 (the PER instantiations)
  double L[3], iL[3];       // periodic lengths / a and their inverses (0: none)
};

__device__ __forceinline__ MutSys mut_sys_of_item(const MutParams& p, int64_t item)
{
  if (!p.table) return p.single;
  int lo = 0, hi = p.nsys - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (p.table[mid].item0 <= item) lo = mid; else hi = mid - 1;
  }
  return p.table[lo];
}

// One unordered pair (or one image of it) with d = (dx, dy, dz) applied on
// both sides: target side u_i += UF f_j + UT t_j, w_i += WF f_j + WT t_j;
// source side u_j += UF^T f_i + WF^T t_i, w_j += UT^T f_i + WT^T t_i.
// sf(k, c), st(k, c): the source's scaled force and torque; fi, ti: the
// target's.  MASKED: a pair with on = false contributes exact zeros.  ROT:
// the source-side sums move one lane down as they are added to (rol1).
template <int MASK, int K, int ACC, typename R, int DOM, bool MASKED, bool ROT, typename JT, int NFK, int NTK,
          typename SF, typename ST>
__device__ __forceinline__ void mutual_apply(R dx, R dy, R dz, R zi, R zj, bool on, const R (&fi)[NFK][3],
                                             const R (&ti)[NTK][3], SF&& sf, ST&& st, Acc<ACC> (&u)[K][3],
                                             Acc<ACC> (&w)[K][3], JT (&ja)[K][BlockTraits<MASK>::OC])
{
  using BT = BlockTraits<MASK>;
  constexpr bool UF = (MASK & kUF) != 0, UT = (MASK & kUT) != 0, WF = (MASK & kWF) != 0, WT = (MASK & kWT) != 0;
  // several right-hand sides: form the pair's blocks once as 3x3 matrices
  constexpr bool kMat = K >= 2;
  auto acc_j = [](JT& a, JT x) {
    if constexpr (ROT) a = rol1(a) + x; else a = a + x;
  };
  // sums that stay where they are, in the pair's type: they seed the products
  constexpr bool CJ = !ROT && std::is_same<JT, R>::value;
  // a pair not taken contributes exact zeros (make_geom_on)
  const Geom<R> g = MASKED ? make_geom_on(dx, dy, dz, zi, zj, on) : make_geom(dx, dy, dz, zi, zj);
  CoefUF<R> cuf;
  CoefRot<R> cut, cwf;
  CoefWT<R> cwt;
  if constexpr (UF) cuf = coef_uf(g, zi, zj, DOM);
  if constexpr (UT || WF) { cut = coef_rot(g, zi, DOM); cwf = coef_rot(g, zj, DOM); }
  if constexpr (WT) cwt = coef_wt(g, DOM);
  if constexpr (kMat) {
    // the pair's blocks as 3x3 matrices (zero for pairs not taken)
    Mat3<R> Mu, Mc, Md, Mw;   // UF, UT, WF, WT of (i, j)
    if constexpr (UF) Mu = mat_uf(g, cuf);
    if constexpr (UT) Mc = mat_ut(g, cut);
    if constexpr (WF) Md = mat_wf(g, cwf);
    if constexpr (WT) Mw = mat_wt(g, cwt);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      R fj[3], tj[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if constexpr (BT::NF) fj[c] = sf(k, c);
        if constexpr (BT::NT) tj[c] = st(k, c);
      }
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        // target side: u_i += UF f_j + UT t_j, w_i += WF f_j + WT t_j
        // source side: u_j += UF^T f_i + WF^T t_i, w_j += UT^T f_i + WT^T t_i
        // (where the accumulator allows, its running sum seeds the
        // target-side chain: no separate add)
        constexpr bool kChain = Acc<ACC>::kChain;
        if constexpr (BT::HU) {
          R x = R(0), y = R(0);
          if constexpr (kChain) x = u[k][r].run();
          if constexpr (CJ) y = ja[k][r];
          if constexpr (UF) {
            x = fma_(Mu.m[r][0], fj[0], fma_(Mu.m[r][1], fj[1], kChain ? fma_(Mu.m[r][2], fj[2], x) : Mu.m[r][2] * fj[2]));
            y = fma_(Mu.m[0][r], fi[k][0], fma_(Mu.m[1][r], fi[k][1], CJ ? fma_(Mu.m[2][r], fi[k][2], y) : Mu.m[2][r] * fi[k][2]));
          }
          if constexpr (UT)
            x = fma_(Mc.m[r][0], tj[0], fma_(Mc.m[r][1], tj[1], r == 2 ? x : fma_(Mc.m[r][2], tj[2], x)));
          if constexpr (WF)
            y = fma_(Md.m[0][r], ti[k][0], fma_(Md.m[1][r], ti[k][1], r == 2 ? y : fma_(Md.m[2][r], ti[k][2], y)));
          if constexpr (kChain) u[k][r].run() = x; else u[k][r].add(x);
          if constexpr (CJ) ja[k][r] = y; else acc_j(ja[k][r], (JT)y);
        }
        if constexpr (BT::HW) {
          constexpr int o = BT::HU ? 3 : 0;
          R x = R(0), y = R(0);
          if constexpr (kChain) x = w[k][r].run();
          if constexpr (CJ) y = ja[k][o + r];
          if constexpr (WT) {
            x = fma_(Mw.m[r][0], tj[0], fma_(Mw.m[r][1], tj[1], kChain ? fma_(Mw.m[r][2], tj[2], x) : Mw.m[r][2] * tj[2]));
            y = fma_(Mw.m[0][r], ti[k][0], fma_(Mw.m[1][r], ti[k][1], CJ ? fma_(Mw.m[2][r], ti[k][2], y) : Mw.m[2][r] * ti[k][2]));
          }
          if constexpr (WF)
            x = fma_(Md.m[r][0], fj[0], fma_(Md.m[r][1], fj[1], r == 2 ? x : fma_(Md.m[r][2], fj[2], x)));
          if constexpr (UT)
            y = fma_(Mc.m[0][r], fi[k][0], fma_(Mc.m[1][r], fi[k][1], r == 2 ? y : fma_(Mc.m[2][r], fi[k][2], y)));
          if constexpr (kChain) w[k][r].run() = x; else w[k][r].add(x);
          if constexpr (CJ) ja[k][o + r] = y; else acc_j(ja[k][o + r], (JT)y);
        }
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      // target side: u_i = UF f_j + UT t_j, w_i = WF f_j + WT t_j;
      // source side: u_j = UF^T f_i + WF^T t_i, w_j = UT^T f_i + WT^T t_i;
      // each product is seeded with the one before it, the target side's
      // first one with the running sum where the accumulator allows
      // (FP32: for the UF block above a wall only.  A seeded chain rounds at the
      // running sum's size with every operation; error against 64 bits of the
      // blocked mode at 9000 blobs, seeded / added: UF 1.75e-7 / 1.96e-7 above
      // a wall but 9.3e-8 / 8.8e-8 without, UF + UT 1.12e-7 / 9.2e-8 without)
      constexpr bool C = Acc<ACC>::kChain && (sizeof(R) == 8 || (DOM == kDomWall && MASK == kUF));
      Vec3<R> ui{}, wi{}, uj{}, wj{};
      if constexpr (C && BT::HU) ui = Vec3<R>{u[k][0].run(), u[k][1].run(), u[k][2].run()};
      if constexpr (C && BT::HW) wi = Vec3<R>{w[k][0].run(), w[k][1].run(), w[k][2].run()};
      if constexpr (CJ && BT::HU) uj = Vec3<R>{ja[k][0], ja[k][1], ja[k][2]};
      if constexpr (CJ && BT::HW) {
        constexpr int o = BT::HU ? 3 : 0;
        wj = Vec3<R>{ja[k][o], ja[k][o + 1], ja[k][o + 2]};
      }
      if constexpr (UF) {
        ui = apply_uf<C>(g, cuf, sf(k, 0), sf(k, 1), sf(k, 2), ui);
        uj = apply_uf_t<CJ>(g, cuf, fi[k][0], fi[k][1], fi[k][2], uj);
      }
      if constexpr (UT) {
        ui = apply_ut<C || UF>(g, cut, st(k, 0), st(k, 1), st(k, 2), ui);
        uj = apply_wf_t<CJ || UF>(g, cwf, ti[k][0], ti[k][1], ti[k][2], uj);
      }
      if constexpr (WF) {
        wi = apply_wf<C>(g, cwf, sf(k, 0), sf(k, 1), sf(k, 2), wi);
        wj = apply_ut_t<CJ>(g, cut, fi[k][0], fi[k][1], fi[k][2], wj);
      }
      if constexpr (WT) {
        wi = apply_wt<C || WF>(g, cwt, st(k, 0), st(k, 1), st(k, 2), wi);
        wj = apply_wt_t<CJ || WF>(g, cwt, ti[k][0], ti[k][1], ti[k][2], wj);
      }
      auto put_j = [&](JT* a, const Vec3<R>& v) {
        if constexpr (CJ) {
          a[0] = v.x; a[1] = v.y; a[2] = v.z;
        } else {
          acc_j(a[0], (JT)v.x); acc_j(a[1], (JT)v.y); acc_j(a[2], (JT)v.z);
        }
      };
      auto put = [](Acc<ACC> (&s)[3], const Vec3<R>& v) {
        if constexpr (C) {
          s[0].run() = v.x; s[1].run() = v.y; s[2].run() = v.z;
        } else {
          s[0].add(v.x); s[1].add(v.y); s[2].add(v.z);
        }
      };
      if constexpr (BT::HU) {
        put(u[k], ui);
        put_j(&ja[k][0], uj);
      }
      if constexpr (BT::HW) {
        constexpr int o = BT::HU ? 3 : 0;
        put(w[k], wi);
        put_j(&ja[k][o], wj);
      }
    }
  }
}

// Output component c (0..OC-1) of right-hand side k for blob gi: the FP64
// self term, damping B and the remaining 1/a of the rotational rows added
// to the pair sum.
__device__ __forceinline__ void finish_output(const double* __restrict__ r, const double* __restrict__ f,
                                              const double* __restrict__ t, double* __restrict__ vel,
                                              double* __restrict__ omg, int mask, int k, int64_t gi, int c,
                                              double sum, int64_t rhs_stride, int64_t out_stride, double a,
                                              double inva, double c1, double c2, int dom, int periodic = 0,
                                              double L0 = 0.0, double L1 = 0.0, double L2 = 0.0)
{
  const bool HU = (mask & (kUF | kUT)) != 0;
  const bool HW = (mask & (kWF | kWT)) != 0;
  const bool wall = dom_has_wall(dom);
  const double z = r[3 * gi + 2];
  const double ze = wall && z <= a ? a : z;
  const double B = wall && z < a ? z * inva : 1.0;
  const double h = ze * inva;
  const double pz = dom == kDomInPlane ? 0.0 : 1.0;   // in plane: P v in, P u out
  const bool is_w = HW && (!HU || c >= 3);
  const int comp = c % 3;
  double fv[3] = {0, 0, 0}, tv[3] = {0, 0, 0};
  if (f) {
    const double* v = f + k * rhs_stride + 3 * gi;
    fv[0] = c1 * B * v[0]; fv[1] = c1 * B * v[1]; fv[2] = pz * c1 * B * v[2];
  }
  if (t) {
    const double* v = t + k * rhs_stride + 3 * gi;
    tv[0] = c2 * B * v[0]; tv[1] = c2 * B * v[1]; tv[2] = pz * c2 * B * v[2];
  }
  double self = 0.0;
  // images of the blob itself outside the central box (pseudo-periodic
  // symmetric kernels): pairs at d = (b_x L_x, b_y L_y, b_z L_z), z_i = z_j
  for (int bx = -(periodic & 1); bx <= (periodic & 1); ++bx)
    for (int by = -((periodic >> 1) & 1); by <= ((periodic >> 1) & 1); ++by)
      for (int bz = -((periodic >> 2) & 1); bz <= ((periodic >> 2) & 1); ++bz) {
        if (bx == 0 && by == 0 && bz == 0) continue;
        const Geom<double> g = make_geom(bx * L0, by * L1, bz * L2, h, h);
        Vec3<double> v{0.0, 0.0, 0.0};
        if (!is_w) {
          if (mask & kUF) {
            const Vec3<double> q = apply_uf(g, coef_uf(g, h, h, dom), fv[0], fv[1], fv[2]);
            v.x += q.x; v.y += q.y; v.z += q.z;
          }
          if (mask & kUT) {
            const Vec3<double> q = apply_ut(g, coef_rot(g, h, dom), tv[0], tv[1], tv[2]);
            v.x += q.x; v.y += q.y; v.z += q.z;
          }
        } else {
          if (mask & kWF) {
            const Vec3<double> q = apply_wf(g, coef_rot(g, h, dom), fv[0], fv[1], fv[2]);
            v.x += q.x; v.y += q.y; v.z += q.z;
          }
          if (mask & kWT) {
            const Vec3<double> q = apply_wt(g, coef_wt(g, dom), tv[0], tv[1], tv[2]);
            v.x += q.x; v.y += q.y; v.z += q.z;
          }
        }
        self += comp == 0 ? v.x : (comp == 1 ? v.y : v.z);
      }
  if (!is_w) {
    if (mask & kUF) { Vec3<double> sv = self_uf_dom(dom, h, fv[0], fv[1], fv[2]); self += comp == 0 ? sv.x : (comp == 1 ? sv.y : sv.z); }
    if (mask & kUT) { Vec3<double> sv = self_ut_dom(dom, h, tv[0], tv[1], tv[2]); self += comp == 0 ? sv.x : (comp == 1 ? sv.y : sv.z); }
    vel[k * out_stride + 3 * gi + comp] = (comp == 2 ? pz : 1.0) * B * (sum + self);
  } else {
    if (mask & kWF) { Vec3<double> sv = self_wf_dom(dom, h, fv[0], fv[1], fv[2]); self += comp == 0 ? sv.x : (comp == 1 ? sv.y : sv.z); }
    if (mask & kWT) { Vec3<double> sv = self_wt_dom(dom, h, tv[0], tv[1], tv[2]); self += comp == 0 ? sv.x : (comp == 1 ? sv.y : sv.z); }
    omg[k * out_stride + 3 * gi + comp] = B * inva * (sum + self);
  }
}

// ---------------------------------------------------------------------------
// Launches of the kernels for few blobs (rmw_wall_direct.hip) and for the
// middle sizes (rmw_wall_blocks.hip).
// ---------------------------------------------------------------------------
// One independent suspension of a direct launch.
struct DirectSys {
  int64_t b0, n;        // first blob, blobs
  int64_t item0;        // first workgroup
};

struct DirectParams {
  const double* r;
  const double* f;          // K right-hand sides rhs_stride apart, or null
  const double* t;
  double* vel;              // outputs, out_stride apart, or null
  double* omg;
  int64_t rhs_stride, out_stride;
  double a, inva, c1, c2;
  const DirectSys* table;   // nullptr -> single
  DirectSys single;
  int nsys;
  int periodic;             // bit d set when L_d > 0
  double L[3], iL[3];       // periodic lengths / a and their inverses (0: none)
};

// Targets per workgroup of the direct kernel for these blocks and
// right-hand sides, and the largest number of right-hand sides per launch.
int direct_targets(int mask, int K);
int direct_max_k(int mask, int domain);
void launch_direct(int domain, int mask, int prec, int K, const DirectParams& q, int64_t wgs, hipStream_t st);

// Symmetric kernel on pairs of 64-blob blocks; q counts tiles and work
// items in blocks (MutSys::n_t, MutParams::chunk_blocks).
void launch_blocks(int domain, int mask, int prec, int K, const MutParams& q, int grid, hipStream_t st);

}  // namespace rmw
