// Per-target accumulator policies of the pair kernels and the minimum-image
// shift count, shared by the kernel files.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/rmw_hip.h"

namespace rmw {

// Per-target accumulator policies.
template <int ACC> struct Acc;
template <> struct Acc<RMW_PREC_F32_F64ACC> {
  static constexpr bool kChain = false;
  double v = 0.0;
  __device__ __forceinline__ void add(float x) { v += (double)x; }
  __device__ __forceinline__ void flush() {}
  __device__ __forceinline__ double get() const { return v; }
};
// kChain: the running sum may seed a product's FMA chain (run()), which
// saves the separate add of each term.
template <> struct Acc<RMW_PREC_F32_BLOCKED> {
  static constexpr bool kChain = true;
  double v = 0.0;
  float p = 0.0f;
  __device__ __forceinline__ void add(float x) { p += x; }
  __device__ __forceinline__ float& run() { return p; }
  __device__ __forceinline__ void flush()
  {
    v += (double)p;
    p = 0.0f;
  }
  __device__ __forceinline__ double get() const { return v + (double)p; }
};
template <> struct Acc<RMW_PREC_F32_KAHAN> {
  static constexpr bool kChain = false;
  float s = 0.0f, c = 0.0f;
  __device__ __forceinline__ void add(float x)
  {
    float y = x - c;
    float t = s + y;
    c = (t - s) - y;
    s = t;
  }
  __device__ __forceinline__ void flush() {}
  __device__ __forceinline__ double get() const { return (double)s - (double)c; }
};
template <> struct Acc<RMW_PREC_F64> {
  static constexpr bool kChain = true;
  double v = 0.0;
  __device__ __forceinline__ void add(double x) { v += x; }
  __device__ __forceinline__ double& run() { return v; }
  __device__ __forceinline__ void flush() {}
  __device__ __forceinline__ double get() const { return v; }
};

// The seed of a chained product and the taking of its result (C), or a plain add.
template <bool C, typename T, class A>
__device__ __forceinline__ T chain_seed(A& a)
{
  if constexpr (C) return a.run();
  else return T(0);
}
template <bool C, typename T, class A>
__device__ __forceinline__ void chain_take(A& a, T x)
{
  if constexpr (C) a.run() = x;
  else a.add(x);
}

constexpr int kSub = 16;  // sources per FP32 sub-sum in the blocked mode

// Minimum-image shift count of mobility_numba.py:184-193: int(d/L + 0.5 sign(d)).
__device__ __forceinline__ double image_count(double d, double L)
{
  double s = (double)((d > 0.0) - (d < 0.0));
  return trunc(d / L + 0.5 * s);
}

// The same number without the division, iL = 1 / L rounded: d * iL is off by
// less than 1e-10 up to 1e5 boxes, which the integer part hides unless it is
// next to an integer; those, larger ones and non-finite ones are divided.
__device__ __forceinline__ double image_count(double d, double L, double iL)
{
  const double v = fma(d, iL, d > 0.0 ? 0.5 : (d < 0.0 ? -0.5 : 0.0));
  const bool safe = fabs(v - rint(v)) > 1e-9 && fabs(v) < 1e5;
  return __builtin_expect(safe, 1) ? trunc(v) : image_count(d, L);
}

// f(dx, dy, dz, central) for the minimum image of d (FP64) and its neighbours
// in the periodic directions (bits of `periodic`); central: the minimum image.
template <typename R, typename F>
__device__ __forceinline__ void each_image(double ddx, double ddy, double ddz, int periodic, const double (&L)[3],
                                           const double (&iL)[3], F&& f)
{
  const int nx = periodic & 1, ny = (periodic >> 1) & 1, nz = (periodic >> 2) & 1;
  auto shifted = [](double d, int b, double len) { return (R)(d + (b < 0 ? -len : (b > 0 ? len : 0.0))); };
  if (nx) ddx -= image_count(ddx, L[0], iL[0]) * L[0];
  if (ny) ddy -= image_count(ddy, L[1], iL[1]) * L[1];
  if (nz) ddz -= image_count(ddz, L[2], iL[2]) * L[2];
  for (int bz = -nz; bz <= nz; ++bz) {
    const R dz = shifted(ddz, bz, L[2]);
    for (int bx = -nx; bx <= nx; ++bx) {
      const R dx = shifted(ddx, bx, L[0]);
      for (int by = -ny; by <= ny; ++by)
        f(dx, shifted(ddy, by, L[1]), dz, bx == 0 && by == 0 && bz == 0);
    }
  }
}

// Sum over the 64 lanes, in every lane: within the rows of 16 by DPP moves
// (a shuffle through LDS takes some 60 cycles per step and half of a double).
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v)
{
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
  return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double row_sum(double v)   // over rows of 16 lanes
{
  v = dpp_add<0xB1>(v);    // quad_perm 1 0 3 2
  v = dpp_add<0x4E>(v);    // quad_perm 2 3 0 1
  v = dpp_add<0x141>(v);   // row_half_mirror
  return dpp_add<0x140>(v);   // row_mirror
}
__device__ __forceinline__ double wave_sum(double v)
{
  v = row_sum(v);
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

}  // namespace rmw
