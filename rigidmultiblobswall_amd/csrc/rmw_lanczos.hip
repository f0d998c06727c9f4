// Lanczos square root: c = scale * sqrt+(T) e_1 for the symmetric
// tridiagonal T built by the Lanczos recurrence (FP64, on the device).
//
// Reference: stochastic_forcing/stochastic_forcing.py:208-227 forms the
// (i+1) x (i+1) tridiagonal h every iteration, takes numpy.linalg.eigh,
// replaces negative eigenvalues by 0 and evaluates
//   noise = V^T Q (|z| factor sqrt(lambda) * Q^T e_1).
// Here the eigen-decomposition is the implicit QL method with Wilkinson
// shifts (Bowdler, Martin, Reinsch & Wilkinson, Numer. Math. 11 (1968) 293,
// the algorithm behind EISPACK tql2), run by one wavefront per right-hand
// side: the scalar recurrence is evaluated redundantly by all 64 lanes, each
// plane rotation is applied to the eigenvector columns with the lanes spread
// over rows.  The kernel is one dependent chain, so it is bound by the latency
// of a rotation.  Up to 64 steps the tridiagonal lives in the lanes'
// registers, the search for a negligible off-diagonal is one ballot, the
// eigenvectors are in LDS with their next column read ahead, and
// 1/sqrt(f^2 + g^2) is the refined hardware estimate of the pair terms (with
// all of it in memory, a correctly rounded hypot and two divisions the launch
// took 35 us on average over 11 Lanczos steps, with d and e in LDS 24, now 20).
// The kernel returns the coefficient vector c (noise = V c), not the noise
// itself.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>

#include "rmw_internal.h"
#include "rmw_pair_terms.h"

namespace rmw {

constexpr int kMaxLanczos = 1024;

// Element i (the same for every lane) of a value that lane i holds.
__device__ __forceinline__ double lane_value(double v, int i)
{
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), i),
                          __builtin_amdgcn_readlane(__double2loint(v), i));
}

// 1/sqrt(f^2 + g^2) times f and g, and the root itself; false when it is 0.
__device__ __forceinline__ bool rotation(double f, double g, double& s, double& c, double& rr)
{
  const double h = fma(f, f, g * g);
  if (__builtin_expect(h > 1e-250 && h < 1e250, 1)) {
    const double inv = rsq(h);
    rr = h * inv;
    s = f * inv;
    c = g * inv;
    return true;
  }
  rr = hypot(f, g);
  if (rr == 0.0) return false;
  s = f / rr;
  c = g / rr;
  return true;
}

// sqrt(g^2 + 1)
__device__ __forceinline__ double root1(double g)
{
  const double h = fma(g, g, 1.0);
  return h < 1e250 ? h * rsq(h) : fabs(g);
}

// Eigen-decomposition of the tridiagonal with diagonal d and off-diagonal e
// (lane i holds d_i and e_i), m <= 64: on return lane i holds eigenvalue i,
// and Z (m x m in LDS, column-major, identity on entry) the eigenvectors, row
// `lane` of which only this lane touches.  Returns 1 if it does not converge.
__device__ int tridiag_ql_lanes(int m, double& d, double& e, double* __restrict__ Z)
{
  const int lane = threadIdx.x;
  const bool in = lane < m;
  for (int l = 0; l < m; ++l) {
    for (int iter = 0;; ++iter) {
      // the first negligible off-diagonal from l on
      const double dn = __shfl_down(d, 1, 64);
      const unsigned long long small =
          __ballot(lane >= l && (lane >= m - 1 || fabs(e) <= DBL_EPSILON * (fabs(d) + fabs(dn))));
      const int mm = __builtin_amdgcn_readfirstlane(__ffsll(small) - 1);
      if (mm == l) break;
      if (iter == 60) return 1;
      const double dl = lane_value(d, l), el = lane_value(e, l);
      double g = (lane_value(d, l + 1) - dl) / (2.0 * el);
      double rr = root1(g);
      g = lane_value(d, mm) - dl + el / (g + copysign(rr, g));
      double s = 1.0, c = 1.0, p = 0.0;
      bool deflated = false;
      double z1 = in ? Z[mm * m + lane] : 0.0;
      double a0 = in ? Z[(mm - 1) * m + lane] : 0.0;
      double di1 = lane_value(d, mm);
      int i = mm - 1;
      for (; i >= l; --i) {
        const double ei = lane_value(e, i), di = lane_value(d, i);
        const double next = in && i > l ? Z[(i - 1) * m + lane] : 0.0;
        const double f = s * ei, b = c * ei;
        if (!rotation(f, g, s, c, rr)) {
          if (lane == i + 1) { e = 0.0; d = di1 - p; }
          if (lane == mm) e = 0.0;
          deflated = true;
          break;
        }
        if (lane == i + 1) e = rr;
        g = di1 - p;
        rr = (di - g) * s + 2.0 * c * b;
        p = s * rr;
        if (lane == i + 1) d = g + p;
        g = c * rr - b;
        if (in) Z[(i + 1) * m + lane] = s * a0 + c * z1;
        z1 = c * a0 - s * z1;
        a0 = next;
        di1 = di;
      }
      if (in) Z[(i + 1) * m + lane] = z1;   // the column the sweep stopped at
      if (deflated) continue;
      if (lane == l) { d -= p; e = g; }
      if (lane == mm) e = 0.0;
    }
  }
  return 0;
}

// The same for any m, d and e in LDS and Z in memory (every lane writes the
// same values to d and e and reads its own, so nothing has to be waited for).
__device__ int tridiag_ql(int m, double* d, double* e, double* __restrict__ Z)
{
  const int lane = threadIdx.x;
  for (int l = 0; l < m; ++l) {
    for (int iter = 0;; ++iter) {
      int mm = l;
      for (; mm < m - 1; ++mm) {
        const double dd = fabs(d[mm]) + fabs(d[mm + 1]);
        if (fabs(e[mm]) <= DBL_EPSILON * dd) break;
      }
      if (mm == l) break;
      if (iter == 60) return 1;
      double g = (d[l + 1] - d[l]) / (2.0 * e[l]);
      double rr = root1(g);
      g = d[mm] - d[l] + e[l] / (g + copysign(rr, g));
      double s = 1.0, c = 1.0, p = 0.0;
      bool deflated = false;
      for (int i = mm - 1; i >= l; --i) {
        const double f = s * e[i], b = c * e[i];
        if (!rotation(f, g, s, c, rr)) {
          e[i + 1] = 0.0;
          d[i + 1] -= p;
          e[mm] = 0.0;
          deflated = true;
          break;
        }
        e[i + 1] = rr;
        g = d[i + 1] - p;
        rr = (d[i] - g) * s + 2.0 * c * b;
        p = s * rr;
        d[i + 1] = g + p;
        g = c * rr - b;
        double* zi = Z + (int64_t)i * m;
        double* zi1 = Z + (int64_t)(i + 1) * m;
        for (int row = lane; row < m; row += 64) {
          const double a0 = zi[row], a1 = zi1[row];
          zi1[row] = s * a0 + c * a1;
          zi[row] = c * a0 - s * a1;
        }
      }
      if (deflated) continue;
      d[l] -= p;
      e[l] = g;
      e[mm] = 0.0;
    }
  }
  return 0;
}

// H of right-hand side r starts at H + r * h_rhs_stride; Lanczos step i wrote
// alpha_i = H[i * ldh + i] and beta_i = H[i * ldh + i + 1].  test (may be
// null): |c - c_prev|, |c_prev| and the status of every right-hand side, with
// c_prev the m - 1 coefficients that c_out held before.  LANES: m <= 64, the
// eigenvectors in LDS.
template <bool LANES>
__global__ __launch_bounds__(64) void tridiag_sqrt_e1_kernel(const double* __restrict__ H, int64_t h_rhs_stride,
                                                             int64_t ldh, int m, const double* __restrict__ scale,
                                                             double* __restrict__ c_out, int64_t c_stride,
                                                             double* __restrict__ zscratch, int* __restrict__ status,
                                                             double* __restrict__ test)
{
  extern __shared__ double s_z[];
  __shared__ double d[LANES ? 64 : kMaxLanczos], e[LANES ? 1 : kMaxLanczos];
  const int r = blockIdx.x;
  const int lane = threadIdx.x;
  const double* Hr = H + r * h_rhs_stride;
  double* Z = LANES ? s_z : zscratch + (int64_t)r * m * m;
  for (int idx = lane; idx < m * m; idx += 64) Z[idx] = (idx % (m + 1) == 0) ? 1.0 : 0.0;
  int fail;
  if constexpr (LANES) {
    double dv = lane < m ? Hr[(int64_t)lane * ldh + lane] : 0.0;
    double ev = lane + 1 < m ? Hr[(int64_t)lane * ldh + lane + 1] : 0.0;
    __syncthreads();
    fail = tridiag_ql_lanes(m, dv, ev, Z);
    d[lane] = dv;
  } else {
    for (int i = lane; i < m; i += 64) {
      d[i] = Hr[(int64_t)i * ldh + i];
      e[i] = (i + 1 < m) ? Hr[(int64_t)i * ldh + i + 1] : 0.0;
    }
    __syncthreads();
    fail = tridiag_ql(m, d, e, Z);
  }
  // sqrt+(lambda) times the first components, which lane 0's row holds
  __syncthreads();
  for (int k = lane; k < m; k += 64) {
    const double lam = d[k];
    d[k] = (lam > 0.0 ? sqrt(lam) : 0.0) * Z[(int64_t)k * m];
  }
  __syncthreads();
  const double sc = scale[r];
  double diff = 0.0, prev = 0.0;
  for (int j = lane; j < m; j += 64) {
    double acc = 0.0;
#pragma unroll 4
    for (int k = 0; k < m; ++k) acc += Z[(int64_t)k * m + j] * d[k];
    const double now = sc * acc;
    if (test) {
      const double old = j < m - 1 ? c_out[r * c_stride + j] : 0.0;
      diff = fma(now - old, now - old, diff);
      prev = fma(old, old, prev);
    }
    c_out[r * c_stride + j] = now;
  }
  if (test) {
    for (int o = 32; o > 0; o >>= 1) {
      diff += __shfl_xor(diff, o, 64);
      prev += __shfl_xor(prev, o, 64);
    }
    if (lane == 0) {
      test[3 * r] = sqrt(diff);
      test[3 * r + 1] = sqrt(prev);
      test[3 * r + 2] = (double)fail;
    }
  }
  if (lane == 0 && status) status[r] = fail;
}

static void launch_tridiag(const double* H, int64_t h_rhs_stride, int64_t ldh, int m, int k, const double* scale,
                           double* c_out, int64_t c_stride, double* scratch, size_t scratch_doubles, int* status,
                           double* test, hipStream_t st)
{
  RMW_REQUIRE(m >= 1 && m <= kMaxLanczos && k >= 1, "bad sizes");
  RMW_REQUIRE(ldh >= m + 1 && c_stride >= m, "bad strides");
  RMW_REQUIRE(scratch && scratch_doubles >= (size_t)k * m * m, "scratch too small");
  if (m <= 64)
    hipLaunchKernelGGL(tridiag_sqrt_e1_kernel<true>, dim3(k), dim3(64), (size_t)m * m * sizeof(double), st, H,
                       h_rhs_stride, ldh, m, scale, c_out, c_stride, scratch, status, test);
  else
    hipLaunchKernelGGL(tridiag_sqrt_e1_kernel<false>, dim3(k), dim3(64), 0, st, H, h_rhs_stride, ldh, m, scale, c_out,
                       c_stride, scratch, status, test);
  RMW_CHECK_HIP(hipGetLastError());
}

}  // namespace rmw

using namespace rmw;

extern "C" int rmw_lanczos_scratch_doubles(int m, int k, size_t* doubles)
{
  return guarded([&] {
    RMW_REQUIRE(doubles && m >= 1 && m <= kMaxLanczos && k >= 1, "bad sizes");
    *doubles = (size_t)k * m * m;
  });
}

// c_out[r * c_stride + j] = scale[r] * (sqrt+(T_r) e_1)_j, j < m, for the k
// tridiagonals T_r read from the Lanczos coefficient arrays H (see kernel).
extern "C" int rmw_lanczos_sqrt_coeffs(const double* H, int64_t h_rhs_stride, int64_t ldh, int m, int k,
                                       const double* scale, double* c_out, int64_t c_stride, double* scratch,
                                       size_t scratch_doubles, int* status, void* stream)
{
  return guarded([&] {
    launch_tridiag(H, h_rhs_stride, ldh, m, k, scale, c_out, c_stride, scratch, scratch_doubles, status, nullptr,
                   (hipStream_t)stream);
  });
}

// The same, with the numbers of the Lanczos stop test: on entry c_out holds
// the m - 1 coefficients of the step before; test[3 r ..] = |c - c_prev|,
// |c_prev| (c_prev padded with 0) and the status.
extern "C" int rmw_lanczos_step_coeffs(const double* H, int64_t h_rhs_stride, int64_t ldh, int m, int k,
                                       const double* scale, double* c_out, int64_t c_stride, double* scratch,
                                       size_t scratch_doubles, double* test, void* stream)
{
  return guarded([&] {
    RMW_REQUIRE(test != nullptr, "test is null");
    launch_tridiag(H, h_rhs_stride, ldh, m, k, scale, c_out, c_stride, scratch, scratch_doubles, nullptr, test,
                   (hipStream_t)stream);
  });
}
