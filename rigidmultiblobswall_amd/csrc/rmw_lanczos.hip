// Lanczos square root: c = scale * sqrt+(T) e_1 for the symmetric
// tridiagonal T built by the Lanczos recurrence (FP64, on the device).
//
// Reference: stochastic_forcing/stochastic_forcing.py:208-227 forms the
// (i+1) x (i+1) tridiagonal h every iteration, takes numpy.linalg.eigh,
// replaces negative eigenvalues by 0 and evaluates
//   noise = V^T Q (|z| factor sqrt(lambda) * Q^T e_1).
// Here sqrt(T) e_1 is a quadrature: sqrt(l) = (2/pi) int l / (l + t^2) dt over
// t > 0, and with t = sqrt(M) e^x (M >= every eigenvalue) the trapezoidal rule
// of step h is off by 2 exp(-pi^2 / h) of sqrt(l) for every l >= 0, plus
// sqrt(M) e^-37 from |x| > 37: 320 nodes reach the last bits of a double
// whatever the condition of T.  The nodes are independent tridiagonal solves
// (T + t^2) x = e_1, one per thread: 2 m short steps instead of the ~m^2
// dependent plane rotations of a QL sweep.  l / (l + s) is taken as
// 1 - s / (l + s) for s < M and as T (T + s)^-1 beyond, so that no term loses
// digits.  Error of c in units of |c| against 50 digits, this / eigh: 11 steps
// at condition 1e4 4e-16 / 5e-15, 25 at 1e6 3e-16 / 1e-14, 40 at 1e13
// 1e-14 / 3e-12.  One T of
// 11 steps takes 6 us, of 60 14, of 100 47, of 400 141 (the QL sweeps, bound by
// the latency of their rotations, took 20 us on average over 11 steps with T in
// registers, 8.0 ms at 100 steps and 254 ms at 400 with T in memory).
// A T with an eigenvalue <= 0 (a negative pivot in a solve) or not finite takes
// the eigen-decomposition instead: implicit QL with Wilkinson shifts (Bowdler,
// Martin, Reinsch & Wilkinson, Numer. Math. 11 (1968) 293, the algorithm
// behind EISPACK tql2) by the first wavefront, the scalar recurrence evaluated
// redundantly by all 64 lanes and the rotations applied to the eigenvector
// columns with the lanes spread over rows.
// The kernel returns the coefficient vector c (noise = V c), not the noise
// itself.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <algorithm>
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
// (With d and e in LDS, as tridiag_ql keeps them for larger m, the recurrence
// waits for their reads: 11 steps 65 us instead of 53, 25 314 / 236, 64 1737 / 1265,
// for a T with a negative eigenvalue.)
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

// 1 / d for positive d of ordinary size
__device__ __forceinline__ double reciprocal(double d)
{
  double y = __builtin_amdgcn_rcp(d);
  y = fma(y, fma(-d, y, 1.0), y);
  return fma(y, fma(-d, y, 1.0), y);
}

constexpr int kQuadNodes = 320, kQuadWaves = kQuadNodes / 64;
constexpr double kQuadRange = 37.0;
constexpr double kQuadLow = 0.635203471872816;   // the weights of the first half's nodes, over sqrt(M)
// Nodes taken at a time by `waves` wavefronts, and the row length in which
// their solutions are kept (padded: rows start in different LDS banks).
__host__ __device__ constexpr int quad_row(int waves) { return 64 * waves + 8; }

// H of right-hand side r starts at H + r * h_rhs_stride; Lanczos step i wrote
// alpha_i = H[i * ldh + i] and beta_i = H[i * ldh + i + 1].  test (may be
// null): |c - c_prev|, |c_prev| and the status of every right-hand side, with
// c_prev the m - 1 coefficients that c_out held before.  LDS (dynamic): a, b,
// the sums P and Q (m each), then the solutions x_0 .. x_(m-1) of 64 * waves
// nodes, which with MEM are in the scratch array instead (it holds m^2).
template <bool MEM>
__global__ __launch_bounds__(kQuadNodes) void sqrt_e1_kernel(const double* __restrict__ H, int64_t h_rhs_stride,
                                                             int64_t ldh, int m, int waves,
                                                             const double* __restrict__ scale,
                                                             double* __restrict__ c_out, int64_t c_stride,
                                                             double* __restrict__ zscratch, int* __restrict__ status,
                                                             double* __restrict__ test)
{
  extern __shared__ double sm[];
  __shared__ double s_max[kQuadWaves], s_red[2][kQuadWaves];
  const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  double *const a = sm, *const b = a + m, *const P = b + m, *const Q = P + m;
  double* const Z = MEM ? zscratch + (int64_t)r * m * m : Q + m;
  const double* Hr = H + r * h_rhs_stride;
  double top = 0.0;   // Gershgorin
  bool ok = true;
  for (int i = tid; i < m; i += kQuadNodes) {
    const double* row = Hr + (int64_t)i * ldh + i;
    const double ai = row[0], bi = i + 1 < m ? row[1] : 0.0, bp = i > 0 ? row[-ldh] : 0.0;
    a[i] = ai;
    b[i] = bi;
    P[i] = 0.0;
    Q[i] = 0.0;
    const double g = fabs(ai) + fabs(bi) + fabs(bp);
    ok = ok && g < 1e140;
    top = fmax(top, g);
  }
  for (int o = 32; o > 0; o >>= 1) top = fmax(top, __shfl_xor(top, o, 64));
  if (lane == 0) s_max[wv] = top;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kQuadWaves; ++w) top = fmax(top, s_max[w]);
  ok = ok && top > 1e-140;   // (b^2 and M e^74 stay ordinary numbers)

  constexpr double h = 2.0 * kQuadRange / kQuadNodes;
  const int ns = quad_row(waves);
  for (int n0 = 0; n0 < kQuadNodes; n0 += 64 * waves) {
    const int node = n0 + tid;
    if (wv < waves && node < kQuadNodes) {
      const double t = sqrt(top) * exp((node - 0.5 * (kQuadNodes - 1)) * h);
      const double s = t * t, w = (2.0 / M_PI) * h * t;
      const bool low = node < kQuadNodes / 2;
      double* x = Z + tid;
      // pivots from the last row up, then the solution from the first down
      double inv = 0.0, bi = 0.0;
#pragma unroll 4
      for (int i = m - 1; i >= 0; --i) {
        const double d = fma(-bi * bi, inv, a[i] + s);
        ok = ok && d > 0.0;
        inv = reciprocal(d);
        x[(int64_t)i * ns] = inv;
        bi = i > 0 ? b[i - 1] : 0.0;
      }
      double xi = low ? w * s * inv : w * inv;
      x[0] = xi;
#pragma unroll 4
      for (int i = 1; i < m; ++i) {
        xi = -b[i - 1] * xi * x[(int64_t)i * ns];
        x[(int64_t)i * ns] = xi;
      }
    }
    __syncthreads();
    // sums over the nodes of each half, eight threads each
    const int n1 = n0 + 64 * waves < kQuadNodes ? n0 + 64 * waves : kQuadNodes;
    for (int task = tid >> 3; task < 2 * m; task += kQuadNodes / 8) {
      const int i = task >> 1, half = task & 1;
      const int lo = half ? (n0 > kQuadNodes / 2 ? n0 : kQuadNodes / 2) : n0;
      const int hi = half ? n1 : (n1 < kQuadNodes / 2 ? n1 : kQuadNodes / 2);
      const double* x = Z + (int64_t)i * ns - n0;
      double sum = 0.0;
#pragma unroll 4
      for (int q = lo + (tid & 7); q < hi; q += 8) sum += x[q];
      for (int o = 4; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 8);
      if ((tid & 7) == 0) (half ? Q : P)[i] += sum;
    }
    __syncthreads();
  }
  int fail = 0;
  const bool quad = __syncthreads_and(ok);
  double* const E = m <= 64 && !MEM ? Z : zscratch + (int64_t)r * m * m;   // eigenvectors
  if (!quad) {
    double *d = P, *e = Q;
    for (int idx = tid; idx < m * m; idx += kQuadNodes) E[idx] = (idx % (m + 1) == 0) ? 1.0 : 0.0;
    for (int i = tid; i < m; i += kQuadNodes) { d[i] = a[i]; e[i] = b[i]; }
    __syncthreads();
    if (wv == 0) {
      if (m <= 64 && !MEM) {
        double dv = lane < m ? d[lane] : 0.0, ev = lane < m ? e[lane] : 0.0;
        fail = tridiag_ql_lanes(m, dv, ev, E);
        if (lane < m) d[lane] = dv;
      } else {
        fail = tridiag_ql(m, d, e, E);
      }
    }
    __syncthreads();
    // sqrt+(lambda) times the first components, which row 0 holds
    for (int k = tid; k < m; k += kQuadNodes) d[k] = (d[k] > 0.0 ? sqrt(d[k]) : 0.0) * E[(int64_t)k * m];
    __syncthreads();
  }
  const double sc = scale[r], first = kQuadLow * sqrt(top);
  double diff = 0.0, prev = 0.0;
  for (int j = tid; j < m; j += kQuadNodes) {
    double acc;
    if (quad) {   // e_1 sum(w) - sum(w s x) over s < M, + T sum(w x) over s >= M
      acc = fma(a[j], Q[j], (j == 0 ? first : 0.0) - P[j]);
      if (j > 0) acc = fma(b[j - 1], Q[j - 1], acc);
      if (j + 1 < m) acc = fma(b[j], Q[j + 1], acc);
    } else {
      acc = 0.0;
#pragma unroll 4
      for (int k = 0; k < m; ++k) acc += E[(int64_t)k * m + j] * P[k];
    }
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
    if (lane == 0) { s_red[0][wv] = diff; s_red[1][wv] = prev; }
    __syncthreads();
    if (tid < 2) {
      double v = s_red[tid][0];
#pragma unroll
      for (int w = 1; w < kQuadWaves; ++w) v += s_red[tid][w];
      test[3 * r + tid] = sqrt(v);
    }
    if (tid == 0) test[3 * r + 2] = (double)fail;
  }
  if (tid == 0 && status) status[r] = fail;
}

static void launch_sqrt_e1(const double* H, int64_t h_rhs_stride, int64_t ldh, int m, int k, const double* scale,
                           double* c_out, int64_t c_stride, double* scratch, size_t scratch_doubles, int* status,
                           double* test, hipStream_t st)
{
  RMW_REQUIRE(m >= 1 && m <= kMaxLanczos && k >= 1, "bad sizes");
  RMW_REQUIRE(ldh >= m + 1 && c_stride >= m, "bad strides");
  RMW_REQUIRE(scratch && scratch_doubles >= (size_t)k * m * m, "scratch too small");
  // as many nodes at a time as their solutions fit into LDS (all up to 60
  // steps, 64 up to 266), then into the scratch array's m doubles per row
  constexpr int kLdsDoubles = 159 * 1024 / 8;
  int waves = kQuadWaves;
  while (waves > 0 && (4 + quad_row(waves)) * m > kLdsDoubles) --waves;
  const bool mem = waves == 0;
  if (mem) waves = std::min(kQuadWaves, (m - 8) / 64);
  const size_t lds = sizeof(double) * (size_t)m * (4 + (mem ? 0 : quad_row(waves)));
  const dim3 g(k), bl(kQuadNodes);
  if (mem) {
    hipLaunchKernelGGL(sqrt_e1_kernel<true>, g, bl, lds, st, H, h_rhs_stride, ldh, m, waves, scale, c_out, c_stride,
                       scratch, status, test);
  } else {
    if (lds > 64 * 1024)
      RMW_CHECK_HIP(hipFuncSetAttribute((const void*)sqrt_e1_kernel<false>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, kLdsDoubles * 8));
    hipLaunchKernelGGL(sqrt_e1_kernel<false>, g, bl, lds, st, H, h_rhs_stride, ldh, m, waves, scale, c_out, c_stride,
                       scratch, status, test);
  }
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
    launch_sqrt_e1(H, h_rhs_stride, ldh, m, k, scale, c_out, c_stride, scratch, scratch_doubles, status, nullptr,
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
    launch_sqrt_e1(H, h_rhs_stride, ldh, m, k, scale, c_out, c_stride, scratch, scratch_doubles, nullptr, test,
                   (hipStream_t)stream);
  });
}
