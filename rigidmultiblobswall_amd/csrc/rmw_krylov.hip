// FP64 Krylov-space vector kernels for GMRES (Arnoldi with classical
// Gram-Schmidt and one re-orthogonalisation, CGS2) and Lanczos.
//
// Vectors are float64, length n; a basis V is stored as nvec rows of
// stride ldv.  Every reduction is two-pass with a fixed order (block
// partials, then one thread per output summing the partials), so results
// are bit-reproducible run to run.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "rmw_accum.h"
#include "rmw_internal.h"

namespace rmw {

constexpr int kKBlock = 256;
constexpr int kMaxDotBlocks = 512;
constexpr int kMaxVec = 1024;

// partial[j * G + g] = sum over the g-th slice of V_j . w  (long vectors:
// each block walks a slice of (n + G - 1) / G elements once per vector)
__global__ __launch_bounds__(kKBlock) void dot_many_partial(const double* __restrict__ V, int64_t ldv, int nvec,
                                                            const double* __restrict__ w, int64_t n,
                                                            double* __restrict__ partial)
{
  __shared__ double red[kKBlock / 64];
  const int G = gridDim.x;
  const int64_t slice = (n + G - 1) / G;
  const int64_t b0 = slice * blockIdx.x;
  const int64_t b1 = b0 + slice < n ? b0 + slice : n;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int j = 0; j < nvec; ++j) {
    const double* v = V + (int64_t)j * ldv;
    double acc = 0.0;
    for (int64_t i = b0 + threadIdx.x; i < b1; i += blockDim.x) acc += v[i] * w[i];
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
    if (lane == 0) red[wv] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
      double s = 0.0;
      for (int k = 0; k < (int)(blockDim.x >> 6); ++k) s += red[k];
      partial[(int64_t)j * G + blockIdx.x] = s;
    }
    __syncthreads();
  }
}

// Same partials when every block owns one slice of kKBlock * E elements:
// the slice of w stays in registers across the vectors, each vector's
// wave sums go to LDS and one barrier per group of 64 vectors publishes
// them (fixed summation order, as above).
constexpr int kDotGroup = 64;

template <int E>
__global__ __launch_bounds__(kKBlock) void dot_many_partial_reg(const double* __restrict__ V, int64_t ldv, int nvec,
                                                                const double* __restrict__ w, int64_t n,
                                                                double* __restrict__ partial)
{
  __shared__ double red[kDotGroup][kKBlock / 64];
  const int G = gridDim.x;
  const int64_t base = (int64_t)blockIdx.x * (kKBlock * E) + threadIdx.x;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  double wr[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int64_t i = base + (int64_t)e * kKBlock;
    wr[e] = i < n ? w[i] : 0.0;
  }
  for (int j0 = 0; j0 < nvec; j0 += kDotGroup) {
    const int jn = nvec - j0 < kDotGroup ? nvec - j0 : kDotGroup;
    for (int jj = 0; jj < jn; ++jj) {
      const double* v = V + (int64_t)(j0 + jj) * ldv;
      double acc = 0.0;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int64_t i = base + (int64_t)e * kKBlock;
        if (i < n) acc = fma(v[i], wr[e], acc);
      }
      for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
      if (lane == 0) red[jj][wv] = acc;
    }
    __syncthreads();
    if ((int)threadIdx.x < jn) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < kKBlock / 64; ++k) s += red[threadIdx.x][k];
      partial[(int64_t)(j0 + threadIdx.x) * G + blockIdx.x] = s;
    }
    __syncthreads();
  }
}

// out[j] = sum_g partial[j * G + g] (sqrt when sqrt_out; + out[j] when
// accumulate): one wavefront per output, lanes stride the partials, then a
// fixed shuffle tree.
__global__ __launch_bounds__(64) void dot_many_final(const double* __restrict__ partial, int G, int nvec,
                                                     double* __restrict__ out, int accumulate, int sqrt_out)
{
  const int j = blockIdx.x;
  if (j >= nvec) return;
  const double* p = partial + (int64_t)j * G;
  double s = 0.0;
  for (int g = threadIdx.x; g < G; g += 64) s += p[g];
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if (threadIdx.x == 0) {
    if (sqrt_out) s = sqrt(s);
    out[j] = accumulate ? out[j] + s : s;
  }
}

// w -= sum_j coef[j] V_j     (coef on the device)
__global__ __launch_bounds__(kKBlock) void sub_combination(const double* __restrict__ V, int64_t ldv, int nvec,
                                                           const double* __restrict__ coef,
                                                           double* __restrict__ w, int64_t n)
{
  __shared__ double c[kMaxVec];
  for (int j = threadIdx.x; j < nvec; j += blockDim.x) c[j] = coef[j];
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    double s = w[i];
    for (int j = 0; j < nvec; ++j) s -= c[j] * V[(int64_t)j * ldv + i];
    w[i] = s;
  }
}

// y = sum_j coef[j] V_j (+ y when accumulate)
__global__ __launch_bounds__(kKBlock) void combination(const double* __restrict__ V, int64_t ldv, int nvec,
                                                       const double* __restrict__ coef, double* __restrict__ y,
                                                       int64_t n, int accumulate)
{
  __shared__ double c[kMaxVec];
  for (int j = threadIdx.x; j < nvec; j += blockDim.x) c[j] = coef[j];
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    double s = accumulate ? y[i] : 0.0;
    for (int j = 0; j < nvec; ++j) s += c[j] * V[(int64_t)j * ldv + i];
    y[i] = s;
  }
}

// y = alpha x + beta y, alpha optionally 1/(*dev_div) (0 -> unit e_0)
__global__ void axpby_kernel(double alpha, const double* __restrict__ x, double beta, double* __restrict__ y,
                             int64_t n, const double* __restrict__ dev_div)
{
  double al = alpha;
  if (dev_div) {
    const double d = *dev_div;
    al = d > 0.0 ? alpha / d : 0.0;
  }
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const double xv = (dev_div && !(*dev_div > 0.0)) ? (i == 0 ? 1.0 : 0.0) : al * x[i];
    y[i] = beta == 0.0 ? xv : xv + beta * y[i];
  }
}

// ---------------------------------------------------------------------------
// One Arnoldi step by CGS2 in four launches, for k independent bases at once
// (blockIdx.y).  Every block owns one slice of kKBlock * E elements, the same
// in all four, and adds the blocks' partial sums of the launch before it by
// itself (a few thousand doubles from L2, in the order of dot_many_final), so
// no launch in between turns partial sums into coefficients.  The chain of
// small launches, not the vectors, was the time of the step: ten launches
// took 35 us at n = 15000 with 11 vectors (13 MB read, 2.7 us at the rate of
// a copy), these 17, and 16 with the first vectors loaded before anything is
// waited for and the sums taken by DPP moves (13200 elements, 8 vectors on
// average: 19.6 before, 16).
// ---------------------------------------------------------------------------
struct ArnoldiParams {
  double* V;            // basis r at V + r * v_rhs, vectors ldv apart
  int64_t ldv, v_rhs;
  double* w;            // candidate r at w + r * w_rhs
  int64_t w_rhs, n;
  double* h;            // coefficients r at h + r * h_rhs
  int64_t h_rhs;
  double* h_host;       // pinned host copy of h of basis 0, or null
  double* part;         // per basis: part1 [m][G], part2 [m][G], part3 [G]
  int64_t part_rhs;
  int m;                // vectors in the basis
};

// coef[j] = sum_g part[j * G + g], j < m: sixteen threads per j.
__device__ __forceinline__ void block_coefs(const double* __restrict__ part, int G, int m, double* coef)
{
  const int sub = threadIdx.x & 15;
  for (int j = threadIdx.x >> 4; j < m; j += kKBlock / 16) {
    double s = 0.0;
#pragma unroll 4
    for (int g = sub; g < G; g += 16) s += part[(int64_t)j * G + g];
    s = row_sum(s);
    if (sub == 0) coef[j] = s;
  }
  __syncthreads();
}

// part[j * G + block] = V_j . w over this block's slice, w in registers; the
// first held_vectors(E) vectors' slices are in registers too (v).
constexpr int held_vectors(int E) { return 16 / E; }   // 32 registers' worth
template <int E>
__device__ __forceinline__ void block_dots(const double* __restrict__ V, int64_t ldv, int m, const double (&wr)[E],
                                           const double (&v)[held_vectors(E)][E], int64_t base, int64_t n,
                                           double* __restrict__ part, int G)
{
  constexpr int kHeld = held_vectors(E);
  __shared__ double red[kDotGroup][kKBlock / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  auto put = [&](int jj, double acc) {
    acc = wave_sum(acc);
    if (lane == 0) red[jj][wv] = acc;
  };
  for (int j0 = 0; j0 < m; j0 += kDotGroup) {
    const int jn = m - j0 < kDotGroup ? m - j0 : kDotGroup;
    int jj = 0;
    if (j0 == 0) {
#pragma unroll
      for (int q = 0; q < kHeld; ++q)
        if (q < jn) {
          double acc = 0.0;
#pragma unroll
          for (int e = 0; e < E; ++e) acc = fma(v[q][e], wr[e], acc);
          put(q, acc);
        }
      jj = kHeld;
    }
#pragma unroll 4
    for (; jj < jn; ++jj) {
      const double* vj = V + (int64_t)(j0 + jj) * ldv;
      double acc = 0.0;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int64_t i = base + (int64_t)e * kKBlock;
        if (i < n) acc = fma(vj[i], wr[e], acc);
      }
      put(jj, acc);
    }
    __syncthreads();
    if ((int)threadIdx.x < jn) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < kKBlock / 64; ++k) s += red[threadIdx.x][k];
      part[(int64_t)(j0 + threadIdx.x) * G + blockIdx.x] = s;
    }
    __syncthreads();
  }
}

// PASS 0: part1 = V . w.  PASS 1: w -= V c1, h = c1, part2 = V . w.  PASS 2:
// w -= V c2, h += c2, part3 = w . w.  PASS 3: V_m = w / |w| (e_0 if 0),
// h_m = |w|.
template <int E, int PASS>
__global__ __launch_bounds__(kKBlock) void arnoldi_pass(ArnoldiParams p)
{
  __shared__ double coef[kMaxVec];
  const int G = gridDim.x, r = blockIdx.y;
  double* V = p.V + r * p.v_rhs;
  double* w = p.w + r * p.w_rhs;
  double* h = p.h + r * p.h_rhs;
  double* part1 = p.part + r * p.part_rhs;
  double* part2 = part1 + (int64_t)p.m * G;
  double* part3 = part2 + (int64_t)p.m * G;
  const int64_t base = (int64_t)blockIdx.x * (kKBlock * E) + threadIdx.x;
  double wr[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int64_t i = base + (int64_t)e * kKBlock;
    wr[e] = i < p.n ? w[i] : 0.0;
  }
  // the slices of the first vectors, loaded before anything has to be waited for
  constexpr int kHeld = held_vectors(E);
  double held[PASS < 3 ? kHeld : 1][E];
  if constexpr (PASS < 3) {
#pragma unroll
    for (int j = 0; j < kHeld; ++j)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int64_t i = base + (int64_t)e * kKBlock;
        held[j][e] = j < p.m && i < p.n ? V[(int64_t)j * p.ldv + i] : 0.0;
      }
  }
  if constexpr (PASS == 0) {
    block_dots<E>(V, p.ldv, p.m, wr, held, base, p.n, part1, G);
  } else if constexpr (PASS == 3) {
    // (every wave by itself, one load each up to 64 blocks)
    double sq = 0.0;
    for (int g = threadIdx.x & 63; g < G; g += 64) sq += part3[g];
    const double norm = sqrt(wave_sum(sq));
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      h[p.m] = norm;
      if (p.h_host) p.h_host[p.m] = norm;
    }
    const double al = norm > 0.0 ? 1.0 / norm : 0.0;
    double* v = V + (int64_t)p.m * p.ldv;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int64_t i = base + (int64_t)e * kKBlock;
      if (i < p.n) v[i] = norm > 0.0 ? al * wr[e] : (i == 0 ? 1.0 : 0.0);
    }
  } else {
    block_coefs(PASS == 1 ? part1 : part2, G, p.m, coef);
    if (blockIdx.x == 0)
      for (int j = threadIdx.x; j < p.m; j += kKBlock) {
        const double v = PASS == 1 ? coef[j] : h[j] + coef[j];
        h[j] = v;
        if (PASS == 2 && p.h_host) p.h_host[j] = v;
      }
#pragma unroll
    for (int j = 0; j < kHeld; ++j)
      if (j < p.m) {
#pragma unroll
        for (int e = 0; e < E; ++e) wr[e] -= coef[j] * held[j][e];
      }
#pragma unroll 4
    for (int j = kHeld; j < p.m; ++j) {
      const double* v = V + (int64_t)j * p.ldv;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int64_t i = base + (int64_t)e * kKBlock;
        if (i < p.n) wr[e] -= coef[j] * v[i];
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int64_t i = base + (int64_t)e * kKBlock;
      if (i < p.n) w[i] = wr[e];
    }
    if constexpr (PASS == 1) {
      block_dots<E>(V, p.ldv, p.m, wr, held, base, p.n, part2, G);
    } else {
      __shared__ double red[kKBlock / 64];
      double acc = 0.0;
#pragma unroll
      for (int e = 0; e < E; ++e) acc = fma(wr[e], wr[e], acc);
      acc = wave_sum(acc);
      if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
      __syncthreads();
      if (threadIdx.x == 0) part3[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
    }
  }
}

template <int E>
static void launch_arnoldi(const ArnoldiParams& p, int G, int k, hipStream_t st)
{
  const dim3 g(G, k), b(kKBlock);
  hipLaunchKernelGGL((arnoldi_pass<E, 0>), g, b, 0, st, p);
  hipLaunchKernelGGL((arnoldi_pass<E, 1>), g, b, 0, st, p);
  hipLaunchKernelGGL((arnoldi_pass<E, 2>), g, b, 0, st, p);
  hipLaunchKernelGGL((arnoldi_pass<E, 3>), g, b, 0, st, p);
}

// h[0..j] = h1 + h2 (CGS2 coefficients)
__global__ void add_vec(const double* __restrict__ a, double* __restrict__ b, int m)
{
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < m) b[j] += a[j];
}

// Dot-product launch: elements per thread E of the register-slice kernel
// (0: the slice-walking kernel) and the number of blocks G <= kMaxDotBlocks.
struct DotLaunch {
  int E, G;
};

static DotLaunch dot_launch(int64_t n)
{
  const DeviceProps& dp = device_props();
  // aim for about two blocks per CU with the fewest elements per thread
  const int64_t want = std::min<int64_t>(kMaxDotBlocks, 2 * (int64_t)dp.cu_count);
  for (int E : {1, 2, 4, 8}) {
    const int64_t g = (n + (int64_t)kKBlock * E - 1) / ((int64_t)kKBlock * E);
    if (g <= want || (E == 8 && g <= kMaxDotBlocks)) return {E, (int)std::max<int64_t>(1, g)};
  }
  int64_t g = (n + 4 * kKBlock - 1) / (4 * kKBlock);
  return {0, (int)std::max<int64_t>(1, std::min<int64_t>(g, kMaxDotBlocks))};
}

static void launch_dot_partial(const DotLaunch& L, hipStream_t st, const double* V, int64_t ldv, int nvec,
                               const double* w, int64_t n, double* partial)
{
  switch (L.E) {
    case 1: hipLaunchKernelGGL(dot_many_partial_reg<1>, dim3(L.G), dim3(kKBlock), 0, st, V, ldv, nvec, w, n, partial); break;
    case 2: hipLaunchKernelGGL(dot_many_partial_reg<2>, dim3(L.G), dim3(kKBlock), 0, st, V, ldv, nvec, w, n, partial); break;
    case 4: hipLaunchKernelGGL(dot_many_partial_reg<4>, dim3(L.G), dim3(kKBlock), 0, st, V, ldv, nvec, w, n, partial); break;
    case 8: hipLaunchKernelGGL(dot_many_partial_reg<8>, dim3(L.G), dim3(kKBlock), 0, st, V, ldv, nvec, w, n, partial); break;
    default: hipLaunchKernelGGL(dot_many_partial, dim3(L.G), dim3(kKBlock), 0, st, V, ldv, nvec, w, n, partial);
  }
}

static void launch_dot_final(hipStream_t st, const double* partial, int G, int nvec, double* out, int accumulate,
                             int sqrt_out)
{
  hipLaunchKernelGGL(dot_many_final, dim3(nvec), dim3(64), 0, st, partial, G, nvec, out, accumulate, sqrt_out);
}

static int stream_blocks(int64_t n)
{
  const DeviceProps& dp = device_props();
  int64_t g = (n + kKBlock - 1) / kKBlock;
  return (int)std::max<int64_t>(1, std::min<int64_t>(g, 8 * (int64_t)dp.cu_count));
}

}  // namespace rmw

using namespace rmw;

extern "C" int rmw_krylov_workspace_size(int64_t n, int max_vectors, size_t* bytes)
{
  return guarded([&] {
    RMW_REQUIRE(bytes && n >= 0 && max_vectors >= 1 && max_vectors <= kMaxVec, "bad arguments");
    // two sets of partial sums of max_vectors and one of a norm (rmw_arnoldi_cgs2)
    *bytes = align_up((size_t)kMaxDotBlocks * (2 * (size_t)max_vectors + 1) * sizeof(double)) +
             align_up(kMaxVec * sizeof(double));
  });
}

// out[j] = V_j . w for j < nvec (device out); with sqrt_out, out[j] = sqrt(...)
extern "C" int rmw_dot_many(const double* V, int64_t ldv, int nvec, const double* w, int64_t n, double* out,
                            int sqrt_out, void* workspace, size_t workspace_bytes, void* stream)
{
  return guarded([&] {
    RMW_REQUIRE(nvec >= 1 && nvec <= kMaxVec && n >= 0, "bad sizes");
    const DotLaunch L = dot_launch(n);
    RMW_REQUIRE(workspace_bytes >= (size_t)L.G * nvec * sizeof(double), "workspace too small");
    hipStream_t st = (hipStream_t)stream;
    double* partial = (double*)workspace;
    launch_dot_partial(L, st, V, ldv, nvec, w, n, partial);
    launch_dot_final(st, partial, L.G, nvec, out, 0, sqrt_out);
    RMW_CHECK_HIP(hipGetLastError());
  });
}

// w -= V[0..nvec) coef   (coef on the device)
extern "C" int rmw_sub_combination(const double* V, int64_t ldv, int nvec, const double* coef, double* w,
                                   int64_t n, void* stream)
{
  return guarded([&] {
    RMW_REQUIRE(nvec >= 1 && nvec <= kMaxVec, "bad nvec");
    hipLaunchKernelGGL(sub_combination, dim3(stream_blocks(n)), dim3(kKBlock), 0, (hipStream_t)stream, V, ldv, nvec,
                       coef, w, n);
    RMW_CHECK_HIP(hipGetLastError());
  });
}

// y = V[0..nvec) coef (+ y if accumulate)
extern "C" int rmw_combination(const double* V, int64_t ldv, int nvec, const double* coef, double* y, int64_t n,
                               int accumulate, void* stream)
{
  return guarded([&] {
    RMW_REQUIRE(nvec >= 1 && nvec <= kMaxVec, "bad nvec");
    hipLaunchKernelGGL(combination, dim3(stream_blocks(n)), dim3(kKBlock), 0, (hipStream_t)stream, V, ldv, nvec,
                       coef, y, n, accumulate);
    RMW_CHECK_HIP(hipGetLastError());
  });
}

// y = alpha x + beta y; when div is non-null alpha is divided by *div
// (device scalar; a zero divisor writes the unit vector e_0 instead).
extern "C" int rmw_axpby(double alpha, const double* x, double beta, double* y, int64_t n, const double* div,
                         void* stream)
{
  return guarded([&] {
    hipLaunchKernelGGL(axpby_kernel, dim3(stream_blocks(n)), dim3(kKBlock), 0, (hipStream_t)stream, alpha, x, beta,
                       y, n, div);
    RMW_CHECK_HIP(hipGetLastError());
  });
}

// Partial sums that every block adds up by itself, at most: beyond (a basis of
// many long vectors) turning them into coefficients once is cheaper.
constexpr int64_t kSelfSums = 32768;
// m^2 n up to which the four launches are taken for one basis of m vectors: they
// save some 16 us of launches, but a block's dot products follow one another, so
// long bases go faster through the separate launches.  Four launches / separate,
// us: n = 15000 58 / 65 at m = 60, 97 / 98 at 100, 162 / 151 at 150; 60000 58 / 66
// at 45, 86 / 86 at 60, 124 / 115 at 80; 200000 55 / 69 at 20, 86 / 91 at 30,
// 131 / 124 at 45; 1000000 59 / 69 at 5, 128 / 122 at 12, 313 / 253 at 30.
// Several bases share the four launches, and the separate ones are made for each
// in turn (four bases of 1000000: 654 / 833 at m = 20).
constexpr double kFusedSize = 1.2e8;

// One CGS2 step of one basis in the launches of the separate operations.
static void arnoldi_separate(const DotLaunch& L, hipStream_t st, double* V, int64_t ldv, int m, double* w, int64_t n,
                             double* h, double* hscratch, double* partial)
{
  const int sb = stream_blocks(n);
  // pass 1
  launch_dot_partial(L, st, V, ldv, m, w, n, partial);
  launch_dot_final(st, partial, L.G, m, h, 0, 0);
  hipLaunchKernelGGL(sub_combination, dim3(sb), dim3(kKBlock), 0, st, V, ldv, m, h, w, n);
  // pass 2 (re-orthogonalisation)
  launch_dot_partial(L, st, V, ldv, m, w, n, partial);
  launch_dot_final(st, partial, L.G, m, hscratch, 0, 0);
  hipLaunchKernelGGL(sub_combination, dim3(sb), dim3(kKBlock), 0, st, V, ldv, m, hscratch, w, n);
  hipLaunchKernelGGL(add_vec, dim3((m + 63) / 64), dim3(64), 0, st, hscratch, h, m);
  // norm and normalisation
  launch_dot_partial(L, st, w, (int64_t)0, 1, w, n, partial);
  launch_dot_final(st, partial, L.G, 1, h + m, 0, 1);
  hipLaunchKernelGGL(axpby_kernel, dim3(sb), dim3(kKBlock), 0, st, 1.0, w, 0.0, V + (int64_t)m * ldv, n,
                     (const double*)(h + m));
}

static void arnoldi_batch(double* V, int64_t ldv, int64_t v_rhs, int j, int k, double* w, int64_t w_rhs, int64_t n,
                          double* h, int64_t h_rhs, double* hscratch, void* workspace, size_t workspace_bytes,
                          hipStream_t st, double* h_host = nullptr)
{
  const int m = j + 1;
  RMW_REQUIRE(m >= 1 && m + 1 <= kMaxVec, "bad Arnoldi index");
  RMW_REQUIRE(k >= 1 && k <= 65535, "bad number of bases");
  const DotLaunch L = dot_launch(n);
  RMW_REQUIRE(workspace_bytes >= (size_t)L.G * (m + 1) * sizeof(double), "workspace too small");
  const int64_t per = (int64_t)L.G * (2 * m + 1);
  // as many bases per launch as the workspace has partial sums for
  const int fit = (int)std::min<int64_t>(k, (int64_t)(workspace_bytes / sizeof(double)) / per);
  if (L.E > 0 && (int64_t)L.G * m <= kSelfSums && fit > 0 &&
      (double)m * m * (double)n <= kFusedSize * (double)fit * fit) {
    for (int r0 = 0; r0 < k; r0 += fit) {
      ArnoldiParams p{V + r0 * v_rhs, ldv, v_rhs, w + r0 * w_rhs, w_rhs, n, h + r0 * h_rhs, h_rhs,
                      h_host, (double*)workspace, per, m};
      const int kk = std::min(fit, k - r0);
      switch (L.E) {
        case 1: launch_arnoldi<1>(p, L.G, kk, st); break;
        case 2: launch_arnoldi<2>(p, L.G, kk, st); break;
        case 4: launch_arnoldi<4>(p, L.G, kk, st); break;
        default: launch_arnoldi<8>(p, L.G, kk, st); break;
      }
    }
  } else {
    for (int r = 0; r < k; ++r)
      arnoldi_separate(L, st, V + r * v_rhs, ldv, m, w + r * w_rhs, n, h + r * h_rhs, hscratch, (double*)workspace);
    if (h_host) RMW_CHECK_HIP(hipMemcpyAsync(h_host, h, (m + 1) * sizeof(double), hipMemcpyDeviceToHost, st));
  }
  RMW_CHECK_HIP(hipGetLastError());
}

// Arnoldi step with CGS2: given basis V[0..j] (j+1 vectors, stride ldv) and
// w, orthogonalise w against the basis twice, store the j+1 coefficients in
// h[0..j], ||w|| in h[j+1] and w/||w|| in V[j+1] (e_0 if ||w|| = 0).
// h and hscratch are device arrays of >= j+2 doubles.
extern "C" int rmw_arnoldi_cgs2(double* V, int64_t ldv, int j, double* w, int64_t n, double* h, double* hscratch,
                                void* workspace, size_t workspace_bytes, void* stream)
{
  return guarded([&] {
    arnoldi_batch(V, ldv, 0, j, 1, w, 0, n, h, 0, hscratch, workspace, workspace_bytes, (hipStream_t)stream);
  });
}

// rmw_arnoldi_cgs2, also leaving h[0..j+1] in pinned host memory, where it may
// be read once the stream has been waited for: no copy behind the kernels.
extern "C" int rmw_arnoldi_cgs2_host(double* V, int64_t ldv, int j, double* w, int64_t n, double* h, double* h_host,
                                     double* hscratch, void* workspace, size_t workspace_bytes, void* stream)
{
  return guarded([&] {
    RMW_REQUIRE(h_host != nullptr, "h_host is null");
    arnoldi_batch(V, ldv, 0, j, 1, w, 0, n, h, 0, hscratch, workspace, workspace_bytes, (hipStream_t)stream, h_host);
  });
}

// The same step for k bases at once: basis r starts at V + r * v_rhs, its
// candidate at w + r * w_rhs, its coefficients at h + r * h_rhs.
extern "C" int rmw_arnoldi_cgs2_batch(double* V, int64_t ldv, int64_t v_rhs, int j, int k, double* w, int64_t w_rhs,
                                      int64_t n, double* h, int64_t h_rhs, double* hscratch, void* workspace,
                                      size_t workspace_bytes, void* stream)
{
  return guarded([&] {
    arnoldi_batch(V, ldv, v_rhs, j, k, w, w_rhs, n, h, h_rhs, hscratch, workspace, workspace_bytes,
                  (hipStream_t)stream);
  });
}
